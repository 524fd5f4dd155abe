// dense_chunks.h -- the grid-strided task loop of the dense real FP64 kernels
// (dense_f64.hip, dense_pair.hip): one matrix's chunks and the block
// reduction into per-block records.
#ifndef SPM_DENSE_CHUNKS_H
#define SPM_DENSE_CHUNKS_H

#include "walk_f64.h"

namespace spm {

// The grid-strided task loop over one matrix's chunks and the block
// reduction into per-block records, for the accumulation policy Term.
// COLD: the matrix is touched first and a chunk start reads the set columns only.
template <int N, int U, class Term, int NC = N - 1, uint32_t FOLD = real::kFoldSteps, bool COLD = true>
__device__ __forceinline__ void dense_chunks(const double* __restrict__ M, const double* __restrict__ x0,
                                             double* __restrict__ partial, uint64_t task_begin,
                                             uint64_t task_end, uint64_t num_chunks, int L, int accumulate)
{
    constexpr bool COMP = Term::kCompensated;
    __shared__ double red[3 * (kDenseBlock / kWave)];
    const uint32_t lane = threadIdx.x & (kWave - 1);
    const uint64_t wave = (uint64_t)blockIdx.x * (kDenseBlock / kWave) + (threadIdx.x / kWave);
    const uint64_t nwave = (uint64_t)gridDim.x * (kDenseBlock / kWave);

    if constexpr (COLD)
        touch_lines<(N + 1 + NC) * N, kDenseBlock>(M, threadIdx.x);  // M is column N - 1 - NC of the first plane
    double acc_hi = 0.0, acc_lo = 0.0, acc_abs = 0.0;
    for (uint64_t task = task_begin + wave; task < task_end; task += nwave) {
        const uint64_t h = task * kWave + lane;
        const bool active = h < num_chunks;  // lanes past the end walk a dummy chunk
        Term term;
        real::walk_gray<N, U, Term, NC, FOLD, COLD>(M, x0, h, L, term);
        if (active) {
            if constexpr (COMP) {
                dd_add(acc_hi, acc_lo, term.t_hi, term.t_lo);
                acc_abs += term.t_abs;
            } else {
                acc_hi += term.t_hi;
            }
        }
    }
    block_reduce_dd(acc_hi, acc_lo, acc_abs, red);
    if (threadIdx.x == 0) {
        double* out = partial + 4 * blockIdx.x;
        if (accumulate) {  // later slice of a long run: add onto this block's record
            dd_add(acc_hi, acc_lo, out[0], out[1]);
            acc_abs += out[2];
        }
        out[0] = acc_hi;
        out[1] = acc_lo;
        out[2] = acc_abs;
        out[3] = 0.0;
    }
}

}  // namespace spm

#endif
