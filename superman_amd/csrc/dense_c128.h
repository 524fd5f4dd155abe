// dense_c128.h -- the task loop and block reduction of the dense complex128
// kernels (dense_c128.hip, dense_c128_pair.hip).
#ifndef SPM_DENSE_C128_H
#define SPM_DENSE_C128_H

#include "walk_c128.h"

namespace spm {
namespace cplx {

// L: log2 of the steps of a chunk (two subsets each when PAIR).
template <int N, bool COMP, bool PAIR>
__device__ __forceinline__ void c128_chunks(const double* __restrict__ M, const double* __restrict__ x0,
                                            double* __restrict__ partial, uint64_t task_begin, uint64_t task_end,
                                            uint64_t num_chunks, int L, int accumulate)
{
    __shared__ double red[3 * (kDenseBlock / kWave)];
    const uint32_t lane = threadIdx.x & (kWave - 1);
    const uint64_t wave = (uint64_t)blockIdx.x * (kDenseBlock / kWave) + (threadIdx.x / kWave);
    const uint64_t nwave = (uint64_t)gridDim.x * (kDenseBlock / kWave);

    // Only a grid with fewer than 64 chunks has idle lanes, and then each
    // lane has exactly one task: such lanes' sums are dropped at the end.
    const bool idle = (uint64_t)lane >= num_chunks;
    touch_lines<4 * N * N, kDenseBlock>(M, threadIdx.x);
    double re_hi = 0.0, re_lo = 0.0, im_hi = 0.0, im_lo = 0.0, abs_sum = 0.0;

    for (uint64_t task = task_begin + wave; task < task_end; task += nwave) {
        const uint64_t h = task * kWave + lane;
        walk_c128<N, COMP, PAIR>(M, x0, h, L, re_hi, re_lo, im_hi, im_lo, abs_sum);
    }
    if (idle) re_hi = re_lo = im_hi = im_lo = abs_sum = 0.0;

    double zero_abs = 0.0;
    block_reduce_dd(re_hi, re_lo, abs_sum, red);
    __syncthreads();
    block_reduce_dd(im_hi, im_lo, zero_abs, red);
    if (threadIdx.x == 0) {
        double* out = partial + 8 * blockIdx.x;
        if (accumulate) {
            dd_add(re_hi, re_lo, out[0], out[1]);
            abs_sum += out[2];
            dd_add(im_hi, im_lo, out[3], out[4]);
        }
        out[0] = re_hi;
        out[1] = re_lo;
        out[2] = abs_sum;
        out[3] = im_hi;
        out[4] = im_lo;
        out[5] = 0.0;
        out[6] = 0.0;
        out[7] = 0.0;
    }
}

}  // namespace cplx
}  // namespace spm

#endif
