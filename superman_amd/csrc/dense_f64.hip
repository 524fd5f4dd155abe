// dense_f64.hip -- single-matrix dense real FP64 Ryser kernel (gfx950).
//
// Replaces the reference's dense GPU kernels
// (Algorithms/GPU/Dense/DenseKernelDefinitions.cuh:37-552: xRegisterMShared,
// xRegisterMSharedKahan and their placement variants).  The per-chunk walk is
// in walk_f64.h, the grid-strided task loop and the block reduction in
// dense_chunks.h; this file holds the kernels that take a matrix as it is
// (those with a column to scale to ones are dense_pair.hip's) and a final
// reduction kernel for spm_dense_f64_noalloc.
#include "dense_chunks.h"
#include "dense_reduce.h"

namespace spm {

template <int N, int U, bool COMP>
__global__ void __launch_bounds__(kDenseBlock) __attribute__((amdgpu_waves_per_eu(real::kDenseWaves<N>)))
dense_f64_kernel(const double* __restrict__ M,   // [2][N][N]: +A then -A, column-major
                 const double* __restrict__ x0,  // x(empty set), N values
                 double* __restrict__ partial,   // [gridDim.x][4]: hi, lo, abs, 0
                 uint64_t task_begin, uint64_t task_end, uint64_t num_chunks, int L,
                 int accumulate)
{
    // Past order 36 a run takes 140 ms and more, nothing of it cold, and the chunk
    // starts that read set columns only can cost the steps' schedule: plain order
    // 38 292.7 ms with them, 281.8 without (order 36 66.7 and 67.7).
    dense_chunks<N, U, real::FpTerm<N, COMP>, N - 1, real::kFoldSteps, N <= 36>(M, x0, partial, task_begin, task_end,
                                                                               num_chunks, L, accumulate);
}

// FP32-product variant for nonnegative, row-scaled matrices (same records
// as the compensated kernel).
template <int N, int U>
__global__ void __launch_bounds__(kDenseBlock) __attribute__((amdgpu_waves_per_eu(real::kDenseWaves<N>)))
dense_f32p_kernel(const double* __restrict__ M, const double* __restrict__ x0, double* __restrict__ partial,
                  uint64_t task_begin, uint64_t task_end, uint64_t num_chunks, int L, int accumulate)
{
    dense_chunks<N, U, real::F32ProdTerm<N>>(M, x0, partial, task_begin, task_end, num_chunks, L, accumulate);
}

// Final reduction of the per-block partials (one block; fixed order).
// `stride` doubles per record, `comps` double-double components per record.
__global__ void __launch_bounds__(256)
reduce_partials_kernel(const double* __restrict__ partial, int nrec, int stride, int comps,
                       double* __restrict__ out)
{
    __shared__ double red[3 * (256 / kWave)];
    double rec[6];
    reduce_partials(partial, nrec, stride, comps, rec, red);
    if (threadIdx.x == 0)
        for (int i = 0; i < 3 * comps; ++i) out[i] = rec[i];
}

// ---------------------------------------------------------------------------
// Instantiation table: N = 1..kMaxN, U = 3 for N >= 5 (blocks of 8 steps),
// U = 0 for the tiny orders.
// ---------------------------------------------------------------------------
template <int N, bool COMP>
const void* dense_f64_ptr()
{
    constexpr int U = real::kDenseUnroll<N>;
    if constexpr (SPM_DENSE_ONLY_N != 0 && N != SPM_DENSE_ONLY_N) return nullptr;
    else return reinterpret_cast<const void*>(&dense_f64_kernel<N, U, COMP>);
}

template <int N>
const void* dense_f32p_ptr()
{
    constexpr int U = real::kDenseUnroll<N>;
    if constexpr (SPM_DENSE_ONLY_N != 0 && N != SPM_DENSE_ONLY_N) return nullptr;
    else return reinterpret_cast<const void*>(&dense_f32p_kernel<N, U>);
}

template <int... Is>
const void* dense_f32p_lookup(int n, std::integer_sequence<int, Is...>)
{
    static const void* const table[] = {nullptr, dense_f32p_ptr<Is + 1>()...};
    return table[n];
}

template <int... Is>
const void* dense_f64_lookup(int n, bool comp, std::integer_sequence<int, Is...>)
{
    static const void* const plain[] = {nullptr, dense_f64_ptr<Is + 1, false>()...};
    static const void* const compd[] = {nullptr, dense_f64_ptr<Is + 1, true>()...};
    return comp ? compd[n] : plain[n];
}

const void* dense_f64_kernel_ptr(int n, bool compensated)
{
    if (n < 1 || n > kMaxN) return nullptr;
    return dense_f64_lookup(n, compensated, std::make_integer_sequence<int, kMaxN>{});
}

const void* dense_f32p_kernel_ptr(int n)
{
    if (n < 1 || n > kMaxN) return nullptr;
    return dense_f32p_lookup(n, std::make_integer_sequence<int, kMaxN>{});
}

int dense_f64_unroll_bits(int n)
{
    return (n >= SPM_DENSE_UNROLL + 2 && n <= SPM_DENSE_PREFETCH_MAX) ? SPM_DENSE_UNROLL : 0;
}

const void* reduce_partials_kernel_ptr() { return reinterpret_cast<const void*>(&reduce_partials_kernel); }

}  // namespace spm
