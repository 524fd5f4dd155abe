// dense_c128.hip -- single-matrix dense complex128 Ryser kernel (gfx950).
//
// Replaces the reference's complex GPU kernels
// (Algorithms/Complex/gpuComputeComplex.cu:39-197, xRegisterMSharedComplex
// and its NOV-specialised twin).  The per-chunk walk is in walk_c128.h, the
// task loop in dense_c128.h; these are the kernels that take a matrix as it is
// (those with a column to scale to ones are dense_c128_pair.hip's).
#include "dense_c128.h"

// SPM_C128_ONLY_N (sweeps only): instantiate a single order.
#ifndef SPM_C128_ONLY_N
#define SPM_C128_ONLY_N 0
#endif

namespace spm {

namespace cplx {

// Minimum waves per SIMD asked of the register allocator, per order: 3 for
// 29..35, where 168 VGPRs keep the 2-step walk free of spills (the one-off
// chunk-start code may spill a few values) and the compiler's own choice
// (up to 200 VGPRs) leaves 2 -- measured 15% faster at n = 32; at 36 the
// walk itself would spill; 1 = the compiler's choice (forcing 4 at n = 24
// measured slower).
// SPM_C128_WAVES_PER_EU (sweeps only) overrides it for every order.
#ifndef SPM_C128_WAVES_PER_EU
#define SPM_C128_WAVES_PER_EU 0
#endif
template <int N>
constexpr int kC128Waves = SPM_C128_WAVES_PER_EU > 0 ? SPM_C128_WAVES_PER_EU : (N >= 29 && N <= 35) ? 3 : 1;

template <int N, bool COMP>
__global__ void __launch_bounds__(kDenseBlock) __attribute__((amdgpu_waves_per_eu(kC128Waves<N>)))
dense_c128_kernel(const double* __restrict__ M,   // [2][N][2N]: +A then -A, column-major, (re, im)
                  const double* __restrict__ x0,  // 2N doubles
                  double* __restrict__ partial,   // [gridDim.x][8]: re hi lo abs, im hi lo 0, 0, 0
                  uint64_t task_begin, uint64_t task_end, uint64_t num_chunks, int L, int accumulate)
{
    c128_chunks<N, COMP, false>(M, x0, partial, task_begin, task_end, num_chunks, L, accumulate);
}

template <int N, bool COMP>
const void* c128_ptr()
{
    if constexpr (SPM_C128_ONLY_N != 0 && N != SPM_C128_ONLY_N) return nullptr;
    else return reinterpret_cast<const void*>(&dense_c128_kernel<N, COMP>);
}

template <int... Is>
const void* c128_lookup(int n, bool comp, std::integer_sequence<int, Is...>)
{
    static const void* const plain[] = {nullptr, c128_ptr<Is + 1, false>()...};
    static const void* const compd[] = {nullptr, c128_ptr<Is + 1, true>()...};
    return comp ? compd[n] : plain[n];
}

}  // namespace cplx

const void* dense_c128_kernel_ptr(int n, bool compensated)
{
    if (n < 1 || n > kMaxComplexN) return nullptr;
    return cplx::c128_lookup(n, compensated, std::make_integer_sequence<int, kMaxComplexN>{});
}

}  // namespace spm
