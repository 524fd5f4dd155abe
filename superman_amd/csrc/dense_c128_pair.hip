// dense_c128_pair.hip -- single-matrix dense complex128 Ryser kernel (gfx950)
// for a matrix whose column 0 is (1, 0) in all but its last two rows, two
// subsets per step (PairProd in walk_c128.h).
//
// VALU issue bounds it: 162 FP64 instructions per subset at order 32 (191 in
// dense_c128_kernel); Haar order 32 takes 10.5-10.8 ms a call (12.7 there),
// Gauss order 24 52 us a run (62), order 30 2.41 ms (2.91).
#include "dense_c128.h"

// SPM_C128_ONLY_N (sweeps only): instantiate a single order.
#ifndef SPM_C128_ONLY_N
#define SPM_C128_ONLY_N 0
#endif

namespace spm {

namespace cplx {

// Minimum waves per SIMD asked of the register allocator, as dense_c128.hip.
template <int N>
constexpr int kPairWaves = (N >= 29 && N <= 35) ? 3 : 1;

template <int N, bool COMP>
__global__ void __launch_bounds__(kDenseBlock) __attribute__((amdgpu_waves_per_eu(kPairWaves<N>)))
dense_c128_pair_kernel(const double* __restrict__ M,   // [2][N][2N]: +A then -A, column-major, (re, im)
                       const double* __restrict__ x0,  // 2N doubles
                       double* __restrict__ partial,   // [gridDim.x][8]: re hi lo abs, im hi lo 0, 0, 0
                       uint64_t task_begin, uint64_t task_end, uint64_t num_chunks, int L, int accumulate)
{
    // a chunk of 2^L subsets is 2^(L-1) steps
    c128_chunks<N, COMP, true>(M, x0, partial, task_begin, task_end, num_chunks, L - 1, accumulate);
}

template <int N, bool COMP>
const void* c128_pair_ptr()
{
    if constexpr (N < kPairMinN || (SPM_C128_ONLY_N != 0 && N != SPM_C128_ONLY_N)) return nullptr;
    else return reinterpret_cast<const void*>(&dense_c128_pair_kernel<N, COMP>);
}

template <int... Is>
const void* c128_pair_lookup(int n, bool comp, std::integer_sequence<int, Is...>)
{
    static const void* const plain[] = {nullptr, c128_pair_ptr<Is + 1, false>()...};
    static const void* const compd[] = {nullptr, c128_pair_ptr<Is + 1, true>()...};
    return comp ? compd[n] : plain[n];
}

}  // namespace cplx

const void* dense_c128_pair_kernel_ptr(int n, bool compensated)
{
    if (n < 1 || n > kMaxComplexN) return nullptr;
    return cplx::c128_pair_lookup(n, compensated, std::make_integer_sequence<int, kMaxComplexN>{});
}

}  // namespace spm
