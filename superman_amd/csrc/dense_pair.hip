// dense_pair.hip -- single-matrix dense real FP64 Ryser kernel (gfx950) for a
// matrix whose column 0 is all ones, two subsets per step (PairTerm in
// walk_f64.h): the walk of dense_f64.hip over columns 1..N-2.
//
// VALU issue bounds it: 62.5 FP64 instructions per subset at order 40 (80.8
// in dense_f64_kernel), no memory traffic to speak of; order 40 takes 1013 ms
// (1269 ms there), order 33 plain 6.3 ms (8.0 ms).  That is 4.6 cycles per
// wave instruction; a loop of such multiplies and FMAs alone takes 4.5 at the
// same 4 waves per SIMD.  127 VGPRs at order 40 allow no fifth wave, and
// asking for 5 at orders 25-38 or 6 below moved no time by more than 2 %.
#include "dense_chunks.h"

namespace spm {

template <int N, int U, bool COMP>
__global__ void __launch_bounds__(kDenseBlock)
dense_pair_kernel(const double* __restrict__ M,   // [2][N][N]: +A then -A, column-major, column 0 all ones
                  const double* __restrict__ x0,  // x(empty set), N values
                  double* __restrict__ partial,   // [gridDim.x][4]: hi, lo, abs, 0
                  uint64_t task_begin, uint64_t task_end, uint64_t num_chunks, int L, int accumulate)
{
    // A chunk of 2^L subsets is 2^(L-1) steps; folds every 16 subsets.
    dense_chunks<N, U, real::PairTerm<N, COMP>, N - 2, real::kFoldSteps / 2>(M + N, x0, partial, task_begin, task_end,
                                                                            num_chunks, L - 1, accumulate);
}

template <int N, bool COMP>
const void* dense_pair_ptr()
{
    if constexpr (N < kPairMinN || (SPM_DENSE_ONLY_N != 0 && N != SPM_DENSE_ONLY_N)) return nullptr;
    else return reinterpret_cast<const void*>(&dense_pair_kernel<N, real::kDenseUnroll<N>, COMP>);
}

template <int... Is>
const void* dense_pair_lookup(int n, bool comp, std::integer_sequence<int, Is...>)
{
    static const void* const plain[] = {nullptr, dense_pair_ptr<Is + 1, false>()...};
    static const void* const compd[] = {nullptr, dense_pair_ptr<Is + 1, true>()...};
    return comp ? compd[n] : plain[n];
}

const void* dense_pair_kernel_ptr(int n, bool compensated)
{
    if (n < 1 || n > kMaxN) return nullptr;
    return dense_pair_lookup(n, compensated, std::make_integer_sequence<int, kMaxN>{});
}

}  // namespace spm
