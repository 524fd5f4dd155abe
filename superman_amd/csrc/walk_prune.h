// walk_prune.h -- exact Ryser sum of an integer matrix over the subsets with
// no zero row only (gfx950 device code of int_prune.hip).
//
//   T = sum_S (-1)^|S| prod_i y_i(S),  y_i(S) = y_i(0) + sum_{j in S} w_i a_ij
//
// (w_i = 1 on rows with even sums, carried halved; 2 otherwise.)  A subset
// with y_i(S) = 0 for some row adds nothing, and on 0/1 and small-integer
// matrices almost every subset has such a row.  The Gray walks visit every
// subset, one flip and one test at a time; here the subsets are a tree over
// groups of 6 columns that is cut where a row is zero for good:
//
//   * The row sums of one subset are packed fields (8 or 16 bits, biased to
//     be nonnegative), NQ dwords in all.  A group's 64 settings add one of
//     64 packed vectors each, tabulated in LDS: one node's 64 children are
//     one LDS read and NQ packed adds, child b in lane b.
//   * Columns are ordered so that the outer groups complete as many rows as
//     they can (prune_plan).  A row whose columns are all set is compared
//     with its zero pattern in all fields of a dword at once; the children
//     left are a ballot, walked depth first by the wave.
//   * The two innermost groups are never walked: lane b takes setting b of
//     group 1, and for each row with entries in group 0 a table in LDS,
//     indexed by the row's sum over the other columns, holds the 64-bit mask
//     of group 0's settings that make the row zero.  The OR of one word per
//     row marks every dead subset of 64 at once (4096 per node and wave).
//   * Surviving subsets go to a queue per wave as column masks; 64 at a time
//     their row sums are read back from the tables and multiplied out, one
//     term per lane, exact mod 2^128.
//
// A zero row costs nothing but its share of one node, so the time follows
// the surviving nodes and terms, not 2^(n-1).
#ifndef SPM_WALK_PRUNE_H
#define SPM_WALK_PRUNE_H

#include "spm_device.h"
#include "spm_kernels.h"
#include "walk_int.h"

namespace spm {
namespace prune {

using ints::const_i32;

__device__ __forceinline__ uint32_t uni(uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); }
__device__ __forceinline__ uint64_t uni(uint64_t v)
{
    return ((uint64_t)uni((uint32_t)(v >> 32)) << 32) | uni((uint32_t)v);
}

// The blob's address passed through an empty asm, so that the scalar loads
// behind it stay where they are used: hoisted out of the task loop, the
// offsets and patterns alone would overflow the SGPR file and come back
// through v_readlane at every use.
__device__ __forceinline__ const const_i32* here(const int* blob)
{
    asm volatile("" : "+s"(blob));
    return (const const_i32*)blob;
}

// d += the packed vector of table entry `e` (16-byte aligned: NQ % 4 == 0).
template <int NQ>
__device__ __forceinline__ void add_entry(uint32_t (&d)[NQ], const uint32_t* tab, uint32_t e)
{
    const uint4* p = (const uint4*)(tab + e * NQ);
#pragma unroll
    for (int i = 0; i < NQ / 4; ++i) {
        const uint4 v = p[i];
        d[4 * i] += v.x;
        d[4 * i + 1] += v.y;
        d[4 * i + 2] += v.z;
        d[4 * i + 3] += v.w;
    }
}

// False when a field selected by `level`'s care mask equals its zero
// pattern.  Per dword: field == zero exactly when the field of x = c ^ Z is
// 0, i.e. when neither x nor (x & 0x7f..) + 0x7f.. has the field's top bit
// (no carry crosses a field); fields not tested are ORed to all ones.
template <int FB, int NQ>
__device__ __forceinline__ bool rows_nonzero(const uint32_t (&c)[NQ], const int* blob_, int level)
{
    constexpr int kFields = NQ * 4 / FB;
    const const_i32* blob = here(blob_);
    constexpr uint32_t kTop = FB == 1 ? 0x80808080u : 0x80008000u;
    const uint32_t used = (uint32_t)blob[kPruneUsed + level];
    const const_i32* care = blob + prune_care_at(NQ, kFields) + level * NQ;
    const const_i32* zero = blob + kPruneZero;
    uint32_t ok = kTop;
#pragma unroll
    for (int q0 = 0; q0 < NQ; q0 += 4)  // 4 dwords a branch: their scalar loads go out together
        if ((used >> q0) & 15u) {
#pragma unroll
            for (int q = q0; q < q0 + 4; ++q) {
                const uint32_t x = c[q] ^ (uint32_t)zero[q];
                ok &= ((x & ~kTop) + ~kTop) | x | ~(uint32_t)care[q];
            }
        }
    return ok == kTop;
}

// prod_i y_i mod 2^128 of one subset's packed sums, y = field + o (padding
// fields are 0 with o = 1).  The host picks `mode` from the rows' bounds:
//   8-bit fields:  0: two rows of a dword multiply exactly in 32 bits, 4 in 64
//     (the host lays a matrix with larger |y| out in 16-bit fields).
//     1: every y is a signed byte; the offset section holds o + 128 packed,
//     and with the top bits flipped the sums are the y themselves, which the
//     multiplier takes as they are (a byte select is part of the instruction):
//     4 rows in 32 bits, 8 in 64.  2: as 1, and 16 rows fit 64 bits, those
//     of dwords 2i, 2i + 1 and their counterparts in the other half (rows
//     that can be zero come first and are carried halved).
//     With offsets added row by row (5 instead of 1 instructions for two
//     rows) a half 0/1 matrix of order 30 took 1.19 times as long.
//   16-bit fields: 0: any |y| < 2^30, 1 row in 32 bits, 2 in 64;  1: 1 and 4
template <int FB, int NQ>
__device__ __forceinline__ unsigned __int128 product(const uint32_t (&c)[NQ], const int* blob_, int mode)
{
    const const_i32* o = here(blob_) + prune_offset_at(NQ);
    constexpr int F = 4 / FB;
    auto y = [&](int q, int k) __attribute__((always_inline)) {
        return (int)((c[q] >> (8 * FB * k)) & (FB == 1 ? 0xffu : 0xffffu)) + o[q * F + k];
    };
    unsigned __int128 p = 1;
    auto times = [&](int q, long long v) __attribute__((always_inline)) {
        p = q == 0 ? (unsigned __int128)(__int128)v : p * (unsigned __int128)(__int128)v;
    };
    if constexpr (FB == 1) {
        if (mode != 0) {
            long long b[NQ / 2];
#pragma unroll
            for (int i = 0; i < NQ / 2; ++i) {
                int a[2];
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const uint32_t z = (c[2 * i + h] + (uint32_t)o[2 * i + h]) ^ 0x80808080u;
                    int lo, hi;  // (the compiler unpacks half of the bytes first)
                    asm("v_mul_i32_i24_sdwa %0, sext(%1), sext(%1) dst_sel:DWORD dst_unused:UNUSED_PAD "
                        "src0_sel:BYTE_0 src1_sel:BYTE_1"
                        : "=v"(lo)
                        : "v"(z));
                    asm("v_mul_i32_i24_sdwa %0, sext(%1), sext(%1) dst_sel:DWORD dst_unused:UNUSED_PAD "
                        "src0_sel:BYTE_2 src1_sel:BYTE_3"
                        : "=v"(hi)
                        : "v"(z));
                    a[h] = lo * hi;
                }
                b[i] = (long long)a[0] * a[1];
            }
            if (mode == 2) {
#pragma unroll
                for (int i = 0; i < NQ / 4; ++i) times(i, b[i] * b[i + NQ / 4]);
            } else {
#pragma unroll
                for (int i = 0; i < NQ / 2; ++i) times(i, b[i]);
            }
        } else {
#pragma unroll
            for (int q = 0; q < NQ; ++q) times(q, (long long)(y(q, 0) * y(q, 1)) * (y(q, 2) * y(q, 3)));
        }
    } else {
        if (mode == 1) {
#pragma unroll
            for (int q = 0; q < NQ; q += 2)
                times(q, ((long long)y(q, 0) * y(q, 1)) * ((long long)y(q + 1, 0) * y(q + 1, 1)));
        } else {
#pragma unroll
            for (int q = 0; q < NQ; ++q) times(q, (long long)y(q, 0) * y(q, 1));
        }
    }
    return p;
}

}  // namespace prune
}  // namespace spm

#endif
