// spm_kernels.h -- host-visible handles to the device kernels.
//
// Each kernel family exposes a lookup returning the __global__ function's
// host stub address, launched with hipLaunchKernel by the drivers.
#pragma once

#include <stddef.h>
#include <stdint.h>

namespace spm {

constexpr int kMaxN = 63;          // 64-bit Gray index (reference README.md:75)
constexpr int kDenseBlock = 256;   // threads per block of the dense kernels

// dense_f64.hip
//   args: (const double* M /* [2][n][n]: +A, -A column-major */, const double* x0, double* partial,
//          uint64_t task_begin, uint64_t task_end, uint64_t num_chunks, int L,
//          int accumulate)
const void* dense_f64_kernel_ptr(int n, bool compensated);
// FP32-product variant (rows pre-scaled by f32prod_scale); same arguments.
const void* dense_f32p_kernel_ptr(int n);
int dense_f64_unroll_bits(int n);
//   args: (const double* partial, int nrec, int stride, int comps, double* out)
const void* reduce_partials_kernel_ptr();

// run_io.hip -- the first and last kernel of a plan's run.
struct RunResult {              // pinned host memory
    unsigned long long word[6]; // hi, lo, abs per component, or T mod 2^128 (lo, hi)
    unsigned long long ticks;   // device time from begin to end, 100 MHz
    unsigned int flag;          // the run's sequence number, stored last
    unsigned int pad;
};
//   begin: (const uint4* src, uint4* dst, unsigned words, uint4* zero, unsigned
//          zwords, unsigned long long* t0), 256 threads
//   end:   (const double* partial, int nrec, int stride, int comps, const
//          unsigned long long* t0, RunResult* host, unsigned seq) or (const
//          unsigned long long* partial, int nrec, t0, host, seq), one block
//          of 256
const void* run_begin_kernel_ptr();
const void* run_end_dd_kernel_ptr();
const void* run_end_i128_kernel_ptr();

// dense_pair.hip -- the same arguments for a matrix whose column 0 is all
// ones; orders kPairMinN..kMaxN, L >= kPairMinChunk.
const void* dense_pair_kernel_ptr(int n, bool compensated);
constexpr int kPairMinN = 6;
constexpr int kPairMinChunk = 3;

// dense_c128.hip -- same arguments as the real kernel; M is [2][n][2n]
// (+A, -A; column-major, interleaved re/im), x0 is 2n doubles, and each
// partial record is 8 doubles (re hi, lo, abs, im hi, lo, 0, 0, 0).
constexpr int kMaxComplexN = 63;
const void* dense_c128_kernel_ptr(int n, bool compensated);
// dense_c128_pair.hip -- for matrices of pair_prepare_complex; orders
// kPairMinN.., L >= kPairMinChunk.
const void* dense_c128_pair_kernel_ptr(int n, bool compensated);

// int_dense.hip -- exact integer walk.
//   args: (const int* M /* [2][n][n]: +2A, -2A column-major */, const int* y0,
//          unsigned long long* partial /* [grid][2] */, uint64_t task_begin,
//          uint64_t task_end, uint64_t num_chunks, int L, int accumulate)
const void* int_dense_kernel_ptr(int n);

// int_small.hip -- exact walk in FP64 for integer matrices whose absolute
// row sums are all below 2^int_small_bits(n) (every 0/1 matrix); same
// arguments as int_dense_kernel except that M is [2][n][n] doubles (+2A,
// -2A) and y0 is n doubles.
const void* int_small_kernel_ptr(int n);
int int_small_bits(int n);

// int_sparse.hip -- exact walk over compressed columns (sparse integer
// matrices); same arguments as int_dense_kernel except that M is the record
// array below and y0 is n + 1 int32 values: y(empty set), then 1 when every
// absolute row sum is below 2^b, b = bit width of n (products may then be
// formed in FP64 groups, as int_small_kernel does), else 0.  A column's
// entries in one plane (+2A or -2A) sit in 16-int records (64 bytes, one
// scalar load):
//   [0] next record of the column (or -1), [1] entries in this record
//   (1..7), [2..8] rows, [9..15] values
// Record 2j + p (p = 0: +2A, 1: -2A) is the first of column j; longer
// columns continue in records after the first 2n (a record that continues
// is full).  A zero column has one entry of value 0 on row 0, so that every
// record's first slot is in use.  Unused slots hold row 0 and value 0 and
// are never read.
const void* int_sparse_kernel_ptr(int n);
constexpr int kSparseRec = 16;   // ints per record
constexpr int kSparseSlots = 7;  // entries per record

// int_prune.hip -- exact sum over the subsets with no zero row
// (walk_prune.h).
//   args: (const int* blob, const uint4* tables, const unsigned long long* in,
//          const unsigned int* in_count, unsigned long long* out, unsigned int* out_count,
//          unsigned int cap, int group, unsigned long long* partial
//          /* [grid][2], its own for each launch */, uint64_t begin, uint64_t
//          end), kPruneBlock threads, dynamic LDS PrunePlan::lds_bytes, a
//          grid of at least kPruneSets waves in every launch but those of a
//          run of one launch.  Launch k of a run takes prefixes
//          of the groups above `group` (in_count null: all settings, [begin,
//          end), end - begin a power of two) and lists the survivors of
//          group's settings in `out`; the last one (nodes true, group 1)
//          walks the listed nodes, with out_count as its work counters.
//          Lists have kPruneSets segments of cap prefixes; a set of counters
//          is kPruneSets lines, all 0 before the run.
// field_bytes 1 (dwords 4, 8, 12, 16) or 2 (dwords 8, 16, 24).
const void* int_prune_kernel_ptr(int field_bytes, int dwords, bool nodes);
//   tables: (const int* blob, int field_bytes, int dwords, uint32_t* tables
//          /* PrunePlan::lds_bytes */), 256 threads, a thread for every 4 bytes
const void* prune_tables_kernel_ptr();
constexpr int kPruneBlock = 512;
constexpr int kPruneLevels = 12;      // column groups of 6 of 62 walked columns, and one
constexpr int kPruneTopBits = 15;     // the first launch has at most 2^15 prefixes
constexpr int kPruneSets = 64;        // counters per launch, one 64-byte line each
constexpr int kPruneCounterStride = 16;
constexpr int kPruneEntriesMax = 2048;  // zero masks (8 bytes each)
constexpr size_t kPruneStaticLds = (kPruneBlock / 64) * (16 + 8 * kPruneLevels + 2048);
constexpr size_t kPruneLdsMax = 65536;
// The blob (ints): the header slots, then sections at places that depend on
// the template's dwords and fields only, so that the kernel's scalar loads
// of them need no offset loaded first.
enum PruneSlot {
    kPruneGroups,   // column groups of 6
    kPruneLeaf,     // leading fields that have zero masks (a multiple of two dwords' fields)
    kPruneTested,   // those of them that are tested (the masks of the others are 0)
    kPruneStride,   // zero masks per field
    kPruneMode,     // product()
    kPruneBits,     // walked columns, n - 1
    kPruneUsed = 8,                               // [kPruneLevels] dwords with a nonzero care mask
    kPruneZero = kPruneUsed + kPruneLevels        // [dwords] packed zero pattern, -o; then:
};
constexpr int prune_offset_at(int dwords) { return kPruneZero + dwords; }              // [fields] o: y = field + o (or packed, product())
constexpr int prune_care_at(int dwords, int fields) { return prune_offset_at(dwords) + fields; }  // [kPruneLevels][dwords]
constexpr int prune_on_at(int dwords, int fields)     // [kMaxN][2][dwords] a column's fields: in the subset, out of it
{
    return prune_care_at(dwords, fields) + kPruneLevels * dwords;
}
constexpr int prune_blob_ints(int dwords, int fields) { return prune_on_at(dwords, fields) + kMaxN * 2 * dwords; }

// Generated SpaRyser kernels walk 2^3-step blocks with L > 3.
constexpr int kCodegenMinN = 5;

}  // namespace spm
