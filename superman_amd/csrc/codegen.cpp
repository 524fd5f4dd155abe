// codegen.cpp -- SpaRyser: per-pattern kernels generated and compiled
// in-process with hiprtc.
//
// Replaces the reference's code generation path
// (Algorithms/GPU/CodeGeneration/KernelGenerator.cuh:114-176,
// UTOrderedKernelCodeGen.cuh:34-583, NaiveKernelCodeGen.cuh:34-365) and its
// driver KernelGenSingleGPU (KernelGenSingleGPU.cuh:47-197).  The reference
// writes generated CUDA into its source tree, exits, has a wrapper rebuild
// the whole program, and re-runs it (wrapper.cpp:271-344); here the source
// is compiled by hiprtc inside the call and the code object is cached by a
// hash of the pattern and values.
//
// What is generated, for a matrix whose entries are integers:
//   * the rows after IO::UTOrder (IO/IO.h:926-1002) for the register-efficient
//     variant (column order = ascending remaining in-degree, so the columns
//     flipped most often -- column 0 every other step -- are the sparsest),
//     or the input order for the naive variant;
//   * y = 2x (x on rows with even sums, whose y is always even) kept
//     entirely in VGPRs (at most 63 int32 per lane: the
//     reference's register-area cost model, UTOrderedKernelCodeGen.cuh:68-132,
//     trades registers against global-memory x for CUDA's 255-register
//     limit, which the 512-entry gfx950 file does not need);
//   * for every column c and direction, the exact row updates
//     y_r += +-2 a_rc as integer literals (the reference prints FP literals
//     with std::to_string -- 6 decimals -- which is lossy for general values),
//     with the zero-row count of each lane kept incrementally;
//   * the same wave-uniform Gray walk as the dense kernels: lane chunks of
//     2^L steps, blocks of 2^U steps whose first flip is a runtime column
//     (a uniform switch) and whose other flips are compile-time columns;
//   * the term prod_r y_r (128-bit) only on lanes whose zero count is 0, and
//     128-bit accumulation (mod 2^128; the host proves |T| < 2^127).
// Compiled code objects are kept per (device, hash) in the process and on
// disk (codegen_get_kernel), so a pattern compiles once per machine.
#include "superman_amd.h"

#include "spm_host.h"
#include "spm_kernels.h"

#include <hip/hip_runtime.h>
#include <hip/hiprtc.h>

#include <sys/stat.h>
#include <unistd.h>

#include <algorithm>
#include <iterator>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <sstream>
#include <string>
#include <vector>

namespace spm {

// ---------------------------------------------------------------------------
// IO::UTOrder (IO/IO.h:926-1002): repeatedly take the first column of least
// remaining in-degree; rows are numbered in the order they are first touched
// and, once numbered, no longer count towards the in-degrees.
// ---------------------------------------------------------------------------
void ut_order_mask(const unsigned char* nz, int n, std::vector<int>& rowPerm, std::vector<int>& colPerm)
{
    rowPerm.assign(n, 0);
    colPerm.assign(n, 0);
    for (int i = 0; i < n; ++i) rowPerm[i] = colPerm[i] = i;
    const unsigned kDone = 0xffffffffu;
    std::vector<unsigned> indeg(n, 0);
    for (int j = 0; j < n; ++j)
        for (int i = 0; i < n; ++i) indeg[j] += nz[i * n + j] != 0;
    std::vector<bool> marked(n, false);
    int nextRow = 0;
    for (int step = 0; step < n; ++step) {
        unsigned mind = kDone;
        int chosen = 0;
        for (int j = 0; j < n; ++j)
            if (indeg[j] < mind) {
                mind = indeg[j];
                chosen = j;
            }
        colPerm[chosen] = step;
        indeg[chosen] = kDone;
        for (int i = 0; i < n; ++i) {
            if (nz[i * n + chosen] == 0 || marked[i]) continue;
            marked[i] = true;
            rowPerm[i] = nextRow++;
            for (int j = 0; j < n; ++j)
                if (indeg[j] != kDone && nz[i * n + j] != 0) --indeg[j];
        }
    }
    for (int i = 0; i < n; ++i)
        if (!marked[i]) rowPerm[i] = nextRow++;
}

void ut_order(const int64_t* a, int n, std::vector<int>& rowPerm, std::vector<int>& colPerm)
{
    std::vector<unsigned char> nz((size_t)n * n);
    for (size_t e = 0; e < nz.size(); ++e) nz[e] = a[e] != 0;
    ut_order_mask(nz.data(), n, rowPerm, colPerm);
}

// newMat[rowPerm[i]][colPerm[j]] = mat[i][j] (IO::applyPermutations, IO/IO.h:1095-1112)
std::vector<int64_t> apply_perm(const int64_t* a, int n, const std::vector<int>& rp, const std::vector<int>& cp)
{
    std::vector<int64_t> b((size_t)n * n);
    for (int i = 0; i < n; ++i)
        for (int j = 0; j < n; ++j) b[(size_t)rp[i] * n + cp[j]] = a[i * n + j];
    return b;
}

// log2 of the steps per generated block.  A block's first flip goes
// through a chain of bit tests on the block index, its 2^U - 1 others are
// straight-line code with the column and direction known at compile time,
// so longer blocks run faster and compile longer (2^U copies of the term
// product; about 2.5e-3 2^U n seconds of hiprtc).  Measured on order-40 0/1
// patterns (config 3 / rows of 4 and 5 entries): U = 3 127.6 / 198.1 ms,
// 0.9 s compile; U = 4 100.0 / 187.1 ms, 1.6 s; U = 5 77.1 / 175.8 ms,
// 3.3 s.  Integer kernels: U = 3 up to order 30 (a permanent there takes
// milliseconds, the compile dominates), 4 up to 45, 5 beyond (one walk
// takes tens of seconds).  Kernels whose terms are rarest (gen_compact_term)
// test them once per block, with one copy of the term product, and afford
// U = 5 from order 31 (config 3: 58 ms with a 0.31 s compile, against 86 ms
// and 0.69 s testing each step with the product in a loop, 100 ms and
// 1.58 s inlined at U = 4; rows of 6 entries at order 40: 272 -> 223 ms,
// 1.72 -> 0.40 s).  With more terms the block replays cost more than they
// save (rows of 8 entries, about 3e-4 of the subsets with no zero row:
// 606 -> 1099 ms).  Real kernels form their term from cached
// suffix products, so their code stays small: U = 5 from order 21 (order
// 40, N(0,1) on 4 entries per row: 136 / 102 / 85 ms at U = 3 / 4 / 5,
// 0.25 s compile each).
int gen_unroll_bits_int(int n, bool compact) { return n <= 30 ? 3 : ((compact || n > 45) ? 5 : 4); }
int gen_unroll_bits_real(int n) { return n <= 20 ? 3 : 5; }

// ---------------------------------------------------------------------------
// Source emitter (integer entries).
// ---------------------------------------------------------------------------
namespace {


// Waves per SIMD asked of the register allocator (0: the compiler's
// choice).  Orders 29..40: the natural allocation (100-127 VGPRs) leaves 4;
// at 96 VGPRs the compiler spills only around the term product and the
// final reduction (config-3 order-40 pattern: 155 -> 141 ms).  Orders
// 41..48: 129-130 VGPRs leave 3; 128 spill at most 8 bytes (order-42
// pattern: 706 -> 590 ms); kernels testing their terms once per block
// (RARE) hold one product and take 5 there too (order 44, 6 entries per
// row: 2158 -> 1892 ms; no gain at 6).  Orders up to 28 reach 5 without it.
int gen_waves_per_simd(int n, bool rare)
{
    if (n >= 29 && n <= 40) return 5;
    if (n >= 41 && n <= 48) return rare ? 5 : 4;
    return 0;
}

// Real kernels hold x as FP64 (2 VGPRs per row); 0 = the compiler's choice.
int gen_real_waves_per_simd(int n)
{
    (void)n;
    return 0;
}

std::string lit(int64_t v)
{
    return std::to_string(v);  // integers are exact in decimal
}

// y_r += D, keeping Z = number of zero rows among the rows that can be zero
// (zr[r]; a row with an odd sum never is); wb = the walk's increments (row
// weight x entry).
void emit_flip_const(std::ostringstream& o, const std::vector<int64_t>& wb, const std::vector<char>& zr, int n,
                     int c, int sgn, const char* ind)
{
    for (int r = 0; r < n; ++r) {
        const int64_t d = wb[(size_t)r * n + c] * sgn;
        if (d == 0) continue;
        o << ind << "y" << r << " += " << lit(d) << ";";
        if (zr[r]) o << " Z += (y" << r << " == 0) - (y" << r << " == " << lit(d) << ");";
        o << "\n";
    }
}

// per-lane direction: D = (d ^ mask) - mask with mask = 0 (add) or -1
// (remove) in each lane
void emit_flip_lane(std::ostringstream& o, const std::vector<int64_t>& wb, const std::vector<char>& zr, int n, int c,
                    const char* mask, const char* ind)
{
    for (int r = 0; r < n; ++r) {
        const int64_t d = wb[(size_t)r * n + c];
        if (d == 0) continue;
        o << ind << "{ const int D = (" << lit(d) << " ^ " << mask << ") - " << mask << "; y" << r << " += D;";
        if (zr[r]) o << " Z += (y" << r << " == 0) - (y" << r << " == D);";
        o << " }\n";
    }
}

// The term of the current subset, on the lanes where no row is zero.  The
// test is a wave-wide ballot with a cold-branch hint: on sparse patterns
// almost no wave holds a nonzero term, and a uniform, not-taken branch costs
// far less per step than a lane-divergent region around the product, an
// inlined 128-bit chain over row pairs.  FOLD (steps of kernels whose terms
// are rarest, gen_compact_term) only folds Z into the block's least zero
// count Zm; SIGN_VAR names a run-time sign (true: subtract).
void emit_term(std::ostringstream& o, int n, bool negative, const char* ind, bool fold = false, bool first = false,
               const char* sign_var = nullptr)
{
    if (fold) {
        o << ind << (first ? "Zm = Z;\n" : "Zm = min(Zm, Z);\n");
        return;
    }
    o << ind << "if (__builtin_expect(__builtin_amdgcn_ballot_w64(Z == 0) != 0, 0)) {\n";
    o << ind << "  if (Z == 0) {\n";
    o << ind << "    unsigned __int128 p = (unsigned __int128)(__int128)y0;\n";
    int r = 1;
    for (; r + 1 < n; r += 2)
        o << ind << "    p *= (unsigned __int128)(__int128)((long long)y" << r << " * (long long)y" << r + 1 << ");\n";
    if (r < n) o << ind << "    p *= (unsigned __int128)(__int128)y" << r << ";\n";
    if (sign_var) o << ind << "    acc = " << sign_var << " ? acc - p : acc + p;\n";
    else o << ind << "    acc " << (negative ? "-" : "+") << "= p;\n";
    o << ind << "  }\n";
    o << ind << "}\n";
}

// Compact kernels test no term per step: each step folds Z into the block's
// least zero count Zm (one VALU op, no branch waiting on a compare).  At the
// end of block M, when some lane's Zm is 0, the wave walks the block back
// from its last step (undoing flips 2^U - 1 .. 1 through flipc, a switch
// over columns 0..U-1), forming each subset's term on the way, and then
// forward again to restore its rows.
void emit_block_replay(std::ostringstream& o, int U, const char* M, const char* ind)
{
    const unsigned last = (1u << U) - 1;
    o << ind << "if (__builtin_expect(__builtin_amdgcn_ballot_w64(Zm == 0) != 0, 0)) {\n";
    o << ind << "#pragma nounroll\n";
    o << ind << "  for (unsigned j = " << last << "u;; --j) {\n";
    o << ind << "    termc((j & 1u) != 0);\n";
    o << ind << "    if (j == 0u) break;\n";
    o << ind << "    const unsigned c = __builtin_ctz(j);\n";
    o << ind << "    const unsigned bit = c == " << U - 1 << "u ? (" << M << " & 1u) : ((j >> (c + 1)) & 1u);\n";
    o << ind << "    flipc(c, ~(-(int)bit));\n";
    o << ind << "  }\n";
    o << ind << "#pragma nounroll\n";
    o << ind << "  for (unsigned j = 1u; j <= " << last << "u; ++j) {\n";
    o << ind << "    const unsigned c = __builtin_ctz(j);\n";
    o << ind << "    const unsigned bit = c == " << U - 1 << "u ? (" << M << " & 1u) : ((j >> (c + 1)) & 1u);\n";
    o << ind << "    flipc(c, -(int)bit);\n";
    o << ind << "  }\n";
    o << ind << "}\n";
}

// A pruned kernel takes a chunk's prefix, the subset's columns >= L, through
// three sieves before it walks the chunk: rows whose columns are all >= L + 12,
// then >= L + 6, then >= L, each tested at the first level that fixes them and
// each dropping every chunk below for good when zero (the term of every
// subset there is).  The prefixes of a level are tested 64 at a time, one per
// lane: 64 blocks (of 64 tasks), the 64 tasks of a live block, the 64 chunks of
// a live task.  (Order 40 has 2^22 blocks: tested one by one in scalar code
// they took 0.5 ms.)
struct Sieve {
    int level;              // columns below are not fixed yet
    std::vector<int> rows;  // rows fixed at this level and not before
};

std::vector<Sieve> sieves(const std::vector<int64_t>& b, const std::vector<char>& zr, int n)
{
    std::vector<Sieve> v = {{kGenPruneChunk + 12, {}}, {kGenPruneChunk + 6, {}}, {kGenPruneChunk, {}}};
    for (int r = 0; r < n; ++r) {
        if (!zr[r]) continue;
        int low = n;
        for (int c = n - 2; c >= 0; --c)
            if (b[(size_t)r * n + c] != 0) low = c;
        for (Sieve& s : v)
            if (low >= s.level) {
                s.rows.push_back(r);
                break;
            }
    }
    return v;
}

// One sieve over the lanes' prefixes, which clears `alive`; g names the 64-bit
// Gray prefix whose bits >= level are the subset's columns.  Leaves the
// (outer) loop's round when no lane is left.
void emit_sieve(std::ostringstream& o, const Sieve& s, const std::vector<int64_t>& wb, const std::vector<int64_t>& y0,
                int n, const char* g, const char* ind)
{
    int k = 0;
    for (int r : s.rows) {
        o << ind << "{ int v = " << lit(y0[r]) << ";";
        for (int c = s.level; c < n - 1; ++c) {
            const int64_t d = wb[(size_t)r * n + c];
            if (d != 0) o << " v += " << lit(d) << " & -(int)((" << g << " >> " << c << ") & 1ull);";
        }
        o << " alive = alive && v != 0; }\n";
        if (++k % 4 == 0) o << ind << "if (__builtin_amdgcn_ballot_w64(alive) == 0) continue;\n";
    }
}

}  // namespace

std::string emit_int_kernel(const std::vector<int64_t>& b, int n, const std::string& name)
{
    const bool compact = gen_compact_term(b.data(), n);
    const bool prune = gen_pruned(b.data(), n);
    const int U = codegen_int_unroll_bits(b.data(), n);
    // y = 2x, halved on rows with even sums (int_row_weights): wb holds the
    // walk's increments w_r b_rc
    std::vector<unsigned char> w(n);
    int_row_weights(b.data(), n, w.data());
    std::vector<int64_t> wb(b.size()), y0(n);
    // a row with an odd sum keeps y = 2x odd (2 a_{r,n-1} - r_r + 2 sum_S
    // a_rj), so it is never zero and stays out of Z: its flips are one add
    std::vector<char> zr(n);
    for (int i = 0; i < n; ++i) {
        int64_t rs = 0;
        for (int j = 0; j < n; ++j) {
            rs += b[(size_t)i * n + j];
            wb[(size_t)i * n + j] = w[i] * b[(size_t)i * n + j];
        }
        y0[i] = 2 * b[(size_t)i * n + n - 1] - rs;
        if (w[i] == 1) y0[i] /= 2;
        zr[i] = (rs & 1) == 0 ? 1 : 0;
    }
    std::ostringstream o;
    o << "// generated: SpaRyser kernel for one " << n << "x" << n << " integer pattern\n";
    o << "extern \"C\" __global__ void __launch_bounds__(256)";
    if (const int w = gen_waves_per_simd(n, compact)) o << " __attribute__((amdgpu_waves_per_eu(" << w << ")))";
    o << "\n";
    o << name << "(unsigned long long* __restrict__ partial, unsigned long long task_begin,\n"
      << "    unsigned long long task_end, unsigned long long num_chunks, int L, int accumulate)\n{\n";
    if (!prune) {
        o << "    __shared__ unsigned long long red[8];\n"
             "    const unsigned lane = threadIdx.x & 63u;\n"
             "    const unsigned long long wave = (unsigned long long)blockIdx.x * 4 + (threadIdx.x >> 6);\n"
             "    const unsigned long long nwave = (unsigned long long)gridDim.x * 4;\n"
             "    const bool idle = (unsigned long long)lane >= num_chunks;\n"
             "    unsigned __int128 acc = 0;\n"
             "    for (unsigned long long task = task_begin + wave; task < task_end; task += nwave) {\n"
             "        const unsigned long long h = task * 64 + lane;\n";
    } else {
        // Blocks (in 2^cut parts when there are few) go to the waves in
        // batches of up to 64, in the order of a bijection of their index
        // (neighbouring prefixes survive alike).  bm and tm: the batch's
        // parts and the part's tasks still to look into.  Live chunks wait
        // in a queue per wave until 64 are walked together.
        const std::vector<Sieve> sv = sieves(b, zr, n);
        const int LC = kGenPruneChunk, bb = n - 1 - LC - 12, cut = std::min(6, std::max(0, 15 - bb));
        const int pb = std::min(6, std::max(0, bb + cut - 13));  // log2 of a batch
        o << "    __shared__ unsigned long long red[8];\n"
             "    __shared__ unsigned long long live[4 * 128];\n"
             "    const unsigned lane = threadIdx.x & 63u;\n"
             "    const unsigned w0 = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);\n"
             "    const unsigned long long nwave = (unsigned long long)gridDim.x * 4;\n"
             "    const unsigned long long parts = (task_end - task_begin) >> " << 6 - cut << ";\n"
             "    unsigned long long* const queue = live + w0 * 128;\n"
             "    unsigned long long pi = (unsigned long long)blockIdx.x * 4 + w0, x = 0, T0 = 0, bm = 0, tm = 0;\n"
             "    unsigned head = 0, tail = 0;\n"
             "    unsigned __int128 total = 0;\n"
             "    for (;;) {\n"
             "        while (tail - head < 64u) {\n"
             "            if (tm == 0) {\n"
             "                if (bm == 0) {\n"
             "                    if (pi >= parts >> " << pb << ") break;\n"
             "                    bool alive = lane < " << (1 << pb) << "u;\n"
             "                    x = (((pi << " << pb << ") + lane) * 0x9e3779b97f4a7c15ull) & (parts - 1);\n"
             "                    x ^= x >> " << std::max(1, (bb + cut) / 2) << ";\n"
             "                    x = task_begin + (((x * 0xbf58476d1ce4e5b9ull) & (parts - 1)) << " << 6 - cut << ");\n"
             "                    pi += nwave;\n"
             "                    const unsigned long long kb = x << " << LC + 6 << ", gb = kb ^ (kb >> 1);\n";
        emit_sieve(o, sv[0], wb, y0, n, "gb", "                    ");
        o << "                    bm = __builtin_amdgcn_ballot_w64(alive);\n"
             "                    continue;\n"
             "                }\n"
             "                const int bl = __builtin_ctzll(bm);\n"
             "                bm &= bm - 1;\n"
             "                T0 = ((unsigned long long)(unsigned)__builtin_amdgcn_readlane((int)(x >> 32), bl) << 32) | "
             "(unsigned)__builtin_amdgcn_readlane((int)(unsigned)x, bl);\n"
             "                bool alive = lane < " << (64 >> cut) << "u;\n"
             "                const unsigned long long kt = (T0 + lane) << " << LC + 6 << ", gt = kt ^ (kt >> 1);\n";
        emit_sieve(o, sv[1], wb, y0, n, "gt", "                ");
        o << "                tm = __builtin_amdgcn_ballot_w64(alive);\n"
             "                continue;\n"
             "            }\n"
             "            const unsigned long long hc = (T0 + __builtin_ctzll(tm)) * 64 + lane, kc = hc << " << LC
          << ", gc = kc ^ (kc >> 1);\n"
             "            tm &= tm - 1;\n"
             "            bool alive = true;\n";
        emit_sieve(o, sv[2], wb, y0, n, "gc", "            ");
        o << "            const unsigned long long lm = __builtin_amdgcn_ballot_w64(alive);\n"
             "            const unsigned at = __builtin_amdgcn_mbcnt_hi((unsigned)(lm >> 32), "
             "__builtin_amdgcn_mbcnt_lo((unsigned)lm, tail));\n"
             "            if (alive) queue[at & 127u] = hc;\n"
             "            tail += (unsigned)__builtin_popcountll(lm);\n"
             "        }\n"
             "        if (tail == head) break;\n"
             "        const unsigned count = min(64u, tail - head);\n"
             "        const unsigned long long h = queue[(head + min(lane, count - 1u)) & 127u];\n"
             "        head += count;\n"
             "        unsigned __int128 acc = 0;\n";
    }
    o << "        int ";
    for (int i = 0; i < n; ++i) o << "y" << i << " = " << lit(y0[i]) << (i + 1 < n ? ", " : ";\n");
    o << "        const unsigned long long k0 = h << L;\n"
         "        const unsigned long long g0 = k0 ^ (k0 >> 1);\n";
    // chunk-start rebuild: columns j >= L-1 whose bit is set in G(h 2^L)
    for (int j = 0; j < n - 1; ++j) {
        bool any = false;
        for (int r = 0; r < n; ++r) any = any || b[(size_t)r * n + j] != 0;
        if (!any) continue;
        o << "        { const int mk = -(int)(((g0 >> " << j << ") & 1ull) & (unsigned)(" << j << " >= L - 1));";
        for (int r = 0; r < n; ++r) {
            const int64_t d = wb[(size_t)r * n + j];
            if (d != 0) o << " y" << r << " += " << lit(d) << " & mk;";
        }
        o << " }\n";
    }
    o << "        int Z = 0";
    for (int i = 0; i < n; ++i)
        if (zr[i]) o << " + (y" << i << " == 0)";
    o << ";\n";
    o << "        const int lm = -(int)(h & 1ull);  // direction of column L-1: -1 = remove\n";
    o << "        const unsigned nblk = 1u << (L - " << U << ");\n"
         "        const unsigned half = nblk >> 1;\n";
    if (compact) {
        o << "        int Zm;  // the block's least Z\n";
        o << "        auto flipc = [&](unsigned c, int mk) __attribute__((always_inline)) {\n"
             "            switch (c) {\n";
        for (int c = 0; c < U; ++c) {
            o << "            case " << c << "u:\n";
            emit_flip_lane(o, wb, zr, n, c, "mk", "                ");
            o << "                break;\n";
        }
        o << "            default: break;\n"
             "            }\n"
             "        };\n";
        o << "        auto termc = [&](bool neg) __attribute__((always_inline)) {\n";
        emit_term(o, n, false, "            ", false, false, "neg");
        o << "        };\n";
    }
    // steps j = 1 .. 2^U - 1 of block m: compile-time columns ctz(j); the
    // direction of column U-1 is bit 0 of m
    auto block_tail = [&](const char* ind) {
        for (int j = 1; j < (1 << U); ++j) {
            const int c = __builtin_ctz(j);
            if (c + 1 < U) {
                const int sgn = ((j >> (c + 1)) & 1) ? -1 : 1;
                emit_flip_const(o, wb, zr, n, c, sgn, ind);
            } else {
                o << ind << "if (m & 1u) {\n";
                emit_flip_const(o, wb, zr, n, c, -1, (std::string(ind) + "    ").c_str());
                o << ind << "} else {\n";
                emit_flip_const(o, wb, zr, n, c, 1, (std::string(ind) + "    ").c_str());
                o << ind << "}\n";
            }
            emit_term(o, n, (j & 1) != 0, ind, compact);
        }
        if (compact) emit_block_replay(o, U, "m", ind);
    };
    o << "        {\n            const unsigned m = 0;\n";
    emit_term(o, n, false, "            ", compact, true);
    block_tail("            ");
    o << "        }\n";
    // block m first flips column U + ctz(m), in the block's direction
    // (bit ctz(m)+1 of m) or, at the middle block, each lane's: one mask,
    // so each column's flip is one branch-free path, found by testing the
    // bits of m from the lowest (half the blocks stop at the first test)
    o << "        for (unsigned m = 1; m < nblk; ++m) {\n"
         "            const int lmm = (m == half) ? lm : -(int)((m >> (__builtin_ctz(m) + 1)) & 1u);\n";
    const int flips = prune ? std::min(n - 1, kGenPruneChunk) : n - 1;  // m has L - U bits
    for (int c = U; c < flips && c - U < 32; ++c) {
        o << "            " << (c == U ? "if" : "} else if") << " (m & " << (1u << (c - U)) << "u) {\n";
        emit_flip_lane(o, wb, zr, n, c, "lmm", "                ");
    }
    if (U < n - 1) o << "            }\n";
    emit_term(o, n, false, "            ", compact, true);
    block_tail("            ");
    o << "        }\n";
    if (prune)
        o << "        if (lane < count) total += acc;\n"
             "    }\n"
             "    unsigned __int128 acc = total;\n";
    else
        o << "    }\n"
             "    if (idle) acc = 0;\n";
    o << "    unsigned long long lo = (unsigned long long)acc, hi = (unsigned long long)(acc >> 64);\n"
         "    for (int off = 32; off >= 1; off >>= 1) {\n"
         "        const unsigned long long olo = __shfl_xor(lo, off, 64);\n"
         "        const unsigned long long ohi = __shfl_xor(hi, off, 64);\n"
         "        const unsigned long long s = lo + olo;\n"
         "        hi = hi + ohi + (s < lo ? 1ull : 0ull);\n"
         "        lo = s;\n"
         "    }\n"
         "    const int w = threadIdx.x >> 6;\n"
         "    if ((threadIdx.x & 63u) == 0) { red[2 * w] = lo; red[2 * w + 1] = hi; }\n"
         "    __syncthreads();\n"
         "    if (threadIdx.x == 0) {\n"
         "        unsigned __int128 t = 0;\n"
         "        for (int i = 0; i < 4; ++i) t += ((unsigned __int128)red[2 * i + 1] << 64) | red[2 * i];\n"
         "        unsigned long long* out = partial + 2 * blockIdx.x;\n"
         "        if (accumulate) t += ((unsigned __int128)out[1] << 64) | out[0];\n"
         "        out[0] = (unsigned long long)t;\n"
         "        out[1] = (unsigned long long)(t >> 64);\n"
         "    }\n"
         "}\n";
    return o.str();
}

// ---------------------------------------------------------------------------
// Source emitter (real FP64 entries).
//
// The reference's generated kernels compute in FP64 with decimal literals
// printed by std::to_string (6 decimals, UTOrderedKernelCodeGen.cuh:292-295),
// exact only for dyadic values with few digits.  Here every literal is the
// hex-float spelling of the matrix entry (%a), so the kernel adds exactly the
// entry's binary64 value.  Exact zeros of x_i(S) need exact cancellation, so
// generic real matrices get no zero-count skip (integer-valued and row-scaled
// integer matrices take the exact integer kernels instead); what they get is
// a product that does not recompute the rows a flip cannot have changed:
//
//   R(c)  = the largest row any of columns 0..c touches (rows in UT order
//           are numbered as columns first touch them, so R grows slowly);
//   S_j   = prod_{r > R(j)} x_r, j = 0..J-1 (cached "suffix" products);
//   term  = (prod_{r <= R(0)} x_r) * S_0.
//
// Flipping column c changes rows <= R(c) only: S_j for j >= c stays valid,
// S_{c-1} .. S_0 are rebuilt from S_c (one level each), and a column c >= J
// rebuilds S_{J-1} from its rows first.  J is chosen per pattern to minimise
// the expected multiplies per step (column c flips every 2^(c+1) steps).
// ---------------------------------------------------------------------------
namespace {

std::string hexlit(double v)
{
    char buf[48];
    std::snprintf(buf, sizeof buf, "%a", v);
    return buf;
}

struct RealLevels {
    std::vector<int> R;  // R[c], c = 0..n-2 (-1: no row yet)
    int J = 1;
};

RealLevels real_levels(const std::vector<double>& b, int n)
{
    RealLevels lv;
    lv.R.assign(std::max(1, n - 1), -1);
    int cur = -1;
    for (int c = 0; c + 1 < n; ++c) {
        for (int r = 0; r < n; ++r)
            if (b[(size_t)r * n + c] != 0.0) cur = std::max(cur, r);
        lv.R[c] = cur;
    }
    if (n < 2) return lv;
    // expected multiplies per step for J levels (column c flips with
    // probability 2^-(c+1) per step; columns >= J rebuild the top level)
    auto cost = [&](int J) {
        const double R0 = lv.R[0];
        double e = R0 + 1.0;
        for (int c = 1; c < J && c < n - 1; ++c) e += std::ldexp(lv.R[c] - R0 + c, -(c + 1));
        const int top = lv.R[std::min(J, n - 1) - 1];
        e += std::ldexp((n - 1 - top) + (top - R0) + J - 1, -J);
        return e;
    };
    double best = 1e300;
    for (int J = 1; J <= std::min(8, n - 1); ++J) {
        const double e = cost(J);
        if (e < best - 1e-9) {
            best = e;
            lv.J = J;
        }
    }
    return lv;
}

// Product of x_lo .. x_hi (inclusive) as an expression in up to four
// independent chains ("1.0" when empty).
std::string prod_expr(int lo, int hi)
{
    if (hi < lo) return "1.0";
    const int k = hi - lo + 1;
    const int chains = k >= 8 ? 4 : k >= 4 ? 2 : 1;
    std::vector<std::string> ch(chains);
    for (int i = 0; i < k; ++i) {
        std::string& c = ch[i % chains];
        c += (c.empty() ? "" : " * ") + std::string("x") + std::to_string(lo + i);
    }
    std::string e;
    for (int i = 0; i < chains; ++i) e += (i ? " * (" : "(") + ch[i] + ")";
    return e;
}

// sgn 0: the per-lane sign in the variable `sign` (x += sign * d, exact for
// sign = +-1)
void emit_real_flip(std::ostringstream& o, const std::vector<double>& b, int n, int c, int sgn, const char* ind,
                    const char* sign = "sd")
{
    for (int r = 0; r < n; ++r) {
        const double d = b[(size_t)r * n + c];
        if (d == 0.0) continue;
        if (sgn == 0)
            o << ind << "x" << r << " = __builtin_fma(" << sign << ", " << hexlit(d) << ", x" << r << ");\n";
        else
            o << ind << "x" << r << " += " << hexlit(sgn > 0 ? d : -d) << ";\n";
    }
}

// S_{from-1} .. S_0 from S_from; from == J rebuilds S_{J-1} from its rows.
void emit_real_levels(std::ostringstream& o, const RealLevels& lv, int n, int from, const char* ind)
{
    const int J = lv.J;
    if (from >= J) {
        o << ind << "S" << J - 1 << " = " << prod_expr(lv.R[J - 1] + 1, n - 1) << ";\n";
        from = J - 1;
    }
    for (int j = from - 1; j >= 0; --j)
        o << ind << "S" << j << " = " << prod_expr(lv.R[j] + 1, lv.R[j + 1]) << " * S" << j + 1 << ";\n";
}

void emit_real_term(std::ostringstream& o, const RealLevels& lv, bool negative, const char* ind)
{
    o << ind << "{ const double P = " << prod_expr(0, lv.R[0]) << "; blk = __builtin_fma(" << (negative ? "-P" : "P")
      << ", S0, blk); ba = __builtin_fma(__builtin_fabs(P), __builtin_fabs(S0), ba); }\n";
}

// ---------------------------------------------------------------------------
// Inner columns summed out.  With the columns >= m set, the sum over all
// settings T of columns 0..m-1,
//   E = sum_T (-1)^|T| prod_r x_r(T),
// is a sum over m binary variables of a product of one factor per row, each
// depending only on the few inner columns its row has entries in.  It is
// formed one column at a time: the factors with column c are multiplied into
// one table over their other columns and c's two settings subtracted.  The
// cost grows with the tables (2^w entries, w columns tied together by shared
// rows), not with 2^m: order 36 with 5 entries per row sums 2^11 subsets in
// about 600 operations, 0.3 per subset against 9 for the walk.  The same
// tables of absolute values, added instead of subtracted, give sum |term|;
// a product of rows alone shares its value (|ab| = |a||b| as rounded).
// E is formed in FP64 under either precision (compensated sums begin with the
// outer steps): it has far fewer roundings than the 2^m terms it replaces, and
// against 80-bit values the results of 88 matrices (orders 26 to 38, 3 to 7
// entries per row) are off by 0.2 of what the walk's are, geometric mean.
// ---------------------------------------------------------------------------
struct Factor {
    std::vector<int> scope;  // columns, ascending; entry i has column scope[k] set when bit k of i is
    std::vector<std::string> val, abs;
    bool pure = true;        // a product of rows: abs is |val|
    int row = -1;            // a single row's, not written out yet (val and abs empty)
};

class Eliminator {
public:
    Eliminator(const std::vector<double>& b, int n, int m) : b_(b), n_(n), m_(m) {}

    // Emits E into `P` and its absolute sum into `A`; without `code` it only
    // counts.  False when an inner column is empty, or as soon as the code
    // passes max_ops instructions or the tables max_peak values.  ops: FP64
    // instructions; peak: table entries alive.
    bool run(int& ops, int& peak, int max_ops, int max_peak, std::string* code = nullptr, const char* ind = "")
    {
        ops = peak = 0;
        max_ops_ = max_ops;
        emit_ = code != nullptr;
        ind_ = ind;
        std::vector<Factor> fs;
        for (int r = 0; r < n_; ++r) {
            Factor f;
            f.row = r;
            for (int c = 0; c < m_; ++c)
                if (b_[(size_t)r * n_ + c] != 0.0) f.scope.push_back(c);
            if (!f.scope.empty()) fs.push_back(std::move(f));
        }
        std::vector<int> left(m_);
        for (int c = 0; c < m_; ++c) left[c] = c;
        while (!left.empty()) {
            size_t pick = 0, least = 99;
            for (size_t i = 0; i < left.size(); ++i) {  // the column whose rows tie the fewest others
                std::vector<int> u;
                for (const Factor& f : fs)
                    if (has(f, left[i])) u = unite(u, f.scope);
                if (u.empty()) return false;
                if (u.size() < least) {
                    least = u.size();
                    pick = i;
                }
            }
            const int c = left[pick];
            left.erase(left.begin() + pick);
            std::vector<Factor> with, rest;
            for (Factor& f : fs) {
                if (has(f, c) && !write_row(f, ops)) return false;
                (has(f, c) ? with : rest).push_back(std::move(f));
            }
            while (with.size() > 2) {  // the pair with the smallest common scope first
                size_t bi = 1, bj = 0, bs = 99;
                for (size_t i = 1; i < with.size(); ++i)
                    for (size_t j = 0; j < i; ++j) {
                        const size_t w = unite(with[i].scope, with[j].scope).size();
                        if (w < bs) {
                            bs = w;
                            bi = i;
                            bj = j;
                        }
                    }
                Factor f;
                if (!multiply(with[bj], with[bi], ops, f)) return false;
                with.erase(with.begin() + bi);
                with[bj] = std::move(f);
            }
            rest.emplace_back();
            if (!sum_out(with, c, ops, rest.back())) return false;
            fs = std::move(rest);
            int alive = 0;
            for (const Factor& f : fs) alive += (f.pure ? 1 : 2) * (int)f.val.size();  // (unwritten rows: none)
            peak = std::max(peak, alive);
            if (peak > max_peak) return false;
        }
        ops += 2 * (int)fs.size();
        if (ops > max_ops || !code) return ops <= max_ops;
        std::string P, A;
        for (const Factor& f : fs) {
            P += (P.empty() ? "" : " * ") + f.val[0];
            A += (A.empty() ? "" : " * ") + f.abs[0];
        }
        line("const double P = " + P + ", A = " + A + ";");
        *code = out_.str();
        return true;
    }

private:
    static bool has(const Factor& f, int c) { return std::find(f.scope.begin(), f.scope.end(), c) != f.scope.end(); }
    static std::vector<int> unite(const std::vector<int>& a, const std::vector<int>& b)
    {
        std::vector<int> u;
        std::set_union(a.begin(), a.end(), b.begin(), b.end(), std::back_inserter(u));
        return u;
    }
    // Index into f of the setting `i` over `scope` (a superset of f's).
    static size_t project(const Factor& f, const std::vector<int>& scope, size_t i)
    {
        size_t k = 0;
        for (size_t p = 0; p < f.scope.size(); ++p) {
            const size_t at = std::lower_bound(scope.begin(), scope.end(), f.scope[p]) - scope.begin();
            k |= ((i >> at) & 1u) << p;
        }
        return k;
    }
    void line(const std::string& t) { out_ << ind_ << t << "\n"; }
    std::string fresh(const char* stem) { return stem + std::to_string(id_++); }
    static std::string fabs(const std::string& v) { return "__builtin_fabs(" + v + ")"; }
    // `count` more instructions, if they are within the limit: asked before a
    // table is written, which has 2^scope entries (rows of 40 entries at m = 16
    // spelled out took 8 s and 0.5 GB before the limits were looked at).
    bool take(int& ops, size_t count)
    {
        if (count > (size_t)(max_ops_ - ops)) return false;
        ops += (int)count;
        return true;
    }

    bool write_row(Factor& f, int& ops)
    {
        if (f.row < 0) return true;
        const size_t entries = size_t(1) << f.scope.size();
        if (!take(ops, entries - 1)) return false;
        if (emit_) {
            f.val.push_back("x" + std::to_string(f.row));
            for (size_t k = 0; k < f.scope.size(); ++k)
                for (size_t i = 0, end = size_t(1) << k; i < end; ++i) {
                    const std::string v = fresh("v");
                    line("const double " + v + " = " + f.val[i] + " + " + hexlit(b_[(size_t)f.row * n_ + f.scope[k]]) +
                         ";");
                    f.val.push_back(v);
                }
            for (const std::string& v : f.val) f.abs.push_back(fabs(v));
        } else {
            f.val.resize(entries);
        }
        f.row = -1;
        return true;
    }
    bool multiply(const Factor& f, const Factor& g, int& ops, Factor& h)
    {
        h.scope = unite(f.scope, g.scope);
        h.pure = f.pure && g.pure;
        const size_t entries = size_t(1) << h.scope.size();
        if (!take(ops, (h.pure ? 1 : 2) * entries)) return false;
        if (!emit_) {
            h.val.resize(entries);
            return true;
        }
        for (size_t i = 0; i < entries; ++i) {
            const size_t fi = project(f, h.scope, i), gi = project(g, h.scope, i);
            const std::string v = fresh("p");
            line("const double " + v + " = " + f.val[fi] + " * " + g.val[gi] + ";");
            h.val.push_back(v);
            if (h.pure) {
                h.abs.push_back(fabs(v));
            } else {
                const std::string u = fresh("q");
                line("const double " + u + " = " + f.abs[fi] + " * " + g.abs[gi] + ";");
                h.abs.push_back(u);
            }
        }
        return true;
    }
    bool sum_out(const std::vector<Factor>& fs, int c, int& ops, Factor& h)
    {
        const std::vector<int> scope = fs.size() == 2 ? unite(fs[0].scope, fs[1].scope) : fs[0].scope;
        const size_t at = std::lower_bound(scope.begin(), scope.end(), c) - scope.begin();
        const bool pure = fs.size() == 2 && fs[0].pure && fs[1].pure;
        h.pure = false;
        for (int s : scope)
            if (s != c) h.scope.push_back(s);
        const size_t entries = size_t(1) << h.scope.size();
        if (!take(ops, (fs.size() == 1 ? 2 : pure ? 3 : 4) * entries)) return false;
        if (!emit_) {
            h.val.resize(entries);
            return true;
        }
        for (size_t i = 0; i < entries; ++i) {
            const size_t i0 = ((i >> at) << (at + 1)) | (i & ((size_t(1) << at) - 1)), i1 = i0 | (size_t(1) << at);
            const std::string v = fresh("t"), u = fresh("u");
            const Factor& f = fs[0];
            const size_t f0 = project(f, scope, i0), f1 = project(f, scope, i1);
            if (fs.size() == 1) {
                line("const double " + v + " = " + f.val[f0] + " - " + f.val[f1] + ";");
                line("const double " + u + " = " + f.abs[f0] + " + " + f.abs[f1] + ";");
            } else {
                const Factor& g = fs[1];
                const size_t g0 = project(g, scope, i0), g1 = project(g, scope, i1);
                const std::string p = fresh("p");
                line("const double " + p + " = " + f.val[f0] + " * " + g.val[g0] + ";");
                line("const double " + v + " = __builtin_fma(-" + f.val[f1] + ", " + g.val[g1] + ", " + p + ");");
                std::string q = fabs(p);
                if (!pure) {
                    q = fresh("q");
                    line("const double " + q + " = " + f.abs[f0] + " * " + g.abs[g0] + ";");
                }
                line("const double " + u + " = __builtin_fma(" + f.abs[f1] + ", " + g.abs[g1] + ", " + q + ");");
            }
            h.val.push_back(v);
            h.abs.push_back(u);
        }
        return true;
    }

    const std::vector<double>& b_;
    int n_, m_;
    const char* ind_ = "";
    bool emit_ = false;
    int max_ops_ = 0;
    int id_ = 0;
    std::ostringstream out_;
};

}  // namespace

// The end of a real kernel: the chunk's sums into the lane's, and the block's
// record.
static void emit_real_tail(std::ostringstream& o)
{
    o << "        if (h < num_chunks) { ddadd(a_hi, a_lo, t_hi, t_lo); a_abs += t_abs; }\n"
         "    }\n"
         "    for (int off = 32; off >= 1; off >>= 1) {\n"
         "        const double oh = __shfl_xor(a_hi, off, 64), ol = __shfl_xor(a_lo, off, 64);\n"
         "        const double oa = __shfl_xor(a_abs, off, 64);\n"
         "        ddadd(a_hi, a_lo, oh, ol);\n"
         "        a_abs += oa;\n"
         "    }\n"
         "    const int w = threadIdx.x >> 6;\n"
         "    if (lane == 0) { red[3 * w] = a_hi; red[3 * w + 1] = a_lo; red[3 * w + 2] = a_abs; }\n"
         "    __syncthreads();\n"
         "    if (threadIdx.x == 0) {\n"
         "        double hh = red[0], ll = red[1], aa = red[2];\n"
         "        for (int i = 1; i < 4; ++i) { ddadd(hh, ll, red[3 * i], red[3 * i + 1]); aa += red[3 * i + 2]; }\n"
         "        double* out = partial + 4 * blockIdx.x;\n"
         "        if (accumulate) { ddadd(hh, ll, out[0], out[1]); aa += out[2]; }\n"
         "        out[0] = hh; out[1] = ll; out[2] = aa; out[3] = 0.0;\n"
         "    }\n"
         "}\n";
}

constexpr int kElimOps = 1000, kElimPeak = 128;

// The number m of inner columns to sum out: the least operations per subset
// among those whose code stays within kElimOps instructions (compile time)
// and whose tables within kElimPeak values, leaving at least 2^19 outer
// settings to share out.  0: walk.  The kernels take up to 512 VGPRs, one
// wave per SIMD: straight-line code has its own parallelism, and at two
// waves (256 VGPRs) the larger ones spill (order 38, 7 per row 6.0 -> 7.4 ms,
// at three 20 ms).  Kernel ms of the walk and at limits of 700 operations with
// 64 values, then 1000 with 128, three N(0,1) matrices each: order 30 with 7 per
// row 0.22-0.24, 0.04-0.09, 0.03-0.06; order 36 with 5 6.5-8.5, 0.06-0.26,
// 0.03-0.18; order 38 with 7 36-39, 2.1-9.5, 2.1-4.3; order 40 with 8 175-191,
// 40-67, 36-57 (1200 operations: the same but for one matrix).  A plan of such
// a kernel takes 0.24-0.37 s, of a walk 0.25-0.33.  Below order 26 a walk takes
// 0.02 ms.
int real_elim_columns(const double* b, int n)
{
    if (n < 26) return 0;
    const std::vector<double> v(b, b + (size_t)n * n);
    int best = 0;
    double least = 1e300;
    for (int m = 3; m <= std::min(16, n - 20); ++m) {
        int ops = 0, peak = 0, outer = 0;
        if (!Eliminator(v, n, m).run(ops, peak, kElimOps, kElimPeak)) continue;
        for (int r = 0; r < n; ++r) {
            bool in = false;
            for (int c = 0; c < m; ++c) in = in || b[(size_t)r * n + c] != 0.0;
            outer += in ? 0 : 1;
        }
        const double cost = std::ldexp(ops + outer + 16.0, -m);
        if (cost < least) {
            least = cost;
            best = m;
        }
    }
    return least < 4.0 ? best : 0;  // the walk takes 4-10 instructions per subset
}

static std::string emit_real_elim_kernel(const std::vector<double>& b, int n, bool compensated,
                                         const std::string& name, int m)
{
    std::vector<double> x0(n);
    for (int i = 0; i < n; ++i) {  // as emit_real_kernel
        double rs = 0.0;
        for (int j = 0; j < n; ++j) rs += b[(size_t)i * n + j];
        x0[i] = b[(size_t)i * n + n - 1] - rs / 2;
    }
    int ops = 0, peak = 0;
    std::string inner;
    Eliminator(b, n, m).run(ops, peak, kElimOps, kElimPeak, &inner, "            ");
    std::ostringstream o;
    o << "// generated: SpaRyser kernel for one " << n << "x" << n << " real matrix (FP64, "
      << (compensated ? "compensated" : "plain") << " sums, " << m << " inner columns summed out in " << ops
      << " operations)\n";
    o << "static __device__ __forceinline__ void ts(double a, double b, double& s, double& e)\n"
         "{ s = a + b; const double bb = s - a; e = (a - (s - bb)) + (b - bb); }\n"
         "static __device__ __forceinline__ void ddadd(double& ah, double& al, double bh, double bl)\n"
         "{ double s, e; ts(ah, bh, s, e); e += al + bl; ah = s + e; al = e - (ah - s); }\n";
    o << "extern \"C\" __global__ void __launch_bounds__(256)\n" << name
      << "(double* __restrict__ partial, unsigned long long task_begin,\n"
         "    unsigned long long task_end, unsigned long long num_chunks, int L, int accumulate)\n{\n";
    o << "    __shared__ double red[12];\n"
         "    const unsigned lane = threadIdx.x & 63u;\n"
         "    const unsigned long long wave = (unsigned long long)blockIdx.x * 4 + (threadIdx.x >> 6);\n"
         "    const unsigned long long nwave = (unsigned long long)gridDim.x * 4;\n"
         "    const int Lo = L - " << m << ";  // a chunk's outer steps, over columns " << m << ".. in Gray order\n"
         "    double a_hi = 0.0, a_lo = 0.0, a_abs = 0.0;\n"
         "    for (unsigned long long task = task_begin + wave; task < task_end; task += nwave) {\n"
         "        const unsigned long long h = task * 64 + lane;\n";
    o << "        double ";
    for (int i = 0; i < n; ++i) o << "x" << i << " = " << hexlit(x0[i]) << (i + 1 < n ? ", " : ";\n");
    o << "        const unsigned long long k0 = h << Lo;\n"
         "        const unsigned long long g0 = k0 ^ (k0 >> 1);\n";
    for (int j = m; j < n - 1; ++j) {
        bool any = false;
        for (int r = 0; r < n; ++r) any = any || b[(size_t)r * n + j] != 0.0;
        if (!any) continue;
        o << "        { const double bj = ((((g0 >> " << j - m << ") & 1ull) != 0ull) && (" << j - m
          << " >= Lo - 1)) ? 1.0 : 0.0;";
        for (int r = 0; r < n; ++r) {
            const double d = b[(size_t)r * n + j];
            if (d != 0.0) o << " x" << r << " = __builtin_fma(bj, " << hexlit(d) << ", x" << r << ");";
        }
        o << " }\n";
    }
    o << "        const double sd = (h & 1ull) ? -1.0 : 1.0;  // direction of the last outer column\n"
         "        double t_hi = 0.0, t_lo = 0.0, t_abs = 0.0, blk = 0.0, ba = 0.0;\n"
         "        const unsigned steps = 1u << Lo, half = steps >> 1;\n"
         "#pragma nounroll\n"
         "        for (unsigned s = 0;;) {\n";
    o << inner;
    std::vector<std::string> chain(4);
    int k = 0;
    for (int r = 0; r < n; ++r) {
        bool in = false;
        for (int c = 0; c < m; ++c) in = in || b[(size_t)r * n + c] != 0.0;
        if (in) continue;
        std::string& c = chain[k++ % 4];
        c += (c.empty() ? "x" : " * x") + std::to_string(r);
    }
    std::string prod;
    for (const std::string& c : chain)
        if (!c.empty()) prod += (prod.empty() ? "(" : " * (") + c + ")";
    o << "            const double S = " << (prod.empty() ? "1.0" : prod) << ";\n"
         "            blk = __builtin_fma((s & 1u) ? -P : P, S, blk);\n"
         "            ba = __builtin_fma(A, __builtin_fabs(S), ba);\n"
         "            ++s;\n"
         "            if ((s & 3u) == 0u || s == steps) "
      << (compensated ? "{ double s_, e_; ts(t_hi, blk, s_, e_); t_hi = s_; t_lo += e_; t_abs += ba; blk = 0.0; ba = 0.0; }\n"
                      : "{ t_hi += blk; t_abs += ba; blk = 0.0; ba = 0.0; }\n")
      << "            if (s == steps) break;\n"
         "            const double sdm = (s == half) ? sd : (((s >> (__builtin_ctz(s) + 1)) & 1u) ? -1.0 : 1.0);\n";
    for (int c = m; c < n - 1 && c - m < 16; ++c) {
        o << "            " << (c == m ? "if" : "} else if") << " (s & " << (1u << (c - m)) << "u) {\n";
        emit_real_flip(o, b, n, c, 0, "                ", "sdm");
    }
    o << "            }\n"
         "        }\n";
    emit_real_tail(o);
    return o.str();
}

std::string emit_real_kernel(const std::vector<double>& b, int n, bool compensated, const std::string& name, int elim)
{
    if (elim > 0) return emit_real_elim_kernel(b, n, compensated, name, elim);
    const int U = gen_unroll_bits_real(n);
    const RealLevels lv = real_levels(b, n);
    std::vector<double> x0(n);
    for (int i = 0; i < n; ++i) {  // x(empty set) with the left-to-right row sum (dpSingleGPU.cuh:62-74)
        double rs = 0.0;
        for (int j = 0; j < n; ++j) rs += b[(size_t)i * n + j];
        x0[i] = b[(size_t)i * n + n - 1] - rs / 2;
    }
    std::ostringstream o;
    o << "// generated: SpaRyser kernel for one " << n << "x" << n << " real matrix (FP64, "
      << (compensated ? "compensated" : "plain") << " sums, " << lv.J << " suffix-product levels)\n";
    o << "static __device__ __forceinline__ void ts(double a, double b, double& s, double& e)\n"
         "{ s = a + b; const double bb = s - a; e = (a - (s - bb)) + (b - bb); }\n"
         "static __device__ __forceinline__ void ddadd(double& ah, double& al, double bh, double bl)\n"
         "{ double s, e; ts(ah, bh, s, e); e += al + bl; ah = s + e; al = e - (ah - s); }\n";
    o << "extern \"C\" __global__ void __launch_bounds__(256)";
    if (const int w = gen_real_waves_per_simd(n)) o << " __attribute__((amdgpu_waves_per_eu(" << w << ")))";
    o << "\n" << name
      << "(double* __restrict__ partial, unsigned long long task_begin,\n"
         "    unsigned long long task_end, unsigned long long num_chunks, int L, int accumulate)\n{\n";
    o << "    __shared__ double red[12];\n"
         "    const unsigned lane = threadIdx.x & 63u;\n"
         "    const unsigned long long wave = (unsigned long long)blockIdx.x * 4 + (threadIdx.x >> 6);\n"
         "    const unsigned long long nwave = (unsigned long long)gridDim.x * 4;\n"
         "    double a_hi = 0.0, a_lo = 0.0, a_abs = 0.0;\n"
         "    for (unsigned long long task = task_begin + wave; task < task_end; task += nwave) {\n"
         "        const unsigned long long h = task * 64 + lane;\n";
    o << "        double ";
    for (int i = 0; i < n; ++i) o << "x" << i << " = " << hexlit(x0[i]) << (i + 1 < n ? ", " : ";\n");
    o << "        const unsigned long long k0 = h << L;\n"
         "        const unsigned long long g0 = k0 ^ (k0 >> 1);\n";
    // chunk-start rebuild in ascending column order (DenseKernelDefinitions.cuh:230-240)
    for (int j = 0; j < n - 1; ++j) {
        bool any = false;
        for (int r = 0; r < n; ++r) any = any || b[(size_t)r * n + j] != 0.0;
        if (!any) continue;
        o << "        { const double bj = ((((g0 >> " << j << ") & 1ull) != 0ull) && (" << j
          << " >= L - 1)) ? 1.0 : 0.0;";
        for (int r = 0; r < n; ++r) {
            const double d = b[(size_t)r * n + j];
            if (d != 0.0) o << " x" << r << " = __builtin_fma(bj, " << hexlit(d) << ", x" << r << ");";
        }
        o << " }\n";
    }
    o << "        double ";
    for (int j = 0; j < lv.J; ++j) o << "S" << j << (j + 1 < lv.J ? ", " : ";\n");
    emit_real_levels(o, lv, n, lv.J, "        ");
    o << "        const double sd = (h & 1ull) ? -1.0 : 1.0;  // direction of column L-1\n"
         "        double t_hi = 0.0, t_lo = 0.0, t_abs = 0.0, blk = 0.0, ba = 0.0;\n";
    o << "        const unsigned nblk = 1u << (L - " << U << ");\n"
         "        const unsigned half = nblk >> 1;\n";
    const std::string fold = compensated
        ? "{ double s_, e_; ts(t_hi, blk, s_, e_); t_hi = s_; t_lo += e_; t_abs += ba; blk = 0.0; ba = 0.0; }\n"
        : "{ t_hi += blk; t_abs += ba; blk = 0.0; ba = 0.0; }\n";
    auto flip = [&](int c, int sgn, const char* ind) {
        emit_real_flip(o, b, n, c, sgn, ind);
        if (c > 0) emit_real_levels(o, lv, n, c, ind);
    };
    auto block_tail = [&](const char* ind) {
        for (int j = 1; j < (1 << U); ++j) {
            const int c = __builtin_ctz(j);
            if (c + 1 < U) {
                flip(c, ((j >> (c + 1)) & 1) ? -1 : 1, ind);
            } else {
                o << ind << "if (m & 1u) {\n";
                flip(c, -1, (std::string(ind) + "    ").c_str());
                o << ind << "} else {\n";
                flip(c, 1, (std::string(ind) + "    ").c_str());
                o << ind << "}\n";
            }
            emit_real_term(o, lv, (j & 1) != 0, ind);
        }
        o << ind << fold;
    };
    o << "        {\n            const unsigned m = 0;\n";
    emit_real_term(o, lv, false, "            ");
    block_tail("            ");
    o << "        }\n";
    // as in the integer kernels: one per-lane sign and a chain of bit tests
    o << "        for (unsigned m = 1; m < nblk; ++m) {\n"
         "            const double sdm = (m == half) ? sd : (((m >> (__builtin_ctz(m) + 1)) & 1u) ? -1.0 : 1.0);\n";
    for (int c = U; c < n - 1 && c - U < 32; ++c) {
        o << "            " << (c == U ? "if" : "} else if") << " (m & " << (1u << (c - U)) << "u) {\n";
        emit_real_flip(o, b, n, c, 0, "                ", "sdm");
        if (c > 0) emit_real_levels(o, lv, n, c, "                ");
    }
    if (U < n - 1) o << "            }\n";
    emit_real_term(o, lv, false, "            ");
    block_tail("            ");
    o << "        }\n";
    emit_real_tail(o);
    return o.str();
}

int real_levels_count(const std::vector<double>& b, int n) { return real_levels(b, n).J; }

// FNV-1a over the values' bit patterns and the generator options.
uint64_t real_pattern_hash(const double* b, int n, int options, int precision)
{
    uint64_t h = 1469598103934665603ull ^ 0x5a5a5a5a5a5a5a5aull;
    auto mix = [&](uint64_t v) {
        for (int k = 0; k < 8; ++k) {
            h ^= (v >> (8 * k)) & 0xff;
            h *= 1099511628211ull;
        }
    };
    mix((uint64_t)n);
    mix((uint64_t)options);
    mix((uint64_t)precision);
    mix((uint64_t)gen_unroll_bits_real(n));
    for (int e = 0; e < n * n; ++e) {
        uint64_t w;
        std::memcpy(&w, b + e, 8);
        mix(w);
    }
    return h;
}

// Whether an integer kernel is pruned: when the rows fixed outside a chunk
// leave less than a quarter of the chunks live (by the row-independence
// estimate; above that the sieves save less than walking 64 chunks that all
// meet nonzero terms costs), and there are blocks of 64 tasks to share out.
// Kernel ms at order 36 with 4, 6 and 8 entries per row and order 40 with 4
// and 8 (0/1): unpruned 5.0 / 19 / 79 / 55 / 560, pruned 0.077 / 0.48 / 2.9 /
// 0.106 / 12.1; order 24 with 4: 0.029 and 0.023.  The chunks are short (2^5
// steps in blocks of 2^2): chunks of 2^9 took 3-5x as long, 2^7 1.3-1.9x, since
// the less of a chunk is walked blind the fewer waves form a product for one
// lane.
bool gen_pruned(const int64_t* b, int n)
{
    if (n < 24) return false;  // 0.02 ms either way
    double live = 1.0;
    for (int r = 0; r < n; ++r) {
        int64_t sum = 0;
        int k = 0, low = n;
        for (int c = n - 1; c >= 0; --c) {
            sum += b[(size_t)r * n + c];
            if (c < n - 1 && b[(size_t)r * n + c] != 0) {
                ++k;
                low = c;
            }
        }
        if ((sum & 1) != 0 || low < kGenPruneChunk) continue;
        double p = 1.0;  // C(k, floor(k/2)) / 2^k
        for (int t = 1; t <= k; ++t) p *= (t <= k / 2 ? double(k - k / 2 + t) / t : 1.0) * 0.5;
        live *= 1.0 - std::min(1.0, p);
    }
    return live < 0.25;
}
int codegen_real_unroll_bits(int n) { return gen_unroll_bits_real(n); }
bool gen_compact_term(const int64_t* b, int n) { return int_nonzero_term_fraction(b, n) < kGenCompactTermQ; }
int codegen_int_unroll_bits(const int64_t* b, int n)
{
    if (gen_pruned(b, n)) return kGenPruneUnroll;
    return gen_unroll_bits_int(n, gen_compact_term(b, n));
}

// FNV-1a over the pattern, values and generator options.
uint64_t pattern_hash(const int64_t* b, int n, int options)
{
    uint64_t h = 1469598103934665603ull;
    auto mix = [&](uint64_t v) {
        for (int k = 0; k < 8; ++k) {
            h ^= (v >> (8 * k)) & 0xff;
            h *= 1099511628211ull;
        }
    };
    mix((uint64_t)n);
    mix((uint64_t)options);
    mix((uint64_t)codegen_int_unroll_bits(b, n));
    mix((uint64_t)gen_compact_term(b, n));
    for (int e = 0; e < n * n; ++e) mix((uint64_t)b[e]);
    return h;
}

// ---------------------------------------------------------------------------
// hiprtc compile and per-device module cache
// ---------------------------------------------------------------------------
namespace {
struct CachedKernel {
    hipModule_t module = nullptr;
    hipFunction_t fn = nullptr;
    double compile_s = 0;
};
std::mutex g_cg_mu;
std::map<std::pair<int, uint64_t>, CachedKernel> g_cg_cache;
const char* const kRtcOpts[] = {"--offload-arch=gfx950", "-O3", "-std=c++17",
                                "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"};
constexpr int kRtcOptCount = (int)(sizeof kRtcOpts / sizeof kRtcOpts[0]);
}  // namespace

int rtc_compile(const std::string& src, const std::string& name, std::vector<char>& code, std::string& log)
{
    hiprtcProgram prog;
    if (hiprtcCreateProgram(&prog, src.c_str(), (name + ".hip").c_str(), 0, nullptr, nullptr) != HIPRTC_SUCCESS)
        return SPM_ECOMPILE;
    const hiprtcResult rc = hiprtcCompileProgram(prog, kRtcOptCount, const_cast<const char**>(kRtcOpts));
    size_t ls = 0;
    hiprtcGetProgramLogSize(prog, &ls);
    log.assign(ls, '\0');
    if (ls) hiprtcGetProgramLog(prog, &log[0]);
    if (rc != HIPRTC_SUCCESS) {
        hiprtcDestroyProgram(&prog);
        return SPM_ECOMPILE;
    }
    size_t cs = 0;
    hiprtcGetCodeSize(prog, &cs);
    code.resize(cs);
    hiprtcGetCode(prog, code.data());
    hiprtcDestroyProgram(&prog);
    return SPM_OK;
}

int codegen_compile_only(const std::string& src, const std::string& name, double* seconds, size_t* code_bytes)
{
    const double t0 = now_seconds();
    std::vector<char> code;
    std::string log;
    const int st = rtc_compile(src, name, code, log);
    if (st != SPM_OK) std::fprintf(stderr, "superman_amd: hiprtc failed for %s:\n%s\n", name.c_str(), log.c_str());
    if (seconds) *seconds = now_seconds() - t0;
    if (code_bytes) *code_bytes = code.size();
    return st;
}

// ---------------------------------------------------------------------------
// On-disk code objects.  Directory: $SPM_KERNEL_CACHE ("" or "0" turns the
// disk cache off), else $XDG_CACHE_HOME/superman_amd, else
// $HOME/.cache/superman_amd.  A file is <kernel name>-<FNV-1a of the source
// and the compile options>.co, so a changed generator or option never
// reuses an old object; it is written under a temporary name and renamed,
// so a reader sees a whole file or none, and one that fails to load is
// compiled again.  Any filesystem failure only means no disk cache.
// ---------------------------------------------------------------------------
namespace {

std::string disk_cache_dir()
{
    const char* e = std::getenv("SPM_KERNEL_CACHE");
    if (e) return (e[0] == 0 || (e[0] == '0' && e[1] == 0)) ? std::string() : std::string(e);
    if (const char* x = std::getenv("XDG_CACHE_HOME"); x && x[0]) return std::string(x) + "/superman_amd";
    if (const char* h = std::getenv("HOME"); h && h[0]) return std::string(h) + "/.cache/superman_amd";
    return std::string();
}

std::string disk_cache_path(const std::string& src, const std::string& name)
{
    const std::string dir = disk_cache_dir();
    if (dir.empty()) return std::string();
    uint64_t h = 1469598103934665603ull;
    auto mix = [&](const char* s) {
        for (const char* c = s; *c; ++c) {
            h ^= (unsigned char)*c;
            h *= 1099511628211ull;
        }
        h ^= 0xff;  // separator
        h *= 1099511628211ull;
    };
    mix(src.c_str());
    for (int k = 0; k < kRtcOptCount; ++k) mix(kRtcOpts[k]);
    char tail[40];
    std::snprintf(tail, sizeof tail, "-%016llx.co", (unsigned long long)h);
    return dir + "/" + name + tail;
}

bool disk_load(const std::string& path, std::vector<char>& code)
{
    if (path.empty()) return false;
    FILE* f = std::fopen(path.c_str(), "rb");
    if (!f) return false;
    std::fseek(f, 0, SEEK_END);
    const long sz = std::ftell(f);
    std::fseek(f, 0, SEEK_SET);
    bool ok = sz > 0;
    if (ok) {
        code.resize((size_t)sz);
        ok = std::fread(code.data(), 1, (size_t)sz, f) == (size_t)sz;
    }
    std::fclose(f);
    return ok;
}

void disk_store(const std::string& path, const std::vector<char>& code)
{
    if (path.empty() || code.empty()) return;
    const std::string dir = path.substr(0, path.rfind('/'));
    for (size_t p = 1; p <= dir.size(); ++p)  // mkdir -p
        if (p == dir.size() || dir[p] == '/') (void)::mkdir(dir.substr(0, p).c_str(), 0755);
    char tmp[32];
    std::snprintf(tmp, sizeof tmp, ".tmp%d", (int)::getpid());
    const std::string t = path + tmp;
    FILE* f = std::fopen(t.c_str(), "wb");
    if (!f) return;
    const bool ok = std::fwrite(code.data(), 1, code.size(), f) == code.size();
    if (std::fclose(f) != 0 || !ok || std::rename(t.c_str(), path.c_str()) != 0) (void)std::remove(t.c_str());
}

}  // namespace

bool codegen_is_cached(int device, uint64_t hash, const std::string& src, const std::string& name)
{
    {
        std::lock_guard<std::mutex> lk(g_cg_mu);
        if (g_cg_cache.count({device, hash})) return true;
    }
    const std::string path = disk_cache_path(src, name);
    struct stat st;
    return !path.empty() && ::stat(path.c_str(), &st) == 0 && st.st_size > 0;
}

int codegen_get_kernel(int device, uint64_t hash, const std::string& src, const std::string& name, hipFunction_t* fn,
                       double* compile_s, bool* cached)
{
    std::lock_guard<std::mutex> lk(g_cg_mu);
    auto it = g_cg_cache.find({device, hash});
    if (it != g_cg_cache.end()) {
        *fn = it->second.fn;
        *compile_s = it->second.compile_s;
        *cached = true;
        return SPM_OK;
    }
    const double t0 = now_seconds();
    const std::string path = disk_cache_path(src, name);
    std::vector<char> code;
    CachedKernel ck;
    if (disk_load(path, code) && hipModuleLoadData(&ck.module, code.data()) == hipSuccess) {
        if (hipModuleGetFunction(&ck.fn, ck.module, name.c_str()) == hipSuccess) {
            ck.compile_s = now_seconds() - t0;  // a load, not a compile
            g_cg_cache[{device, hash}] = ck;
            *fn = ck.fn;
            *compile_s = ck.compile_s;
            *cached = false;
            return SPM_OK;
        }
        (void)hipModuleUnload(ck.module);
        ck = CachedKernel();
    }
    code.clear();
    std::string log;
    int st = rtc_compile(src, name, code, log);
    if (st != SPM_OK) {
        std::fprintf(stderr, "superman_amd: hiprtc failed for %s:\n%s\n", name.c_str(), log.c_str());
        return st;
    }
    disk_store(path, code);
    if (hipModuleLoadData(&ck.module, code.data()) != hipSuccess) return SPM_EHIP;
    if (hipModuleGetFunction(&ck.fn, ck.module, name.c_str()) != hipSuccess) return SPM_EHIP;
    ck.compile_s = now_seconds() - t0;
    g_cg_cache[{device, hash}] = ck;
    *fn = ck.fn;
    *compile_s = ck.compile_s;
    *cached = false;
    return SPM_OK;
}

}  // namespace spm
