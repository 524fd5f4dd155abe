// int_prune.hip -- single-matrix exact integer Ryser kernel over the subsets
// with no zero row (walk_prune.h has the method; prune_plan in prune.cpp lays
// out the matrix for it).
//
// What bounds it: VALU issue on the surviving nodes (about 5 instructions
// per testable row and node of 4096 subsets) and terms (at order 30 about 105
// instructions per 64 terms and 9 for each round of the queue); no memory but
// the tables (10 to 60 KB, once per block).  Half 0/1 order 30, a run: 247 to 312
// us over four matrices with 15 to 18 even rows.
#include "walk_prune.h"

namespace spm {
namespace prune {

// The tables that every block of the walk keeps in LDS, once in memory: built
// by each block itself (200 instructions an entry of a zero mask, the columns'
// fields from memory one after another) they took 13 to 18 us of every launch.
//   group g, setting s -> packed sum of its columns' fields;
//   row r (field r of the packed vector), sum c over the columns outside
//   group 0 -> the settings s of group 0 whose sum with c is the row's zero.
// One thread per dword of the first and per mask of the second.
__global__ void __launch_bounds__(256)
prune_tables_kernel(const int* __restrict__ blob, int field_bytes, int dwords, uint32_t* __restrict__ tables)
{
    const uint32_t F = 4 / (uint32_t)field_bytes, NQ = (uint32_t)dwords;
    const uint32_t sums = (uint32_t)blob[kPruneGroups] * 64 * NQ;
    const int B = blob[kPruneBits];
    const int* on = blob + prune_on_at(dwords, dwords * (int)F);
    const uint32_t t = blockIdx.x * 256 + threadIdx.x;
    if (t < sums) {
        const uint32_t q = t % NQ, s = (t / NQ) & 63u, g = t / (64 * NQ);
        uint32_t v = 0;
#pragma unroll
        for (int b = 0; b < 6; ++b) {
            const int j = 6 * (int)g + b;
            if (j < B) v += (uint32_t)on[(2 * j + (((s >> b) & 1u) ? 0 : 1)) * dwords + (int)q];
        }
        tables[t] = v;
        return;
    }
    const uint32_t e = t - sums, stride = (uint32_t)blob[kPruneStride];
    if (e >= (uint32_t)blob[kPruneLeaf] * stride) return;
    const uint32_t r = e / stride, c = e % stride;
    const uint32_t sh = 8 * (uint32_t)field_bytes * (r % F), fm = field_bytes == 1 ? 0xffu : 0xffffu;
    auto field = [&](uint32_t x) __attribute__((always_inline)) { return (x >> sh) & fm; };
    uint32_t y = 0, d[6];  // the row's sum over group 0, first of the empty setting
#pragma unroll
    for (int b = 0; b < 6; ++b) {
        const int* col = on + 2 * b * dwords + (int)(r / F);
        const uint32_t off = field((uint32_t)col[dwords]);
        d[b] = field((uint32_t)col[0]) - off;
        y += off;
    }
    const uint32_t zero = field((uint32_t)blob[kPruneZero + r / F]) - c;
    unsigned long long m = y == zero ? 1ull : 0ull;
#pragma unroll
    for (uint32_t k = 1; k < 64; ++k) {  // in Gray order
        const uint32_t s = k ^ (k >> 1), b = (uint32_t)__builtin_ctz(k);
        y += ((s >> b) & 1u) ? d[b] : 0u - d[b];
        m |= y == zero ? 1ull << s : 0ull;
    }
    ((unsigned long long*)(tables + sums))[e] = r < (uint32_t)blob[kPruneTested] ? m : 0ull;
}

// The tree is walked breadth first, one launch per column group from the
// outermost, through lists of the prefixes that survive (NODES false: a wave
// takes a prefix, tests the 64 settings of group `group` and appends the
// survivors), then over the listed nodes (NODES true).  Depth first, one wave
// per outer prefix, the heaviest prefixes kept a few waves busy long after
// the rest (0/1 order 40, 4 per row: 0.53 ms for 0.04 ms of VALU time).
//
// A list has `sets` segments of `cap` prefixes, each with its counter; a
// prefix that does not fit is walked depth first where it is found.  The
// first launch has no list: its prefixes are all settings of the groups from
// `group` + 1 (group 1: the nodes) outward, [begin, end), a power of two.
//
// 8 waves per SIMD where the registers allow it without spills to memory:
// half 0/1 order 31 548 us, 580 at the 6 that the compiler's own scalar
// registers leave.
template <int FB, int NQ, bool NODES>
__global__ void __launch_bounds__(kPruneBlock) __attribute__((amdgpu_waves_per_eu(NODES && FB == 1 && NQ <= 8 ? 8 : 4)))
int_prune_kernel(const int* __restrict__ blob_, const uint4* __restrict__ tables,
                 const unsigned long long* __restrict__ in,
                 const unsigned int* __restrict__ in_count, unsigned long long* __restrict__ out,
                 unsigned int* __restrict__ out_count, unsigned int cap, int group,
                 unsigned long long* __restrict__ partial, uint64_t begin, uint64_t end)
{
    constexpr int F = 4 / FB;
    constexpr int kWaves = kPruneBlock / kWave;
    constexpr uint32_t kMany = 12;
    extern __shared__ __attribute__((aligned(16))) uint32_t lds[];
    __shared__ unsigned long long red[2 * kWaves];
    __shared__ unsigned long long stack[kWaves * kPruneLevels];
    __shared__ unsigned long long queues[kWaves * 2 * kWave];
    __shared__ unsigned long long obufs[NODES ? 1 : kWaves * 2 * kWave];
    const const_i32* blob = (const const_i32*)blob_;
    const int G = blob[kPruneGroups];
    const int nleaf = blob[kPruneLeaf], stride = blob[kPruneStride], mode = blob[kPruneMode];
    const uint32_t lane = threadIdx.x & (kWave - 1);
    const uint32_t w = uni(threadIdx.x / kWave);

    // Prefixes are handed out in equal sets, one for every sets-th wave.
    const uint32_t waves = gridDim.x * kWaves, wave = blockIdx.x * kWaves + w;
    uint32_t sets = kPruneSets;
    while (sets > waves) sets >>= 1;
    const uint32_t set = wave & (sets - 1);
    const uint32_t total = (uint32_t)(end - begin), share = max(1u, total / sets);
    const uint32_t count = in_count ? min(uni(in_count[set * kPruneCounterStride]), cap) : set < total ? share : 0u;
    // Runs of nodes, or batches of 64 prefixes whose settings are split over
    // 2^cut waves where that leaves waves idle; `step`: waves of this set.
    const uint32_t step = (waves - set + sets - 1) / sets;
    const uint32_t run = max(1u, min(8u, count * sets / (waves * 8)));
    const uint32_t batches = (count + kWave - 1) / kWave;
    uint32_t cut = 0;
    if (!NODES)
        while (cut < 6 && (batches << cut) < 2 * step) ++cut;
    if (!__syncthreads_or(wave / sets * (NODES ? run : 1u) < (NODES ? count : batches << cut))) {
        if (threadIdx.x == 0) partial[2 * blockIdx.x] = partial[2 * blockIdx.x + 1] = 0;
        return;  // no tables for nothing (order 28, 4 per row: 35 -> 28 us a run)
    }

    uint32_t* tab = lds;
    unsigned long long* zt = (unsigned long long*)(lds + (size_t)G * 64 * NQ);
    {
        const uint32_t words = ((uint32_t)G * 64 * NQ * 4 + (uint32_t)(nleaf * stride) * 8) / 16;
#pragma unroll 4
        for (uint32_t i = threadIdx.x; i < words; i += kPruneBlock) ((uint4*)lds)[i] = tables[i];
        __syncthreads();
    }

    unsigned long long* queue = queues + w * 2 * kWave;
    unsigned long long* stk = stack + w * kPruneLevels;
    uint32_t head = 0, tail = 0;  // queue positions, mod 128
    unsigned __int128 acc = 0;

    // The queue's first `count` <= 64 subsets, one per lane.  Subsets of one
    // node (`own`) take their sums from the node's nb and two tables, others
    // from every group's table (at order 30, half 0/1: 4 and 10 LDS reads of
    // 16 bytes per term).
    auto flush = [&](uint32_t count, bool own, const uint32_t (&nb)[NQ]) __attribute__((always_inline)) {
        const uint64_t m = queue[(head + lane) & (2 * kWave - 1)];
        uint32_t c[NQ];
        if (own) {
#pragma unroll
            for (int q = 0; q < NQ; ++q) c[q] = nb[q];
            add_entry<NQ>(c, tab, 64 + ((uint32_t)(m >> 6) & 63u));
            add_entry<NQ>(c, tab, (uint32_t)m & 63u);
        } else {
#pragma unroll
            for (int q = 0; q < NQ; ++q) c[q] = 0;
            for (int g = 0; g < G; ++g) add_entry<NQ>(c, tab, (uint32_t)g * 64 + ((uint32_t)(m >> (6 * g)) & 63u));
        }
        const unsigned __int128 p = product<FB, NQ>(c, blob_, mode);
        const bool neg = (__builtin_popcountll(m) & 1) != 0;
        if (lane < count) acc = neg ? acc - p : acc + p;
        head += count;
    };

    uint32_t lt[NQ];  // this lane's setting of group 1
#pragma unroll
    for (int q = 0; q < NQ; ++q) lt[q] = 0;
    add_entry<NQ>(lt, tab, 64 + lane);

    // A node with every column outside groups 0 and 1 set (`prefix`, packed
    // sums nb): 4096 subsets.
    auto node = [&](const uint32_t (&nb)[NQ], uint64_t prefix) __attribute__((always_inline)) {
        uint32_t c[NQ];
#pragma unroll
        for (int q = 0; q < NQ; ++q) c[q] = nb[q] + lt[q];
        const bool live = rows_nonzero<FB, NQ>(c, blob_, 1);
        if (__builtin_amdgcn_ballot_w64(live) == 0) return;
        uint32_t lo = live ? 0u : ~0u, hi = lo;  // dead settings of group 0
        bool any = true;
        const unsigned long long* z = zt;
#pragma unroll
        for (int q0 = 0; q0 < NQ; q0 += 2)
            if (any && q0 * F < nleaf) {
                unsigned long long m[2 * F];
#pragma unroll
                for (int k = 0; k < 2 * F; ++k) {
                    m[k] = z[(c[q0 + k / F] >> (8 * FB * (k % F))) & (FB == 1 ? 0xffu : 0xffffu)];
                    z += stride;
                }
#pragma unroll
                for (int k = 0; k < 2 * F; ++k) {
                    lo |= (uint32_t)m[k];
                    hi |= (uint32_t)(m[k] >> 32);
                }
                any = __builtin_amdgcn_ballot_w64((lo & hi) != ~0u) != 0;
            }
        if (!any) return;
        lo = ~lo;
        hi = ~hi;
        const uint32_t first = tail, plo = (uint32_t)prefix, phi = (uint32_t)(prefix >> 32);
        // Subset `code` of the node into the queue, from each lane with `has`
        // (m, their ballot).
        auto push = [&](bool has, uint64_t m, uint32_t code) __attribute__((always_inline)) {
            const uint32_t at = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                                          __builtin_amdgcn_mbcnt_lo((uint32_t)m, tail));
            if (has) queue[at & (2 * kWave - 1)] = ((uint64_t)phi << 32) | (plo | code);
            tail += (uint32_t)__builtin_popcountll(m);
            if (tail - head >= (uint32_t)kWave) flush(kWave, (int32_t)(head - first) >= 0, nb);
        };
        // A few lanes hold most of the subsets (half 0/1 order 30: 6 a lane,
        // 28 the most).  A lane with many gives them all at once, setting by
        // setting to the lanes; the others one each a round.
        uint64_t many =
            __builtin_amdgcn_ballot_w64((uint32_t)(__builtin_popcount(lo) + __builtin_popcount(hi)) > kMany);
        if (many != 0) {
            const uint32_t keep = (uint32_t)(__builtin_popcount(lo) + __builtin_popcount(hi)) > kMany ? 0u : ~0u;
            do {
                const int r = __builtin_ctzll(many);
                many &= many - 1;
                const uint64_t m = ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)hi, r) << 32) |
                                   (uint32_t)__builtin_amdgcn_readlane((int)lo, r);
                push(((m >> lane) & 1u) != 0, m, ((uint32_t)r << 6) | lane);
            } while (many != 0);
            lo &= keep;
            hi &= keep;
        }
        uint32_t code = lane << 6;
        uint32_t left = lo;
        for (;;) {  // the words one after the other: 9 instructions a round, 16 for both as one word
            const uint64_t m = __builtin_amdgcn_ballot_w64(left != 0);
            if (m == 0) {
                if (code & 32u) break;
                code |= 32u;
                left = hi;
                continue;
            }
            push(left != 0, m, code | (uint32_t)__builtin_ctz(left));
            left &= left - 1;
        }
    };

    auto sums = [&](uint32_t (&c)[NQ], uint64_t prefix, int g) __attribute__((always_inline)) {  // groups >= g
#pragma unroll
        for (int q = 0; q < NQ; ++q) c[q] = 0;
        for (; g < G; ++g) add_entry<NQ>(c, tab, (uint32_t)g * 64 + ((uint32_t)(prefix >> (6 * g)) & 63u));
    };
    // Prefix `id` of this set: from the list, or of all settings an odd
    // multiplier's spread, the set's own run of multiples (neighbouring
    // settings survive alike, and so do those that share their low bits).
    auto prefix_of = [&](uint32_t id) __attribute__((always_inline)) {
        if (in_count) return (uint64_t)in[(size_t)set * cap + id];
        return (begin + (((set * share + id) * 0x9e3779b1u) & (total - 1))) << (6 * group + 6);
    };
    if constexpr (NODES) {
        // Runs of nodes, after each wave's first through a counter per set
        // (the nodes' terms differ: an even share fixed beforehand ends 30 %
        // later at half 0/1 order 32); the next run is fetched while one is
        // walked, and one counter for all would cost 12 ns a fetch in atomics
        // on one address.
        unsigned int* next_run = out_count + set * kPruneCounterStride;
        auto fetch = [&]() __attribute__((always_inline)) {  // past every wave's first run
            return step * run + atomicAdd(next_run, lane == 0 ? run : 0u);
        };
        uint32_t id = wave / sets * run, next = 0;
        if (id < count) next = fetch();
        while (id < count) {
            const uint32_t last = min(id + run, count);
            for (; id < last; ++id) {
                const uint64_t prefix = uni(prefix_of(id));
                uint32_t nb[NQ];
                sums(nb, prefix, 2);
                if (!in_count && __builtin_amdgcn_ballot_w64(rows_nonzero<FB, NQ>(nb, blob_, 2)) == 0) continue;
                node(nb, prefix);
            }
            id = uni(next);
            if (id < count) next = fetch();
        }
    } else {
        unsigned int* listed = out_count + set * kPruneCounterStride;
        unsigned long long* seg = out + (size_t)set * cap;
        uint32_t cur[NQ];  // packed sums of the groups set so far
        uint64_t left = 0;  // settings of group g still to visit
        int g = group;
        auto expand = [&]() __attribute__((always_inline)) {
            uint32_t c[NQ];
#pragma unroll
            for (int q = 0; q < NQ; ++q) c[q] = cur[q];
            add_entry<NQ>(c, tab, (uint32_t)g * 64 + lane);
            left = __builtin_amdgcn_ballot_w64(rows_nonzero<FB, NQ>(c, blob_, g));
        };
        // Survivors wait in LDS until 64 go to the list with one atomic (an
        // atomic per expansion made this launch 5x as long at order 40).
        unsigned long long* obuf = obufs + w * 2 * kWave;
        uint32_t found = 0, listed_upto = 0;  // positions in obuf, mod 128
        auto append = [&](uint32_t n) __attribute__((always_inline)) {
            if (n == 0) return;
            const uint32_t at = uni(atomicAdd(listed, lane == 0 ? n : 0u)) + lane;
            const uint64_t mine = obuf[(listed_upto + lane) & (2 * kWave - 1)];
            listed_upto += n;
            if (lane < n && at < cap) seg[at] = mine;
            // What does not fit is walked depth first: `cur` holds the groups
            // above g, stk[] the settings left of the groups between.
            uint64_t over = __builtin_amdgcn_ballot_w64(lane < n && at >= cap);
            while (over != 0) {
                const int b = __builtin_ctzll(over);
                over &= over - 1;
                uint64_t prefix = ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(mine >> 32), b) << 32) |
                                  (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)mine, b);
                sums(cur, prefix, group);
                g = group;
                for (;;) {
                    if (g == 2) {
                        node(cur, prefix);
                        left = g < group ? uni((uint64_t)stk[g]) : 0;
                    } else {
                        --g;
                        expand();
                    }
                    while (left == 0 && ++g < group) left = uni((uint64_t)stk[g]);
                    if (g >= group) break;
                    const uint32_t s = (uint32_t)__builtin_ctzll(left);
                    left &= left - 1;
                    stk[g] = left;
                    prefix = ((prefix >> (6 * g + 6)) << (6 * g + 6)) | ((uint64_t)s << (6 * g));
                    sums(cur, prefix, g);
                }
            }
            g = group;
        };
        // 64 prefixes, one per lane, against the settings of the group one
        // after the other (the other way round, 64 settings against one
        // prefix, every lane forms the same prefix's sums: 200 instructions
        // per prefix instead of about 40).  Where that leaves waves idle the
        // settings are split over 2^cut of them.
        const uint32_t used = (uint32_t)blob[kPruneUsed + group];
        const const_i32* care = blob + prune_care_at(NQ, NQ * F) + group * NQ;
        for (uint32_t u = wave / sets; u < (batches << cut); u += step) {
            const uint32_t id = (u >> cut) * kWave + lane, each = 64u >> cut;
            bool valid = id < count;
            const uint64_t prefix = prefix_of(valid ? id : 0u);
            uint32_t c0[NQ];
            sums(c0, prefix, group + 1);
            // the outermost groups' rows, not tested before a first launch
            if (!in_count) valid = valid && rows_nonzero<FB, NQ>(c0, blob_, group + 1);
            if (__builtin_amdgcn_ballot_w64(valid) == 0) continue;
            for (uint32_t s = (u & ((1u << cut) - 1u)) * each, last = s + each; s < last; ++s) {
                constexpr uint32_t kTop = FB == 1 ? 0x80808080u : 0x80008000u;
                const uint4* p = (const uint4*)(tab + ((uint32_t)group * 64 + s) * NQ);
                uint32_t ok = kTop;
#pragma unroll
                for (int q0 = 0; q0 < NQ; q0 += 4)  // rows_nonzero on the dwords the group completes
                    if ((used >> q0) & 15u) {
                        const uint4 v = p[q0 / 4];
                        const uint32_t t[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
                        for (int k = 0; k < 4; ++k) {
                            const uint32_t x = (c0[q0 + k] + t[k]) ^ (uint32_t)blob[kPruneZero + q0 + k];
                            ok &= ((x & ~kTop) + ~kTop) | x | ~(uint32_t)care[q0 + k];
                        }
                    }
                const bool alive = valid && ok == kTop;
                const uint64_t m = __builtin_amdgcn_ballot_w64(alive);
                const uint32_t at = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                                              __builtin_amdgcn_mbcnt_lo((uint32_t)m, found));
                if (alive) obuf[at & (2 * kWave - 1)] = prefix | ((uint64_t)s << (6 * group));
                found += (uint32_t)__builtin_popcountll(m);
                if (found - listed_upto >= (uint32_t)kWave) append(kWave);
            }
        }
        append(found - listed_upto);
    }
    {
        uint32_t none[NQ] = {};
        flush(tail - head, false, none);
    }

    // Block sum mod 2^128.
    unsigned long long slo = (unsigned long long)acc, shi = (unsigned long long)(acc >> 64);
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        const unsigned long long olo = __shfl_xor(slo, off, kWave);
        const unsigned long long ohi = __shfl_xor(shi, off, kWave);
        const unsigned long long s = slo + olo;
        shi = shi + ohi + (s < slo ? 1ull : 0ull);
        slo = s;
    }
    if (lane == 0) {
        red[2 * w] = slo;
        red[2 * w + 1] = shi;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned __int128 s = 0;
        for (int i = 0; i < kWaves; ++i) s += ((unsigned __int128)red[2 * i + 1] << 64) | red[2 * i];
        unsigned long long* rec = partial + 2 * blockIdx.x;
        rec[0] = (unsigned long long)s;
        rec[1] = (unsigned long long)(s >> 64);
    }
}

template <int FB, int NQ>
const void* ptr(bool nodes)
{
    return nodes ? reinterpret_cast<const void*>(&int_prune_kernel<FB, NQ, true>)
                : reinterpret_cast<const void*>(&int_prune_kernel<FB, NQ, false>);
}

}  // namespace prune

const void* prune_tables_kernel_ptr() { return reinterpret_cast<const void*>(&prune::prune_tables_kernel); }

const void* int_prune_kernel_ptr(int field_bytes, int dwords, bool nodes)
{
    using namespace prune;
    if (field_bytes == 1) {
        switch (dwords) {
        case 4: return ptr<1, 4>(nodes);
        case 8: return ptr<1, 8>(nodes);
        case 12: return ptr<1, 12>(nodes);
        case 16: return ptr<1, 16>(nodes);
        default: return nullptr;
        }
    }
    switch (dwords) {
    case 8: return ptr<2, 8>(nodes);
    case 16: return ptr<2, 16>(nodes);
    case 24: return ptr<2, 24>(nodes);
    default: return nullptr;
    }
}

}  // namespace spm
