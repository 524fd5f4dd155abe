// prune.cpp -- host layout of an integer matrix for int_prune_kernel
// (walk_prune.h): column order, packed fields, zero patterns, product plan
// and the split into tasks.
#include "spm_host.h"
#include "spm_kernels.h"

#include <algorithm>
#include <cmath>

namespace spm {

namespace {

// -log2 of the share of subsets that leave a row of k entries nonzero, the
// row taken by itself (int_nonzero_term_fraction's rule).
double row_bits(int k)
{
    if (k == 0) return 60.0;
    double p = 1.0;  // C(k, floor(k/2)) / 2^k
    for (int t = 1; t <= k; ++t) p *= (t <= k / 2 ? double(k - k / 2 + t) / t : 1.0) * 0.5;
    return -std::log2(1.0 - std::min(p, 0.999));
}

// Columns from the inside out: each next column is the one that touches the
// least weight of rows not touched yet, so that the outer columns complete
// as many rows as they can.  The first column is tried over the lightest few
// and the order with the least estimated node count is kept.
std::vector<int> inner_first_order(const std::vector<uint64_t>& rows_of, const std::vector<double>& bits, int n,
                                   double* nodes, double* upper)
{
    const int B = n - 1;
    auto weight = [&](uint64_t m) {
        double s = 0;
        for (; m; m &= m - 1) s += bits[__builtin_ctzll(m)];
        return s;
    };
    double all = 0;
    for (int i = 0; i < n; ++i) all += bits[i];
    std::vector<int> starts(n);
    for (int j = 0; j < n; ++j) starts[j] = j;
    std::vector<double> cw(n);
    for (int j = 0; j < n; ++j) cw[j] = weight(rows_of[j]);
    std::stable_sort(starts.begin(), starts.end(), [&](int x, int y) { return cw[x] < cw[y]; });
    std::vector<int> best;
    double best_cost = 1e300;
    constexpr int kStarts = 6;
    for (int s = 0; s < std::min(n, kStarts); ++s) {
        std::vector<int> ord;
        uint64_t touched = 0, used = 0;
        double tw = 0, n2 = 0, up = 0;
        for (int k = 0; k < n; ++k) {
            int pick = -1;
            double pw = 1e300;
            if (k == 0) {
                pick = starts[s];
                pw = cw[pick];
            } else {
                for (int j : starts) {
                    if ((used >> j) & 1ull) continue;
                    const double v = weight(rows_of[j] & ~touched);
                    if (v < pw - 1e-12) {
                        pw = v;
                        pick = j;
                    }
                }
            }
            ord.push_back(pick);
            used |= uint64_t(1) << pick;
            touched |= rows_of[pick];
            tw += pw;
            // settings of the columns outside the first 6 g that survive
            if ((k + 1) % 6 == 0 && k + 1 >= 12 && k + 1 <= B) {
                const double v = std::exp2(double(B - k - 1) - (all - tw));
                (k + 1 == 12 ? n2 : up) += v;
            }
        }
        const double cost = n2 + 0.5 * up;
        if (cost < best_cost) {
            best_cost = cost;
            best = ord;
            *nodes = n2;
            *upper = up;
        }
        if (all == 0.0) break;  // no row is ever zero: nothing to order by
    }
    return best;
}

// A row's bounds in the plan's column order: field = sum of positive entries
// in S and of |negative| entries outside S (times w), y = field + o.  The
// last column is in no subset: its entry is in o alone, which can be far
// larger than the field.
struct Row {
    int src, low, o, width, outer;
    bool test;
};

// The layout with fields of fb bytes.  False when it has no kernel, its tables
// do not fit, or 8-bit fields leave a product that product() would not form
// exactly.
bool lay_out(const int64_t* a, int n, const unsigned char* w, const std::vector<int>& ord, std::vector<Row> rows, int fb,
             PrunePlan& p)
{
    const int B = n - 1, G = (B + 5) / 6;
    const int F = 4 / fb;
    const int nq = fb == 1 ? 4 * ((n + 15) / 16) : 8 * ((n + 15) / 16);
    if (fb == 2 && nq > 24) return false;

    // Fields: group 0's tested rows with zero masks first (those with the
    // fewest masks, while all fit), filled up to whole pairs of dwords with
    // the narrowest of the others; then the other tested rows by the group
    // that completes them; then the rest.  Padding fields are constant 0.
    const size_t table = (size_t)G * 64 * nq * 4;
    if (table + kPruneStaticLds > kPruneLdsMax) return false;
    const int room = (int)std::min<size_t>(kPruneEntriesMax, (kPruneLdsMax - kPruneStaticLds - table) / 8);
    const int fields = nq * F;
    for (int i = n; i < fields; ++i) rows.push_back({-1, G, 1, 0, 0, false});
    auto leaf = [](const Row& r) { return r.test && r.low == 0; };
    std::stable_sort(rows.begin(), rows.end(), [&](const Row& x, const Row& y) {
        if (leaf(x) != leaf(y)) return leaf(x);
        return x.outer < y.outer;
    });
    int tested = 0;
    while (tested < fields && leaf(rows[tested])) ++tested;
    int nleaf = 0, stride = 0;
    for (; tested > 0; --tested) {
        nleaf = (tested + 2 * F - 1) / (2 * F) * (2 * F);
        std::stable_sort(rows.begin() + tested, rows.end(),
                         [](const Row& x, const Row& y) { return x.outer < y.outer; });
        stride = 0;
        for (int i = 0; i < std::min(nleaf, fields); ++i) stride = std::max(stride, rows[i].outer + 1);
        if (nleaf <= fields && (int64_t)nleaf * stride <= room) break;
        rows[tested - 1].test = false;  // its zeros come out of the product
    }
    if (tested == 0) nleaf = stride = 0;
    std::stable_sort(rows.begin() + nleaf, rows.end(), [](const Row& x, const Row& y) {
        if (x.test != y.test) return x.test;
        return x.test && x.low < y.low;
    });

    int t = B >= 18 ? 3 : 2;
    while (B - 6 * t > kPruneTopBits) ++t;
    p.first_group = t;
    p.prefixes = uint64_t(1) << (B - 6 * t);

    // Exact product groups: bits of the rows' values in runs of `len` fields
    // at i and i + half (0: none).
    auto top = [&](int i) {  // the largest |y|
        return std::max<int64_t>(1, std::max(std::abs((int64_t)rows[i].o), std::abs((int64_t)rows[i].o + rows[i].width)));
    };
    auto run_bits = [&](int len, int half) {
        double worst = 0;
        for (int i = 0; i < (half ? half : fields); i += len) {
            double s = 0;
            for (int k = i; k < i + len; ++k)
                for (int j = k; j < fields; j += half ? half : fields) s += std::log2((double)top(j));
            worst = std::max(worst, s);
        }
        return worst;
    };
    int mode = 0;
    if (fb == 1) {
        bool bytes = true;
        for (const Row& r : rows) bytes = bytes && r.o >= -128 && r.o + r.width <= 127;
        mode = !bytes ? 0 : run_bits(8, fields / 2) < 62.9 ? 2 : 1;
        // two rows of a dword multiply in 32 bits (fours of such pairs then
        // fit 64); 16-bit fields form every product in 64
        for (int i = 0; mode == 0 && i < fields; i += 2)
            if (top(i) * top(i + 1) > INT32_MAX) return false;
    } else {
        mode = run_bits(4, 0) < 62.9 ? 1 : 0;
    }

    std::vector<int>& b = p.blob;
    b.assign(prune_blob_ints(nq, fields), 0);
    auto put = [&](int* v, int field, uint32_t x) {
        v[field / F] = (int)((uint32_t)v[field / F] + (x << (8 * fb * (field % F))));
    };
    int* o = b.data() + prune_offset_at(nq);
    for (int i = 0; i < fields; ++i) {
        if (fb == 1 && mode != 0) put(o, i, (uint32_t)(rows[i].o + 128));
        else o[i] = rows[i].o;
    }
    for (int i = 0; i < fields; ++i)
        if (rows[i].test) put(b.data() + kPruneZero, i, (uint32_t)-rows[i].o);
    int* care = b.data() + prune_care_at(nq, fields);
    for (int i = tested; i < fields; ++i)
        if (rows[i].test) put(care + (size_t)std::min(rows[i].low, t) * nq, i, fb == 1 ? 0xffu : 0xffffu);
    for (int g = 0; g <= t; ++g)
        for (int q = 0; q < nq; ++q)
            if (care[(size_t)g * nq + q] != 0) b[kPruneUsed + g] = (int)((uint32_t)b[kPruneUsed + g] | (1u << q));
    int* on = b.data() + prune_on_at(nq, fields);
    for (int k = 0; k < B; ++k)
        for (int i = 0; i < fields; ++i) {
            if (rows[i].src < 0) continue;
            const int64_t v = w[rows[i].src] * a[(size_t)rows[i].src * n + ord[k]];
            if (v != 0) put(on + (size_t)(2 * k + (v < 0 ? 1 : 0)) * nq, i, (uint32_t)(v < 0 ? -v : v));
        }
    b[kPruneGroups] = G;
    b[kPruneLeaf] = nleaf;
    b[kPruneTested] = tested;
    b[kPruneStride] = stride;
    b[kPruneMode] = mode;
    b[kPruneBits] = B;
    p.field_bytes = fb;
    p.dwords = nq;
    p.lds_bytes = (int)(table + (size_t)nleaf * stride * 8);
    return true;
}

}  // namespace

bool prune_plan(const int64_t* a, int n, const unsigned char* w, PrunePlan& p)
{
    if (n < kPruneMinN || n > kMaxN) return false;
    const int B = n - 1, G = (B + 5) / 6;

    std::vector<double> bits(n, 0.0);
    std::vector<uint64_t> rows_of(n, 0);
    for (int i = 0; i < n; ++i) {
        int k = 0;
        for (int j = 0; j < n; ++j) k += a[(size_t)i * n + j] != 0 ? 1 : 0;
        if (w[i] != 1) continue;  // an odd row sum: never zero
        bits[i] = row_bits(k);
        for (int j = 0; j < n; ++j)
            if (a[(size_t)i * n + j] != 0) rows_of[j] |= uint64_t(1) << i;
    }
    double nodes = 0, upper = 0;
    const std::vector<int> ord = inner_first_order(rows_of, bits, n, &nodes, &upper);

    std::vector<Row> rows(n);
    int64_t widest = 0;
    for (int i = 0; i < n; ++i) {
        Row& r = rows[i];
        int64_t sum = 0, width = 0, neg = 0, inner = 0;
        r.src = i;
        r.low = G;
        for (int j = 0; j < n; ++j) sum += a[(size_t)i * n + j];
        for (int k = 0; k < B; ++k) {
            const int64_t v = w[i] * a[(size_t)i * n + ord[k]], m = v < 0 ? -v : v;
            width += m;
            if (v < 0) neg += m;
            if (k < 6) inner += m;
            if (v != 0) r.low = std::min(r.low, k / 6);
        }
        const int64_t y0 = (2 * a[(size_t)i * n + ord[B]] - sum) / (w[i] == 1 ? 2 : 1);
        widest = std::max(widest, width);
        if (width > 0xffff) return false;
        r.o = (int)(y0 - neg);
        r.width = (int)width;
        r.outer = (int)(width - inner);
        r.test = w[i] == 1 && -r.o >= 0 && -r.o <= r.width;
    }
    p.nodes = nodes;
    p.upper = upper;
    return (widest <= 0xff && lay_out(a, n, w, ord, rows, 1, p)) || lay_out(a, n, w, ord, rows, 2, p);
}

// Whether the pruned walk is the faster one.  Its time, fitted to kernel
// times at orders 24-48: 18 us and 8 us a launch, 0.4 ns a node and 4.8e-12
// (n + 40) / 70 s a surviving term, against the walks' rates (int_walk_costs,
// launches 15 us).  Measured on both sides of the line, pruned against the
// best walk: half 0/1 order 24 57 against 39 us, order 25 58 against 61, order
// 28 0.14 against 0.37 ms; 3 per row (every term survives) order 26 130
// against 105 us, order 28 0.42 against 0.38 ms; 4 per row order 25 26 against
// 37 us.  (90 % ones order 30 is left to the FP64 walk: 1.49 against 1.08 ms.)
// The row-independence estimate of the surviving share runs low where rows are
// alike, so nodes and terms count double; from order 30, where a wrong choice
// costs milliseconds, a sample of the subsets says.
bool prune_preferred(const int64_t* a, int n, const PrunePlan& p)
{
    const IntWalkCosts c = int_walk_costs(a, n);
    double q = std::min(1.0, 2.0 * c.q);
    if (n >= 30) {
        constexpr int kSamples = 128;
        uint64_t x = 0x9e3779b97f4a7c15ull;
        int nonzero = 0;
        for (int s = 0; s < kSamples; ++s) {
            x ^= x << 13;
            x ^= x >> 7;
            x ^= x << 17;
            bool nz = true;
            for (int i = 0; i < n && nz; ++i) {
                const int64_t* r = a + (size_t)i * n;
                int64_t y = 2 * r[n - 1], sum = r[n - 1];
                for (int j = 0; j + 1 < n; ++j) {
                    y += ((x >> j) & 1ull) ? 2 * r[j] : 0;
                    sum += r[j];
                }
                nz = y != sum;
            }
            nonzero += nz ? 1 : 0;
        }
        q = std::min(1.0, 1.25 * std::max(c.q, double(nonzero) / kSamples));
    }
    const double subsets = std::ldexp(1.0, n - 1);
    const double pruned = 1.8e-5 + 8e-6 * (p.first_group - 1) +
                          4e-10 * std::min(2.0 * p.nodes, std::ldexp(1.0, n - 13)) +
                          q * subsets * 4.8e-12 * (n + 40) / 70.0;
    const double walk = n >= 26 ? std::min(c.sparse, std::min(c.fp64, c.int32)) : std::min(c.fp64, c.int32);
    return pruned < 1.5e-5 + subsets * walk;
}

}  // namespace spm
