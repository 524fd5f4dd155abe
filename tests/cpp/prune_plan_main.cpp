// The pruned walk's layout of one integer matrix (prune_plan, host only).
// stdin: n, then n*n entries.  stdout: "none", or "field_bytes dwords mode"
// and one line "o width" per field.
#include "spm_host.h"
#include "spm_kernels.h"

#include <cstdio>
#include <vector>

int main()
{
    int n = 0;
    if (std::scanf("%d", &n) != 1 || n < 1 || n > spm::kMaxN) return 2;
    std::vector<int64_t> a((size_t)n * n);
    for (int64_t& v : a) {
        long long x;
        if (std::scanf("%lld", &x) != 1) return 2;
        v = x;
    }
    std::vector<unsigned char> w(n);
    spm::int_row_weights(a.data(), n, w.data());
    spm::PrunePlan p;
    if (!spm::prune_plan(a.data(), n, w.data(), p)) {
        std::printf("none\n");
        return 0;
    }
    const int fb = p.field_bytes, F = 4 / fb, nq = p.dwords, fields = nq * F;
    const int* b = p.blob.data();
    const int mode = b[spm::kPruneMode];
    std::printf("%d %d %d\n", fb, nq, mode);
    auto field = [&](const int* v, int i) {
        return (int)(((unsigned)v[i / F] >> (8 * fb * (i % F))) & (fb == 1 ? 0xffu : 0xffffu));
    };
    const int* o = b + spm::prune_offset_at(nq);
    const int* on = b + spm::prune_on_at(nq, fields);
    for (int i = 0; i < fields; ++i) {
        int width = 0;
        for (int k = 0; k < 2 * b[spm::kPruneBits]; ++k) width += field(on + (size_t)k * nq, i);
        std::printf("%d %d\n", fb == 1 && mode != 0 ? field(o, i) - 128 : o[i], width);
    }
    return 0;
}
