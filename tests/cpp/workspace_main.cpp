// The plan-memory pool over the fake HIP calls: what it holds idle must not
// make an allocation fail.
#include "workspace.h"

#include "superman_amd.h"

#include <hip/hip_runtime.h>

#include <cstdio>

#define CHECK(x)                                         \
    do {                                                 \
        if (!(x)) {                                      \
            std::printf("line %d: %s\n", __LINE__, #x); \
            return 1;                                    \
        }                                                \
    } while (0)

int main()
{
    using namespace spm;
    constexpr size_t K = 1024;
    Workspace* w[4];
    g_budget = 1024 * K;
    for (auto& p : w) CHECK(workspace_get(0, 10 * K, K, &p) == SPM_OK);
    for (auto p : w) workspace_put(p, true);
    CHECK(g_used > 0);  // kept
    Workspace* big = nullptr;
    CHECK(workspace_get(0, 900 * K, K, &big) == SPM_OK && big->dev_bytes >= 900 * K);
    CHECK(g_used <= g_budget);
    workspace_put(big, false);
    CHECK(g_used == 0 && g_blocks == 0);

    // no room for the rounded size, but for what was asked; twice, as a plan's
    // second run of calls would
    g_budget = 700 * K;
    for (int i = 0; i < 2; ++i) {
        CHECK(workspace_get(0, 600 * K, 100 * K, &big) == SPM_OK);
        CHECK(big->dev_bytes >= 600 * K && big->host_bytes >= 100 * K);
        CHECK((char*)big->result_host >= big->host + 100 * K);
        workspace_put(big, true);
    }
    CHECK(workspace_get(0, 701 * K, K, &big) == SPM_ENOMEM && big == nullptr);
    CHECK(g_used == 0 && g_blocks == 0);  // a failed call keeps nothing
    std::printf("ok\n");
    return 0;
}
