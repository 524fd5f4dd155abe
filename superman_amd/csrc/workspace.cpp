// workspace.cpp -- the pool of plan memory.
//
// A one-shot call builds a plan, runs it and drops it.  Its device blocks and
// pinned memory used to come from the runtime each time, 25-60 us of a call
// that takes 10 us on the GPU.  Dropped workspaces wait here instead, at most
// kIdleMax of them and kIdleBytes of device memory per device; whatever
// exceeds that is freed, and all of them are when an allocation fails: a call
// that fits the device without the pool fits it with the pool.  A workspace belongs to one plan at a time, and a plan
// gives it back only after its last run's result has arrived, so no two
// streams or threads ever share one.
#include "workspace.h"

#include "superman_amd.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>
#include <vector>

namespace spm {
namespace {

constexpr size_t kIdleMax = 8;
constexpr size_t kIdleBytes = size_t(256) << 20;
constexpr size_t kDevMin = size_t(256) << 10;  // every dense plan fits
constexpr size_t kHostMin = size_t(64) << 10;

std::mutex g_mu;
std::vector<Workspace*> g_idle;

void release(Workspace* w)
{
    if (w->dev) (void)hipFree(w->dev);
    if (w->host) (void)hipHostFree(w->host);
    delete w;
}

Workspace* allocate(int device, size_t dev_bytes, size_t host_bytes)
{
    Workspace* w = new Workspace;
    w->device = device;
    w->dev_bytes = dev_bytes;
    w->host_bytes = host_bytes;
    if (hipMalloc((void**)&w->dev, dev_bytes) != hipSuccess ||
        hipHostMalloc((void**)&w->host, host_bytes + sizeof(RunResult), hipHostMallocMapped | hipHostMallocCoherent) !=
            hipSuccess ||
        hipHostGetDevicePointer((void**)&w->host_dev, w->host, 0) != hipSuccess) {
        (void)hipGetLastError();
        release(w);
        return nullptr;
    }
    w->result_host = (RunResult*)(w->host + host_bytes);
    w->result = (RunResult*)(w->host_dev + host_bytes);
    w->result_host->flag = 0;
    return w;
}

void release_idle()
{
    std::vector<Workspace*> drop;
    {
        std::lock_guard<std::mutex> lk(g_mu);
        drop.swap(g_idle);
    }
    for (Workspace* w : drop) release(w);
}

size_t rounded(size_t bytes, size_t least)
{
    size_t s = least;
    while (s < bytes) s *= 2;
    return s;
}

}  // namespace

int workspace_get(int device, size_t dev_bytes, size_t host_bytes, Workspace** out)
{
    const size_t need = rounded(dev_bytes, kDevMin), hneed = rounded(host_bytes, kHostMin);
    {
        std::lock_guard<std::mutex> lk(g_mu);
        for (size_t i = g_idle.size(); i-- > 0;) {  // the latest first; not a large block for a small plan
            Workspace* w = g_idle[i];
            if (w->device == device && w->dev_bytes >= need && w->dev_bytes <= 4 * need && w->host_bytes >= hneed) {
                g_idle.erase(g_idle.begin() + i);
                *out = w;
                return SPM_OK;
            }
        }
    }
    Workspace* w = allocate(device, need, hneed);
    if (!w) {
        release_idle();
        w = allocate(device, need, hneed);
    }
    if (!w) w = allocate(device, (dev_bytes + 255) & ~size_t(255), (host_bytes + 255) & ~size_t(255));
    *out = w;
    return w ? SPM_OK : SPM_ENOMEM;
}

void workspace_put(Workspace* w, bool idle)
{
    if (!w) return;
    std::vector<Workspace*> drop;
    if (!idle) {
        drop.push_back(w);  // hipFree waits for the device
    } else {
        std::lock_guard<std::mutex> lk(g_mu);
        g_idle.push_back(w);
        for (;;) {  // the oldest go when the device's idle ones are too many or too large
            size_t bytes = 0, count = 0, oldest = g_idle.size();
            for (size_t i = g_idle.size(); i-- > 0;)
                if (g_idle[i]->device == w->device) {
                    bytes += g_idle[i]->dev_bytes;
                    ++count;
                    oldest = i;
                }
            if (count <= kIdleMax && bytes <= kIdleBytes) break;
            drop.push_back(g_idle[oldest]);
            g_idle.erase(g_idle.begin() + oldest);
        }
    }
    for (Workspace* d : drop) release(d);
}

}  // namespace spm
