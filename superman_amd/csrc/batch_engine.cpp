// batch_engine.cpp -- the batch engine and serving loop behind spm_batch_* and
// spm_serve_* (include/superman_amd.h).
//
// An engine owns `slots` batch contexts, each with its own HIP stream, a
// pinned staging buffer, a device arena (header, request descriptors, item
// table, matrix data), item and result records, the work counters and,
// optionally, a captured hipGraph of the batch's launch sequence
//   upload (a kernel that copies the staged batch and zeroes the counters)
//   -> walk kernel(s).
// Each request's result is published by the walk kernel itself into
// host-mapped memory followed by a per-request flag, so progress() hands a
// result out as soon as its flag shows, without waiting for the rest of the
// batch; the batch's completion event only frees the slot.
// Requests are prepared on the host at submission (x(empty), +/- planes;
// integer checks), queue in FIFO order, and are admitted into the next batch
// while it stays within the slot's request, item, byte and work budgets.
// A batch is launched as soon as a slot is free, so requests that arrive
// while earlier batches run are admitted into the next slot and start on
// the device as the earlier batch's waves drain (continuous batching).
#include "superman_amd.h"

#include "spm_batch.h"
#include "spm_host.h"
#include "spm_kernels.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <deque>
#include <limits>
#include <memory>
#include <mutex>
#include <string>
#include <thread>
#include <unordered_map>
#include <utility>
#include <vector>

namespace spm {
namespace {

size_t align_up(size_t v, size_t a) { return (v + a - 1) / a * a; }

// Seconds a finished batch may wait for a result's flag to reach host memory.
constexpr double kPublishWait = 1.0;
// Throughput the autotuner gives up for latency: for the fused kernel, and
// for smaller chunks (a request spread over more lanes finishes sooner).
constexpr double kLatencyMargin = 0.05;

// Re-runs of a request whose result failed its checks (item records of
// another batch in its reduction, an integer sum that is not a multiple of
// 2^(n-1)) before it completes with SPM_EHIP.
constexpr int kMaxRetries = 2;

// FP64-op units per Gray subset (work estimates for budgets and ordering),
// by device walk.
double ops_per_subset(int dev_kind, int n)
{
    switch (dev_kind) {
    case kBatchComplex: return 8.0 * n;
    case kBatchInt: return 12.0 * n;
    case kBatchIntSmall: return 5.0 * n;
    default: return 2.0 * n;
    }
}

// Kernel range / counter of a device walk: 1 real, 2 complex, 3 integer.
int walk_group(int dev_kind) { return dev_kind == kBatchIntSmall ? kBatchInt : dev_kind; }

struct Req {
    uint64_t ticket = 0, tag = 0;
    int kind = 0, n = 0;
    int dev_kind = 0;           // device walk (kBatch*)
    std::vector<uint8_t> data;  // planes, then x0 at x0_rel (64-byte aligned)
    size_t x0_rel = 0;
    int L = 0;
    uint64_t chunks = 0;
    uint32_t items = 0;
    double work = 0;
    double t_submit = 0, t_deadline = 0, t_launch = 0;
    bool cancelled = false;
    int index = -1;             // position in a run/replay, -1 for served requests
    int retries = 0;            // re-runs after a result failed its checks
};

struct Slot {
    hipStream_t stream = nullptr;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    hipGraph_t graph[2] = {nullptr, nullptr};  // [organisation], captured when first used
    hipGraphExec_t exec[2] = {nullptr, nullptr};
    int own_int = 0;                // organisation of the current batch (kOwnIntWork)
    uint8_t* h_stage = nullptr;     // host-mapped, coherent: read by the upload kernel
    uint8_t* dh_stage = nullptr;    // its device address
    uint8_t* d_arena = nullptr;
    double* d_item = nullptr;
    double* h_res = nullptr;        // host-mapped result records [max_requests][8]
    unsigned int* h_flag = nullptr; // host-mapped flags [max_requests]: seq when published
    double* dh_res = nullptr;       // device addresses of the two
    unsigned int* dh_flag = nullptr;
    uint32_t seq = 0;               // batch number of the slot's current batch
    std::vector<char> taken;        // result already handed out (per staged request)
    unsigned int* d_counter = nullptr;  // [4] work counters, then [max_requests] item counts
    std::vector<Req*> reqs;
    bool busy = false;
    bool fault = false;
    double t_launch = 0, t_ready = 0;
};

}  // namespace
}  // namespace spm

using namespace spm;

struct spm_batch {
    spm_batch_config cfg{};
    spm_batch_tuning tune{};
    bool chosen[4] = {false, false, false, false};  // [kind]: the caller set log2_chunk (geometry)
    bool all_fused = false;  // no kernel of their own for the integers (autotuning on a mix's integer requests)
    int cus = 0;
    int max_wpc[4] = {0, 0, 0, 0};  // resident waves per CU: [0] fused, [kind] one-kind kernel
    size_t desc_off = 0, item_off = 0, data_off = 0, stage_bytes = 0;
    std::vector<Slot> slots;
    std::deque<Req*> pending;
    std::deque<spm_completion> done;
    std::unordered_map<uint64_t, Req*> live;
    uint64_t next_ticket = 1;
    int fault_launches = 0;
    uint64_t batches = 0;
    double busy_since = -1, busy_total = 0;
    std::string last_error;  // the last failed HIP call, for spm_batch_last_error
    uint64_t late_publish = 0;  // results whose flag arrived after their batch's completion event
    uint64_t retried = 0;       // requests run again after a result failed its checks
    int bad_results = 0;        // results still to be failed on purpose (spm_batch_inject_bad_results)
    std::mutex mu;
};

namespace {

bool dry(const spm_batch* b) { return b->cfg.executor == SPM_EXEC_DRYRUN; }

// The default tuning.  One fused launch: every request's items are in the
// work queue at once, where the three one-kind kernels run one after another
// and each ends in its own thinly filled tail (256 mixed requests of orders 8
// to 24: 2.45 -> 2.08 ms, 64 of orders 8 to 20: 0.94 -> 0.51 ms, 24 of orders
// 4 to 14: 0.32 -> 0.18 ms).  Chunks of 2^8 complex and 2^9 integer steps: the
// last item to start ends a batch, and with 2^9 and 2^10 steps 48 requests of
// orders 10 to 25 took 1.04 instead of 0.95 ms; chunks half as long again (and
// 2^8 real ones) spend more on chunk starts (400 requests 4.1 -> 4.4 ms).
constexpr int kBatchFused = 1;
// With more than this much integer work (Req::work, about 2.5e-14 s each), and
// more than half of its work integer, a fused batch leaves the integer items to
// their own kernel, launched behind the other kinds'.  The complex walk's 195
// VGPRs leave the fused kernel 2 waves per SIMD, the integer kernel has 4 and
// walks 1.1 times as fast; but a launch more ends in a tail more, and small
// integer requests wait for the other kinds.  Fused / own: integers only, 300 of
// orders 22 to 25 7.52 / 6.84 ms, 20 of 26 to 28 5.64 / 5.10, 12 of 26 to 28
// (1.3e11) 2.69 / 2.41, 300 of 14 to 20 (5e9) 1.59 / 1.64; 300 a quarter real
// 7.35 / 6.88, half real 8.78 / 8.53, a quarter complex (65 % integer work) 9.12 /
// 9.07, half complex (38 %) 10.2 / 10.6, a quarter integer (29 %) 9.9 / 10.3.
constexpr double kOwnIntWork = 1e11;
constexpr int kBatchChunk[4] = {0, 10, 8, 9};  // [kind]
// The least chunk sizes of a request whose items at those exceed the engine's.
constexpr int kBatchChunkWide[4] = {0, 10, 9, 10};
// A request is split over up to 2^10 chunks (16 wavefronts) before its chunks
// grow beyond 2^5 steps, since one wavefront's serial walk bounds a batch of
// small orders: 32 requests of orders 4 to 16 take 0.21 instead of 0.26 ms.  2^12 chunks cost
// 400 requests of orders 8 to 25 2 % (4.13 -> 4.20 ms) in chunk starts.
constexpr int kSplitChunks = 10;
constexpr int kSplitSteps = 5;

// Chunk size for a request: L >= 2 for the pipelined walks (n >= 3); n = 2
// walks one 2-step chunk per lane (L = 1) and n = 1 its single subset.  It
// follows from the request and the engine's configuration alone.  The target is
// an upper limit: small requests are split further, by whatever target (with the
// autotuner's sizes set on a second engine and taken as they are, the serving mix
// at the plain path's load had a p99 of 1.95 instead of 1.86 ms).  The item budget
// lengthens chunks of the engine's own sizes only: one that the caller set is
// refused there.
void geometry(const spm_batch* b, Req* r)
{
    const int B = r->n - 1;
    const int target = b->tune.log2_chunk[r->kind];
    auto items = [&](int L) { return ((uint64_t(1) << (B - L)) + kWaveLanes - 1) / kWaveLanes; };
    int L;
    if (r->n == 1) L = 0;
    else if (r->n == 2) L = 1;
    else {
        auto whole = [&](int steps) { return std::max(2, std::min(steps, B - 6)); };  // at least one full wavefront
        L = std::min(whole(target), std::max(kSplitSteps, B - kSplitChunks));
        if (items(L) > (uint64_t)b->cfg.max_items)
            L = whole(b->chosen[r->kind] ? target : std::max(target, kBatchChunkWide[r->kind]));
    }
    r->L = L;
    r->chunks = uint64_t(1) << (B - L);
    r->items = (uint32_t)items(L);
    const double ops = ops_per_subset(r->dev_kind, r->n);
    r->work = std::ldexp(1.0, B) * ops;
}

int prepare(const spm_request* q, Req* r)
{
    if (!q || !q->a) return SPM_EINVAL;
    if (q->kind != SPM_KIND_REAL && q->kind != SPM_KIND_COMPLEX && q->kind != SPM_KIND_INT) return SPM_EINVAL;
    const int n = q->n;
    if (n < 1 || n > kBatchMaxN) return SPM_EINVAL;
    const int w = q->kind == SPM_KIND_COMPLEX ? 2 : 1;
    for (int e = 0; e < w * n * n; ++e)
        if (!std::isfinite(q->a[e])) return SPM_EINVAL;
    r->kind = q->kind;
    r->n = n;
    r->tag = q->tag;
    if (q->kind == SPM_KIND_INT) {
        std::vector<int64_t> ai((size_t)n * n);
        for (int e = 0; e < n * n; ++e) {
            const double v = q->a[e];
            if (v != std::floor(v) || std::fabs(v) > 1073741824.0) return SPM_ENOTINT;
            ai[e] = (int64_t)v;
        }
        std::vector<int> y0(n);
        double lb = 0;
        const int st = int_prepare(ai.data(), n, y0.data(), &lb);
        if (st != SPM_OK) return st;
        if (int_small_ok(ai.data(), n)) {  // FP64 walk: planes and y0 as doubles
            r->dev_kind = kBatchIntSmall;
            const size_t planes = sizeof(double) * 2 * (size_t)n * n;
            r->x0_rel = align_up(planes, kBatchAlign);
            r->data.assign(r->x0_rel + sizeof(double) * n, 0);
            int_small_planes(ai.data(), n, (double*)r->data.data());
            double* yd = (double*)(r->data.data() + r->x0_rel);
            for (int i = 0; i < n; ++i) yd[i] = (double)y0[i];
        } else {
            r->dev_kind = kBatchInt;
            const size_t planes = sizeof(int) * 2 * (size_t)n * n;
            r->x0_rel = align_up(planes, kBatchAlign);
            r->data.assign(r->x0_rel + sizeof(int) * n, 0);
            int_planes(ai.data(), n, (int*)r->data.data());
            std::memcpy(r->data.data() + r->x0_rel, y0.data(), sizeof(int) * n);
        }
    } else {
        r->dev_kind = q->kind == SPM_KIND_COMPLEX ? kBatchComplex : kBatchReal;
        const size_t planes = sizeof(double) * 2 * (size_t)w * n * n;
        r->x0_rel = align_up(planes, kBatchAlign);
        r->data.assign(r->x0_rel + sizeof(double) * w * n, 0);
        dense_prepare(q->a, n, w, (double*)r->data.data(), (double*)(r->data.data() + r->x0_rel));
    }
    return SPM_OK;
}

// Puts a request whose result failed its checks back at the head of the
// queue; false once its re-runs are used up.
bool requeue(spm_batch* b, Req* r)
{
    if (r->retries >= kMaxRetries || r->cancelled) return false;
    ++r->retries;
    ++b->retried;
    b->pending.push_front(r);
    return true;
}

void complete(spm_batch* b, Req* r, int status, const double* rec, double t_done, float batch_ms)
{
    spm_completion c;
    std::memset(&c, 0, sizeof c);
    c.ticket = r->ticket;
    c.tag = r->tag;
    c.t_submit = r->t_submit;
    c.t_launch = r->t_launch;
    c.t_done = t_done;
    spm_result& res = c.result;
    if (status == SPM_OK && r->cancelled) status = SPM_ECANCELLED;
    if (status == SPM_OK && b->bad_results > 0) {
        --b->bad_results;
        b->last_error = "injected bad result";
        if (requeue(b, r)) return;
        status = SPM_EHIP;
    } else if (status == SPM_OK && rec && rec[kBatchStale] != 0.0) {
        // the reduction read item records that were not this batch's
        status = SPM_EHIP;
        b->last_error = "batch execution: " + std::to_string((long long)rec[kBatchStale]) + " of " +
                        std::to_string(r->items) + " item records of a request (n = " + std::to_string(r->n) +
                        ") were not this batch's when its last item finished";
        if (requeue(b, r)) return;
    } else if (status == SPM_OK && rec) {
        if (r->kind == SPM_KIND_INT) {
            uint64_t w[2];
            std::memcpy(w, rec, 16);
            status = int_fill_result(r->n, w[0], w[1], &res);
            if (status != SPM_OK)
                b->last_error = "batch execution: integer sum of a request (n = " + std::to_string(r->n) +
                                ", L = " + std::to_string(r->L) + ", " + std::to_string(r->items) +
                                " items) is not a multiple of 2^(n-1)";
            if (status != SPM_OK && requeue(b, r)) return;
        } else {
            dense_fill_result(r->n, r->kind == SPM_KIND_COMPLEX, true, rec, &res);
        }
    } else if (status == SPM_OK) {  // dry run: scheduled, nothing computed
        res.re = res.im = std::numeric_limits<double>::quiet_NaN();
        res.n = r->n;
        res.subsets = uint64_t(1) << (r->n - 1);
    }
    res.status = status;
    res.kernel_ms = batch_ms;
    res.seconds = t_done - r->t_submit;
    res.launches = rec ? 1 : 0;
    b->live.erase(r->ticket);
    b->done.push_back(c);
    delete r;
}

void free_graph(Slot& s)
{
    for (int o = 0; o < 2; ++o) {
        if (s.exec[o]) (void)hipGraphExecDestroy(s.exec[o]);
        if (s.graph[o]) (void)hipGraphDestroy(s.graph[o]);
        s.exec[o] = nullptr;
        s.graph[o] = nullptr;
    }
}

void free_slot(Slot& s)
{
    free_graph(s);
    if (s.stream) (void)hipStreamDestroy(s.stream);
    if (s.ev0) (void)hipEventDestroy(s.ev0);
    if (s.ev1) (void)hipEventDestroy(s.ev1);
    if (s.h_stage) (void)hipHostFree(s.h_stage);
    if (s.h_res) (void)hipHostFree(s.h_res);
    if (s.h_flag) (void)hipHostFree(s.h_flag);
    if (s.d_arena) (void)hipFree(s.d_arena);
    if (s.d_item) (void)hipFree(s.d_item);
    if (s.d_counter) (void)hipFree(s.d_counter);
    s = Slot();
}

int grid_for(const spm_batch* b, int q)
{
    int wpc = b->max_wpc[q];
    if (b->tune.waves_per_cu > 0) wpc = std::min(wpc, std::max(kDenseBlock / kWaveLanes, b->tune.waves_per_cu));
    return std::max(1, b->cus * wpc / (kDenseBlock / kWaveLanes));
}

// The launch sequence of one batch after its arena upload.  Each request's
// result is reduced inside the walk kernel by the wave that finishes its last
// item and published to the slot's host-mapped records.
hipError_t enqueue(spm_batch* b, Slot& s)
{
    hipError_t e;
    unsigned int* done = s.d_counter + 64;
    {
        unsigned int n_done = (unsigned int)b->cfg.max_requests;
        void* args[] = {&s.dh_stage, &s.d_arena, &s.d_counter, &done, &n_done};
        e = hipLaunchKernel(batch_stage_kernel_ptr(), dim3(kStageBlocks), dim3(256), args, 0, s.stream);
        if (e != hipSuccess) return e;
    }
    constexpr int kMask[4] = {15, 1, 2, 12};
    constexpr int kLaunches[3][3] = {{0, -1, -1}, {0, 3, -1}, {1, 2, 3}};  // fused; fused and own integers; one a kind
    for (int q : kLaunches[b->tune.fused ? s.own_int : 2]) {
        if (q < 0) break;
        void* args[] = {&s.d_arena, &s.d_item, &s.d_counter, &done, &s.dh_res, &s.dh_flag};
        e = hipLaunchKernel(batch_walk_kernel_ptr(kMask[q]), dim3(grid_for(b, q)), dim3(kDenseBlock), args, 0, s.stream);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

hipError_t capture(spm_batch* b, Slot& s)
{
    hipError_t e = hipStreamBeginCapture(s.stream, hipStreamCaptureModeRelaxed);
    if (e != hipSuccess) return e;
    hipError_t e1 = enqueue(b, s);
    hipGraph_t g = nullptr;
    e = hipStreamEndCapture(s.stream, &g);
    if (e1 != hipSuccess) {
        if (g) (void)hipGraphDestroy(g);
        return e1;
    }
    if (e != hipSuccess) return e;
    s.graph[s.own_int] = g;
    return hipGraphInstantiate(&s.exec[s.own_int], g, nullptr, nullptr, 0);
}

// Admission: FIFO with skip-ahead, within the slot's budgets.  Requests past
// their deadline complete with SPM_ETIMEDOUT here.
std::vector<Req*> admit(spm_batch* b, double now)
{
    std::vector<Req*> out;
    size_t bytes = 0;
    uint64_t items = 0;
    double work = 0;
    for (auto it = b->pending.begin(); it != b->pending.end() && (int)out.size() < b->cfg.max_requests;) {
        Req* r = *it;
        if (r->cancelled) {
            it = b->pending.erase(it);
            complete(b, r, SPM_ECANCELLED, nullptr, now, 0.f);
            continue;
        }
        if (r->t_deadline > 0 && now > r->t_deadline) {
            it = b->pending.erase(it);
            complete(b, r, SPM_ETIMEDOUT, nullptr, now, 0.f);
            continue;
        }
        geometry(b, r);
        const size_t rb = align_up(r->data.size(), kBatchAlign);
        const bool fits = bytes + rb <= b->cfg.arena_bytes && items + r->items <= (uint64_t)b->cfg.max_items &&
                          (out.empty() || b->cfg.max_batch_work <= 0 || work + r->work <= b->cfg.max_batch_work);
        if (fits) {
            out.push_back(r);
            bytes += rb;
            items += r->items;
            work += r->work;
            it = b->pending.erase(it);
        } else {
            ++it;
        }
    }
    return out;
}

// Writes header, descriptors, item table and data into the slot's staging
// buffer; returns the bytes to upload.  Item order: shortest request first
// (fused: over all kinds; else grouped by kernel), so that small
// requests publish their results early; a large request's items are all of
// one size, so the batch's tail is at most one item long.
size_t stage(spm_batch* b, Slot& s, std::vector<Req*>& rs)
{
    double work = 0, int_work = 0;
    for (const Req* r : rs) {
        work += r->work;
        int_work += walk_group(r->dev_kind) == kBatchInt ? r->work : 0;
    }
    s.own_int = b->tune.fused && !b->all_fused && int_work > kOwnIntWork && int_work > 0.5 * work ? 1 : 0;
    auto group = [&](const Req* r) {  // launched after one another, in this order
        const int g = walk_group(r->dev_kind);
        return !b->tune.fused ? g : s.own_int && g == kBatchInt ? 1 : 0;
    };
    std::stable_sort(rs.begin(), rs.end(), [&](const Req* x, const Req* y) {
        return group(x) != group(y) ? group(x) < group(y) : x->work < y->work;
    });
    uint8_t* h = s.h_stage;
    BatchHeader hd;
    std::memset(&hd, 0, sizeof hd);
    hd.requests = (uint32_t)rs.size();
    hd.seq = s.seq;
    hd.desc_off = (uint32_t)b->desc_off;
    hd.item_off = (uint32_t)b->item_off;
    BatchRequestDesc* desc = (BatchRequestDesc*)(h + b->desc_off);
    uint32_t* item_req = (uint32_t*)(h + b->item_off);
    size_t data = b->data_off;
    uint32_t item = 0;
    for (int k = 0; k < 4; ++k) hd.range_begin[k] = hd.range_end[k] = 0;
    for (size_t j = 0; j < rs.size(); ++j) {
        Req* r = rs[j];
        const int grp = walk_group(r->dev_kind);
        if (hd.range_end[grp] == 0 && hd.range_begin[grp] == 0) hd.range_begin[grp] = item;
        BatchRequestDesc d;
        std::memset(&d, 0, sizeof d);
        d.kind = (uint32_t)r->dev_kind;
        d.n = (uint32_t)r->n;
        d.L = r->L;
        d.items = r->items;
        d.num_chunks = r->chunks;
        d.mat_off = data;
        d.x0_off = data + r->x0_rel;
        d.item_base = item;
        std::memcpy(desc + j, &d, sizeof d);
        std::memcpy(h + data, r->data.data(), r->data.size());
        data += align_up(r->data.size(), kBatchAlign);
        for (uint32_t t = 0; t < r->items; ++t) item_req[item + t] = (uint32_t)j;
        item += r->items;
        hd.range_end[grp] = item;
    }
    hd.items = item;
    hd.range_begin[0] = 0;
    hd.range_end[0] = s.own_int ? hd.range_begin[kBatchInt] : item;
    hd.bytes = data;
    std::memcpy(h, &hd, sizeof hd);
    return data;
}

int launch(spm_batch* b, Slot& s, std::vector<Req*>& rs, double now)
{
    s.reqs = rs;
    s.busy = true;
    s.fault = false;
    s.t_launch = now;
    for (Req* r : rs) r->t_launch = now;
    ++b->batches;
    if (b->busy_since < 0) b->busy_since = now;
    if (b->fault_launches > 0) {
        --b->fault_launches;
        s.fault = true;
        return SPM_OK;
    }
    if (dry(b)) {
        double work = 0;
        for (Req* r : rs) work += r->work;
        s.t_ready = now + 20e-6 + work / 2e13;
        return SPM_OK;
    }
    ++s.seq;
    (void)stage(b, s, rs);  // the upload kernel reads the staged size from the header
    s.reqs = rs;  // staged order = record order
    s.taken.assign(rs.size(), 0);
    DeviceGuard g(b->cfg.device);
    if (!g.ok()) return SPM_EHIP;
    auto fail = [&](hipError_t e, const char* what) {
        b->last_error = std::string(what) + ": " + hipGetErrorName(e);
        return SPM_EHIP;
    };
    hipError_t e = hipEventRecord(s.ev0, s.stream);
    if (e != hipSuccess) return fail(e, "hipEventRecord");
    if (b->cfg.use_graph) {
        if (!s.exec[s.own_int] && (e = capture(b, s)) != hipSuccess) {
            free_graph(s);
            return fail(e, "graph capture");
        }
        if ((e = hipGraphLaunch(s.exec[s.own_int], s.stream)) != hipSuccess) return fail(e, "hipGraphLaunch");
    } else if ((e = enqueue(b, s)) != hipSuccess) {
        return fail(e, "kernel launch");
    }
    e = hipEventRecord(s.ev1, s.stream);
    if (e != hipSuccess) return fail(e, "hipEventRecord");
    return SPM_OK;
}

void fail_slot(spm_batch* b, Slot& s, int status, double now)
{
    for (Req* r : s.reqs)
        if (r) complete(b, r, status, nullptr, now, 0.f);
    s.reqs.clear();
    s.busy = false;
}

// A request's result is on the host: its flag holds the slot's batch number
// and its record is whole -- its own tag and a matching check word (the
// record's words are stored before the flag, but each read here checks
// them all).
bool published(const Slot& s, size_t j)
{
    if (__atomic_load_n(s.h_flag + j, __ATOMIC_ACQUIRE) != s.seq) return false;
    uint64_t w[kBatchRec];
    std::memcpy(w, s.h_res + j * kBatchRec, sizeof w);
    return w[kBatchTag] == batch_tag(s.seq, (uint32_t)j) && w[kBatchCheck] == record_check(w);
}

// Retires finished slots; returns how many were retired.
int retire(spm_batch* b, double now)
{
    int got = 0;
    for (Slot& s : b->slots) {
        if (!s.busy) continue;
        if (s.fault) {
            fail_slot(b, s, SPM_EFAULTINJ, now);
            ++got;
            continue;
        }
        if (dry(b)) {
            if (now < s.t_ready) continue;
            for (Req* r : s.reqs) complete(b, r, SPM_OK, nullptr, now, 0.f);
            s.reqs.clear();
            s.busy = false;
            ++got;
            continue;
        }
        // results already published by the kernel (flag and record tag)
        for (size_t j = 0; j < s.reqs.size(); ++j) {
            if (s.taken[j] || !published(s, j)) continue;
            s.taken[j] = 1;
            complete(b, s.reqs[j], SPM_OK, s.h_res + j * kBatchRec, now, -1.f);
            s.reqs[j] = nullptr;
        }
        const hipError_t e = hipEventQuery(s.ev1);
        if (e == hipErrorNotReady) continue;
        if (e != hipSuccess) {
            b->last_error = std::string("batch execution: ") + hipGetErrorName(e);
            for (size_t j = 0; j < s.reqs.size(); ++j)
                if (!s.taken[j]) complete(b, s.reqs[j], SPM_EHIP, nullptr, now, 0.f);
            s.reqs.clear();
            s.busy = false;
            ++got;
            continue;
        }
        // The batch's kernels are over, so every result has been stored; a
        // store to host memory may still be on its way when the completion
        // is seen, so each missing flag gets a bounded wait before it counts
        // as an error.
        for (size_t j = 0; j < s.reqs.size(); ++j) {
            if (s.taken[j]) continue;
            bool ok = published(s, j);
            if (!ok) {
                const double give_up = now_seconds() + kPublishWait;
                while (!(ok = published(s, j)) && now_seconds() < give_up) std::this_thread::yield();
                if (ok) ++b->late_publish;
                else b->last_error = "batch execution: a result was not published by the end of its batch";
            }
            complete(b, s.reqs[j], ok ? SPM_OK : SPM_EHIP, ok ? s.h_res + j * kBatchRec : nullptr, now, -1.f);
        }
        s.reqs.clear();
        s.busy = false;
        ++got;
    }
    return got;
}

int progress(spm_batch* b, int* in_flight)
{
    double now = now_seconds();
    retire(b, now);
    for (Slot& s : b->slots) {
        if (s.busy || b->pending.empty()) continue;
        std::vector<Req*> rs = admit(b, now);
        if (rs.empty()) break;
        const int st = launch(b, s, rs, now);
        if (st != SPM_OK) fail_slot(b, s, st, now);
    }
    int busy = 0;
    for (const Slot& s : b->slots) busy += s.busy ? 1 : 0;
    now = now_seconds();
    if (busy == 0 && b->busy_since >= 0) {
        b->busy_total += now - b->busy_since;
        b->busy_since = -1;
    }
    if (in_flight) *in_flight = busy;
    return SPM_OK;
}

bool idle(const spm_batch* b)
{
    if (!b->pending.empty()) return false;
    for (const Slot& s : b->slots)
        if (s.busy) return false;
    return true;
}

int submit(spm_batch* b, const spm_request* q, double t_submit, int index, uint64_t* ticket)
{
    if ((int)b->pending.size() >= b->cfg.max_pending) return SPM_EAGAIN;
    std::unique_ptr<Req> r(new Req);
    int st = prepare(q, r.get());
    if (st != SPM_OK) return st;
    geometry(b, r.get());
    if (align_up(r->data.size(), kBatchAlign) > b->cfg.arena_bytes || r->items > (uint32_t)b->cfg.max_items)
        return SPM_ENOMEM;
    r->ticket = b->next_ticket++;
    r->t_submit = t_submit;
    r->t_deadline = q->deadline_s > 0 ? t_submit + q->deadline_s : 0;
    r->index = index;
    if (ticket) *ticket = r->ticket;
    b->live[r->ticket] = r.get();
    b->pending.push_back(r.release());
    return SPM_OK;
}

void set_status(spm_result* out, int st)
{
    std::memset(out, 0, sizeof *out);
    out->status = st;
}

// Drives `count` requests through the engine: all at t = 0 (arrival_s =
// NULL) or at their arrival times.  Per-request results/latencies by index.
int drive(spm_batch* b, int count, const spm_request* reqs, const double* arrival_s, spm_result* out,
          double* latency_s, spm_serve_stats* stats)
{
    if (count < 0 || (count > 0 && (!reqs || !out))) return SPM_EINVAL;
    if (!idle(b) || !b->done.empty()) return SPM_EAGAIN;
    std::unordered_map<uint64_t, int> index;
    std::vector<double> lat(count, 0.0);
    const uint64_t batches0 = b->batches;
    const uint64_t late0 = b->late_publish;
    const uint64_t retried0 = b->retried;
    b->busy_total = 0;
    b->busy_since = -1;
    const double t0 = now_seconds();
    int next = 0, finished = 0, first_err = SPM_OK;
    double t_last = t0;
    while (finished < count) {
        double now = now_seconds();
        while (next < count && (!arrival_s || t0 + arrival_s[next] <= now)) {
            uint64_t tk = 0;
            const double t_arr = arrival_s ? t0 + arrival_s[next] : t0;
            const int st = submit(b, reqs + next, t_arr, next, &tk);
            if (st == SPM_EAGAIN) break;  // queue full: retry after progress
            if (st != SPM_OK) {
                set_status(out + next, st);
                lat[next] = 0.0;
                if (first_err == SPM_OK) first_err = st;
                ++finished;
            } else {
                index[tk] = next;
            }
            ++next;
        }
        int busy = 0;
        progress(b, &busy);
        bool any = false;
        while (!b->done.empty()) {
            const spm_completion c = b->done.front();
            b->done.pop_front();
            auto it = index.find(c.ticket);
            if (it == index.end()) continue;
            const int i = it->second;
            out[i] = c.result;
            lat[i] = c.t_done - (arrival_s ? t0 + arrival_s[i] : t0);
            if (c.result.status != SPM_OK && first_err == SPM_OK) first_err = c.result.status;
            t_last = std::max(t_last, c.t_done);
            ++finished;
            any = true;
        }
        if (!any && busy == 0 && b->pending.empty() && next < count && arrival_s) {
            // idle until the next arrival
            const double wait = t0 + arrival_s[next] - now_seconds();
            if (wait > 200e-6) std::this_thread::sleep_for(std::chrono::duration<double>(wait - 100e-6));
        }
    }
    // Results are handed out before their batch's kernels finish; leave the
    // engine idle (every slot retired) for the next caller.
    for (;;) {
        int busy = 0;
        progress(b, &busy);
        if (busy == 0) break;
        std::this_thread::yield();
    }
    if (latency_s)
        for (int i = 0; i < count; ++i) latency_s[i] = lat[i];
    if (stats) {
        std::memset(stats, 0, sizeof *stats);
        std::vector<double> ok;
        for (int i = 0; i < count; ++i) {
            if (out[i].status == SPM_OK) ok.push_back(lat[i]);
            else ++stats->failed;
        }
        stats->completed = ok.size();
        stats->batches = b->batches - batches0;
        stats->late_publish = b->late_publish - late0;
        stats->retried = b->retried - retried0;
        const double first = arrival_s && count > 0 ? t0 + arrival_s[0] : t0;
        stats->wall_s = t_last - first;
        stats->perms_per_s = stats->wall_s > 0 ? ok.size() / stats->wall_s : 0.0;
        if (!ok.empty()) {
            std::sort(ok.begin(), ok.end());
            auto pct = [&](double p) {
                const size_t k = (size_t)std::min<double>(ok.size() - 1, std::ceil(p * ok.size()) - 1);
                return ok[k];
            };
            stats->p50_s = pct(0.50);
            stats->p99_s = pct(0.99);
            double s = 0;
            for (double v : ok) s += v;
            stats->mean_s = s / ok.size();
            stats->max_s = ok.back();
        }
        stats->mean_batch = stats->batches ? double(count) / stats->batches : 0.0;
        stats->device_busy = stats->wall_s > 0 ? std::min(1.0, b->busy_total / stats->wall_s) : 0.0;
    }
    return first_err;
}

}  // namespace

extern "C" void spm_batch_config_default(spm_batch_config* c)
{
    if (!c) return;
    std::memset(c, 0, sizeof *c);
    c->device = 0;
    c->slots = 2;
    c->max_requests = 1024;
    c->max_items = 1 << 16;
    c->arena_bytes = size_t(64) << 20;
    c->max_pending = 1 << 16;
    c->max_batch_work = 0;
    c->use_graph = 1;
    c->executor = SPM_EXEC_DEVICE;
}

extern "C" int spm_batch_create(const spm_batch_config* cfg, spm_batch** out)
{
    if (!cfg || !out) return SPM_EINVAL;
    *out = nullptr;
    if (cfg->slots < 1 || cfg->slots > 8 || cfg->max_requests < 1 || cfg->max_requests > (1 << 20) ||
        cfg->max_items < 1 || cfg->max_items > (1 << 26) || cfg->arena_bytes < 1024 || cfg->max_pending < 1)
        return SPM_EINVAL;
    if (cfg->executor != SPM_EXEC_DEVICE && cfg->executor != SPM_EXEC_DRYRUN) return SPM_EINVAL;
    std::unique_ptr<spm_batch> b(new spm_batch);
    b->cfg = *cfg;
    b->tune.fused = kBatchFused;
    b->tune.waves_per_cu = 0;
    std::copy(kBatchChunk, kBatchChunk + 4, b->tune.log2_chunk);
    b->desc_off = align_up(sizeof(BatchHeader), kBatchAlign);
    b->item_off = align_up(b->desc_off + sizeof(BatchRequestDesc) * cfg->max_requests, kBatchAlign);
    b->data_off = align_up(b->item_off + sizeof(uint32_t) * cfg->max_items, kBatchAlign);
    b->stage_bytes = b->data_off + align_up(cfg->arena_bytes, kBatchAlign);
    b->slots.resize(cfg->slots);
    if (dry(b.get())) {
        b->cus = 256;
        for (int q = 0; q < 4; ++q) b->max_wpc[q] = 8;
        *out = b.release();
        return SPM_OK;
    }
    int st = device_cus(cfg->device, &b->cus);
    if (st != SPM_OK) return st;
    DeviceGuard g(cfg->device);
    if (!g.ok()) return SPM_EHIP;
    const int masks[4] = {15, 1, 2, 12};
    for (int q = 0; q < 4; ++q) {
        int bpc = 0;
        st = blocks_per_cu(cfg->device, batch_walk_kernel_ptr(masks[q]), kDenseBlock, &bpc);
        if (st != SPM_OK) return st;
        b->max_wpc[q] = bpc * (kDenseBlock / kWaveLanes);
    }
    for (Slot& s : b->slots) {
        bool ok = hipStreamCreateWithFlags(&s.stream, hipStreamNonBlocking) == hipSuccess &&
                  hipEventCreate(&s.ev0) == hipSuccess && hipEventCreate(&s.ev1) == hipSuccess;
        if (!ok) {
            for (Slot& t : b->slots) free_slot(t);
            return SPM_EHIP;
        }
        ok = hipHostMalloc(&s.h_stage, b->stage_bytes, hipHostMallocMapped | hipHostMallocCoherent) ==
                 hipSuccess &&
             hipHostMalloc(&s.h_res, sizeof(double) * kBatchRec * cfg->max_requests,
                           hipHostMallocMapped | hipHostMallocCoherent) == hipSuccess &&
             hipHostMalloc(&s.h_flag, sizeof(unsigned int) * cfg->max_requests,
                           hipHostMallocMapped | hipHostMallocCoherent) == hipSuccess &&
             hipMalloc(&s.d_arena, b->stage_bytes) == hipSuccess &&
             hipMalloc(&s.d_item, sizeof(double) * kBatchRec * (size_t)cfg->max_items) == hipSuccess &&
             hipMalloc(&s.d_counter, sizeof(unsigned int) * (64 + (size_t)cfg->max_requests)) == hipSuccess;
        if (!ok) {
            for (Slot& t : b->slots) free_slot(t);
            return SPM_ENOMEM;
        }
        std::memset(s.h_flag, 0, sizeof(unsigned int) * cfg->max_requests);
        if (hipHostGetDevicePointer((void**)&s.dh_res, s.h_res, 0) != hipSuccess ||
            hipHostGetDevicePointer((void**)&s.dh_flag, s.h_flag, 0) != hipSuccess ||
            hipHostGetDevicePointer((void**)&s.dh_stage, s.h_stage, 0) != hipSuccess) {
            for (Slot& t : b->slots) free_slot(t);
            return SPM_EHIP;
        }
    }
    *out = b.release();
    return SPM_OK;
}

extern "C" int spm_batch_destroy(spm_batch* b)
{
    if (!b) return SPM_OK;
    {
        std::lock_guard<std::mutex> lk(b->mu);
        if (!dry(b)) {
            DeviceGuard g(b->cfg.device);
            for (Slot& s : b->slots)
                if (s.stream) (void)hipStreamSynchronize(s.stream);
            for (Slot& s : b->slots) free_slot(s);
        }
        for (Slot& s : b->slots)
            for (Req* r : s.reqs) delete r;  // (null entries were handed out)
        for (Req* r : b->pending) delete r;
    }
    delete b;
    return SPM_OK;
}

extern "C" int spm_batch_get_tuning(const spm_batch* b, spm_batch_tuning* t)
{
    if (!b || !t) return SPM_EINVAL;
    *t = b->tune;
    return SPM_OK;
}

static int set_tuning_locked(spm_batch* b, const spm_batch_tuning* t)
{
    if (t->fused != 0 && t->fused != 1) return SPM_EINVAL;
    if (t->waves_per_cu < 0 || t->waves_per_cu > 64) return SPM_EINVAL;
    for (int k = 1; k < 4; ++k)
        if (t->log2_chunk[k] < 2 || t->log2_chunk[k] > 30) return SPM_EINVAL;
    for (const Slot& s : b->slots)
        if (s.busy) return SPM_EAGAIN;
    b->tune = *t;
    for (Slot& s : b->slots) free_graph(s);  // grids and kernels are baked into the graphs
    return SPM_OK;
}

extern "C" int spm_batch_set_tuning(spm_batch* b, const spm_batch_tuning* t)
{
    if (!b || !t) return SPM_EINVAL;
    std::lock_guard<std::mutex> lk(b->mu);
    const spm_batch_tuning was = b->tune;
    const int st = set_tuning_locked(b, t);
    for (int k = 1; st == SPM_OK && k < 4; ++k)  // (a value written back as it was read is no choice)
        if (t->log2_chunk[k] != was.log2_chunk[k]) b->chosen[k] = true;
    return st;
}

extern "C" int spm_batch_run(spm_batch* b, int count, const spm_request* reqs, spm_result* out)
{
    if (!b) return SPM_EINVAL;
    std::lock_guard<std::mutex> lk(b->mu);
    return drive(b, count, reqs, nullptr, out, nullptr, nullptr);
}

extern "C" int spm_batch_autotune(spm_batch* b, int count, const spm_request* sample, int reps, spm_batch_tuning* best,
                                  double* best_seconds)
{
    if (!b || count < 1 || !sample || reps < 1) return SPM_EINVAL;
    std::lock_guard<std::mutex> lk(b->mu);
    if (!idle(b)) return SPM_EAGAIN;
    std::vector<spm_result> out(count);
    auto time_it = [&](const spm_batch_tuning& t, int cnt, const spm_request* rq, double* sec) -> int {
        int st = set_tuning_locked(b, &t);
        if (st != SPM_OK) return st;
        double bestt = 1e300;
        for (int r = 0; r < reps + 1; ++r) {  // first pass warms up (graph capture, caches)
            const double t0 = now_seconds();
            st = drive(b, cnt, rq, nullptr, out.data(), nullptr, nullptr);
            const double dt = now_seconds() - t0;
            if (st != SPM_OK) return st;
            if (r > 0) bestt = std::min(bestt, dt);
        }
        *sec = bestt;
        return SPM_OK;
    };
    // A candidate whose launches fail on the device side (SPM_EHIP) is
    // dropped; the starting tuning and the winner must run.
    auto candidate = [&](const spm_batch_tuning& t, int cnt, const spm_request* rq, double* sec) -> int {
        const int rc = time_it(t, cnt, rq, sec);
        if (rc == SPM_EHIP) {
            *sec = 1e300;
            return SPM_OK;
        }
        return rc;
    };
    spm_batch_tuning cur = b->tune, win = cur;
    double win_s = 1e300;
    int st = time_it(cur, count, sample, &win_s);
    if (st != SPM_OK) return st;
    // 1) kernel organisation and persistent grid size.  The fused kernel
    // walks every kind in one shortest-first order, so a small request of
    // any kind finishes early; the per-kind kernels run one after another on
    // the slot's stream, so the last kind's requests wait for the others.
    // Fused is kept unless per-kind is faster by more than kLatencyMargin.
    spm_batch_tuning org_best[2] = {win, win};
    double org_s[2] = {1e300, 1e300};
    for (int fused = 0; fused <= 1; ++fused) {
        for (int wpc : {0, 4, 8, 12, 16}) {
            spm_batch_tuning t = win;
            t.fused = fused;
            t.waves_per_cu = wpc;
            double s = 0;
            st = candidate(t, count, sample, &s);
            if (st != SPM_OK) return st;
            if (s < org_s[fused]) {
                org_s[fused] = s;
                org_best[fused] = t;
            }
        }
    }
    const int org = org_s[1] <= org_s[0] * (1.0 + kLatencyMargin) ? 1 : 0;
    if (org_s[org] < 1e300) {  // (the starting tuning is one of the candidates)
        win_s = org_s[org];
        win = org_best[org];
    }
    // 2) chunk size per kind, timed on that kind's share of the sample: the
    // smallest L within kLatencyMargin of the fastest.  A smaller chunk
    // spreads a request over more lanes; on the serving mix, complex chunks
    // of 2^10 instead of 2^11 took p50 / p99 at 80 % load from 1.07 / 4.3 ms
    // to 0.78 / 3.7 ms for 1-3 % of throughput.
    for (int k = 1; k < 4; ++k) {
        std::vector<spm_request> sub;
        for (int i = 0; i < count; ++i)
            if (sample[i].kind == k) sub.push_back(sample[i]);
        if (sub.empty()) continue;
        struct AllFused {
            spm_batch* b;
            ~AllFused() { b->all_fused = false; }
        } scope{b};
        b->all_fused = (int)sub.size() < count;
        // (L, seconds), the starting chunk first: it must run, the others
        // are dropped (1e300) when their launches fail
        std::vector<std::pair<int, double>> tried(1, {win.log2_chunk[k], 0.0});
        st = time_it(win, (int)sub.size(), sub.data(), &tried[0].second);
        if (st != SPM_OK) return st;
        for (int L = 6; L <= 13; ++L) {
            if (L == win.log2_chunk[k]) continue;
            spm_batch_tuning t = win;
            t.log2_chunk[k] = L;
            double sec = 0;
            st = candidate(t, (int)sub.size(), sub.data(), &sec);
            if (st != SPM_OK) return st;
            tried.push_back({L, sec});
        }
        std::sort(tried.begin(), tried.end());
        double fastest = 1e300;
        for (const auto& c : tried) fastest = std::min(fastest, c.second);
        for (const auto& c : tried)
            if (c.second < 1e300 && c.second <= fastest * (1.0 + kLatencyMargin)) {
                win.log2_chunk[k] = c.first;
                break;
            }
    }
    st = time_it(win, count, sample, &win_s);
    if (st != SPM_OK) return st;
    if (best) *best = win;
    if (best_seconds) *best_seconds = win_s;
    return SPM_OK;
}

extern "C" int spm_serve_submit(spm_batch* b, const spm_request* req, uint64_t* ticket)
{
    if (!b) return SPM_EINVAL;
    std::lock_guard<std::mutex> lk(b->mu);
    return submit(b, req, now_seconds(), -1, ticket);
}

extern "C" int spm_serve_progress(spm_batch* b, int* in_flight)
{
    if (!b) return SPM_EINVAL;
    std::lock_guard<std::mutex> lk(b->mu);
    return progress(b, in_flight);
}

extern "C" int spm_serve_poll(spm_batch* b, spm_completion* out, int max, int* got)
{
    if (!b || !got || max < 0 || (max > 0 && !out)) return SPM_EINVAL;
    std::lock_guard<std::mutex> lk(b->mu);
    progress(b, nullptr);
    int k = 0;
    while (k < max && !b->done.empty()) {
        out[k++] = b->done.front();
        b->done.pop_front();
    }
    *got = k;
    return SPM_OK;
}

extern "C" int spm_serve_cancel(spm_batch* b, uint64_t ticket)
{
    if (!b) return SPM_EINVAL;
    std::lock_guard<std::mutex> lk(b->mu);
    auto it = b->live.find(ticket);
    if (it == b->live.end()) return SPM_EINVAL;
    it->second->cancelled = true;
    return SPM_OK;
}

extern "C" int spm_serve_pending(spm_batch* b, int* queued, int* in_flight)
{
    if (!b) return SPM_EINVAL;
    std::lock_guard<std::mutex> lk(b->mu);
    if (queued) *queued = (int)b->pending.size();
    if (in_flight) {
        int k = 0;
        for (const Slot& s : b->slots)
            if (s.busy)
                for (const Req* r : s.reqs) k += r ? 1 : 0;
        *in_flight = k;
    }
    return SPM_OK;
}

extern "C" int spm_serve_replay(spm_batch* b, int count, const spm_request* reqs, const double* arrival_s,
                                spm_result* out, double* latency_s, spm_serve_stats* stats)
{
    if (!b || !arrival_s) return SPM_EINVAL;
    for (int i = 1; i < count; ++i)
        if (arrival_s[i] < arrival_s[i - 1]) return SPM_EINVAL;
    std::lock_guard<std::mutex> lk(b->mu);
    return drive(b, count, reqs, arrival_s, out, latency_s, stats);
}

extern "C" const char* spm_batch_last_error(spm_batch* b)
{
    if (!b) return "";
    std::lock_guard<std::mutex> lk(b->mu);
    thread_local std::string copy;
    copy = b->last_error;
    return copy.c_str();
}

extern "C" int spm_batch_counters(spm_batch* b, uint64_t* late_publish, uint64_t* retried)
{
    if (!b) return SPM_EINVAL;
    std::lock_guard<std::mutex> lk(b->mu);
    if (late_publish) *late_publish = b->late_publish;
    if (retried) *retried = b->retried;
    return SPM_OK;
}

extern "C" int spm_batch_inject_fault(spm_batch* b, int launches)
{
    if (!b || launches < 0) return SPM_EINVAL;
    std::lock_guard<std::mutex> lk(b->mu);
    b->fault_launches = launches;
    return SPM_OK;
}

extern "C" int spm_batch_inject_bad_results(spm_batch* b, int results)
{
    if (!b || results < 0) return SPM_EINVAL;
    std::lock_guard<std::mutex> lk(b->mu);
    b->bad_results = results;
    return SPM_OK;
}
