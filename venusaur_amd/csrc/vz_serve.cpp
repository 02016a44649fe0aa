// vz_serve.cpp -- the serving form and the autotuner.
//
// Serving: a host thread owns a few streams, each with the buffers of its
// launches (a slot).  Requests are queued FIFO by vzServerSubmit; whenever a
// slot is idle the requests at the head of the queue that fit it and the HBM
// budget are rendered as one launch on its stream, at once and beside the
// launches of the other slots, which the GPU works through in the order they
// came: new work overlaps with requests already on the GPU (continuous
// batching) and takes over the CUs that finishing launches leave.  BVHs stay
// resident (vzScene objects owned by the caller) and the slots' buffers are
// kept, so admission and release never synchronise the device.  The nearest
// reference analogue is the interactive loop that keeps the GAS and
// accumulator resident across frames (Core/Core.cpp:358-430,
// Core/Renderer.h:37-54).
//
// Autotuner: times the caller's batch over candidate buffer sizes, camera
// tiles and refill thresholds and keeps the fastest (segments per
// millisecond), cached per context.
#include <algorithm>
#include <chrono>
#include <condition_variable>
#include <cstring>
#include <deque>
#include <thread>
#include <unordered_map>

#include "vz_internal.h"
#include "vz_path.h"

using namespace vz;

namespace {

struct Pending {
    uint64_t id;
    const vzScene_st* scene;
    vzLaunchParams params;
    size_t bytes;
    double submit_ms;
};

struct Active {
    uint64_t id;
    const vzScene_st* scene;
    size_t bytes;
    double submit_ms, admit_ms;
};

// Requests rendered by one launch, or one request of several launches.
struct Flight {
    PathSlot slot;
    hipStream_t stream = nullptr;
    Event done{hipEventDisableTiming};
    std::vector<Active> active;  // empty: idle
    bool large = false;
};

// Launches side by side: the second takes over the CUs that the first one's
// last paths leave.  A burst of 20 requests (1k to 200k spheres, 256 to 1024
// pixels square, 4 to 64 samples, one of 1088) took 195 ms with 2, 209 with
// 1, 202 with 3 and 203 with 4.
constexpr uint32_t kServeStreams = 2;
// Paths of a launch of several requests at most.  A launch's requests finish
// together: the burst's p50 latency is 92 ms at 8M paths, 101 at 32M and 116
// at 64M, its throughput the same within 1%.
constexpr uint64_t kServeGroupPaths = 16u << 20;

}  // namespace

struct vzServer_st {
    vzContext ctx = nullptr;
    vzServeConfig cfg{};
    PathWork* work = nullptr;
    PathOptions opt;
    uint64_t slot_budget = 0;
    std::vector<Flight> flights;
    std::thread worker;
    std::mutex mu;
    std::condition_variable cv_work, cv_done;
    std::deque<Pending> pending;
    std::unordered_map<uint64_t, vzRequestResult> results;
    size_t n_active = 0;
    uint64_t next_id = 1;
    size_t used_bytes = 0;
    bool stop = false;
    vzStatus fatal = VZ_SUCCESS;
    std::string fatal_msg;
    std::chrono::steady_clock::time_point t0;

    double now_ms() const
    {
        return std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    }
    void loop();
    std::vector<Pending> admit();
    vzStatus start(Flight& f, const std::vector<Pending>& group);
    void harvest(Flight& f);
    // A request no longer needs its scene (finished, rejected or dropped).
    static void release_scene(const vzScene_st* sc)
    {
        const_cast<vzScene_st*>(sc)->server_refs.fetch_sub(1);
    }
    // A request that will never run (mu held).
    void reject(const Pending& p, vzStatus status)
    {
        release_scene(p.scene);
        vzRequestResult r{};
        r.request_id = p.id;
        r.submit_ms = p.submit_ms;
        r.admit_ms = r.finish_ms = now_ms();
        r.status = status;
        results[p.id] = r;
    }
    ~vzServer_st()
    {
        for (Flight& f : flights) {
            f.slot.free();
            if (f.stream) (void)hipStreamDestroy(f.stream);
        }
    }
};

// The next launch's requests, in arrival order, while they fit the budget,
// the table and the slot (mu held).
std::vector<Pending> vzServer_st::admit()
{
    std::vector<Pending> group;
    uint64_t paths = 0;
    const uint64_t most = std::min<uint64_t>(slot_budget / kPathBytes, kServeGroupPaths);
    while (!pending.empty() && n_active < cfg.max_active) {
        const Pending& p = pending.front();
        if (p.bytes > cfg.hbm_budget_bytes) {  // can never fit
            reject(p, VZ_ERROR_CAPACITY);
            pending.pop_front();
            continue;
        }
        if (used_bytes + p.bytes > cfg.hbm_budget_bytes) break;  // wait for memory
        const uint64_t n = path_count(p.params, opt);
        if (!group.empty() && paths + n > most) break;
        paths += n;
        used_bytes += p.bytes;
        n_active++;
        group.push_back(p);
        pending.pop_front();
        if (paths > most) break;  // a large request renders by itself
    }
    return group;
}

vzStatus vzServer_st::start(Flight& f, const std::vector<Pending>& group)
{
    std::vector<PathItem> items;
    std::vector<const PathItem*> ptr;
    items.reserve(group.size());
    for (const Pending& p : group) items.push_back(PathItem{p.scene, p.params});
    for (const PathItem& it : items) ptr.push_back(&it);
    uint64_t paths = 0;
    for (const PathItem& it : items) paths += path_count(it.params, opt);
    f.slot.used = 0;
    f.large = group.size() == 1 && paths * kPathBytes > slot_budget;
    if (f.large) {
        uint64_t budget = slot_budget;
        uint32_t passes = 0;
        VZ_TRY(path_reserve_one(f.slot, items[0], opt, &budget, 0, &passes));
        return path_enqueue_one(work, f.slot, items[0], opt, passes, false, f.stream, nullptr);
    }
    VZ_TRY(slot_reserve(f.slot, paths));
    return path_enqueue_many(work, f.slot, ptr.data(), (uint32_t)ptr.size(), opt, false, f.stream);
}

// Results of a flight whose launches have finished.
void vzServer_st::harvest(Flight& f)
{
    std::lock_guard<std::mutex> lk(mu);
    const double t = now_ms();
    for (size_t i = 0; i < f.active.size(); i++) {
        const Active& a = f.active[i];
        release_scene(a.scene);
        vzRequestResult r{};
        r.request_id = a.id;
        r.submit_ms = a.submit_ms;
        r.admit_ms = a.admit_ms;
        r.finish_ms = t;
        r.segments = f.large ? f.slot.h_totals[0] : f.slot.h_totals[kPathStats + i];
        r.status = VZ_SUCCESS;
        results[a.id] = r;
        used_bytes -= a.bytes;
        n_active--;
    }
    f.active.clear();
    cv_done.notify_all();
}

void vzServer_st::loop()
{
    (void)hipSetDevice(ctx->device);
    auto fail = [&](vzStatus s) {
        std::lock_guard<std::mutex> lk(mu);
        fatal = s;
        fatal_msg = vzGetLastError();
        stop = true;
        cv_done.notify_all();
    };
    for (;;) {
        bool progress = false, busy = false;
        // 1. finished launches
        for (Flight& f : flights) {
            if (f.active.empty()) continue;
            const hipError_t e = hipEventQuery(f.done.e);
            if (e == hipSuccess) {
                harvest(f);
                progress = true;
            } else if (e == hipErrorNotReady) {
                busy = true;
            } else {
                set_error(VZ_ERROR_HIP, std::string("a launch failed: ") + hipGetErrorString(e));
                fail(VZ_ERROR_HIP);
                goto out;
            }
        }
        // 2. queued requests onto idle slots
        for (Flight& f : flights) {
            if (!f.active.empty()) continue;
            std::vector<Pending> group;
            {
                std::lock_guard<std::mutex> lk(mu);
                if (pending.empty()) break;
                group = admit();
                const double t = now_ms();
                for (const Pending& p : group)
                    f.active.push_back(Active{p.id, p.scene, p.bytes, p.submit_ms, t});
                if (group.empty()) {
                    cv_done.notify_all();  // rejected ones, if any
                    break;
                }
            }
            const vzStatus s = start(f, group);
            if (s == VZ_ERROR_CAPACITY || s == VZ_ERROR_OUT_OF_MEMORY) {
                // nothing of the group was enqueued beyond what the stream
                // finishes: wait for it, and for memory if others run
                (void)hipStreamSynchronize(f.stream);
                std::lock_guard<std::mutex> lk(mu);
                f.active.clear();
                for (auto p = group.rbegin(); p != group.rend(); ++p) {
                    used_bytes -= p->bytes;
                    n_active--;
                    if (busy || group.size() > 1) pending.push_front(*p);
                    else reject(*p, s);
                }
                if (!busy && group.size() > 1) {
                    // even an idle device does not hold the group: fewer at a time
                    slot_budget = std::max<uint64_t>(slot_budget / 2, kPathBytes);
                    progress = true;
                }
                cv_done.notify_all();
                break;
            }
            if (s != VZ_SUCCESS || hipEventRecord(f.done.e, f.stream) != hipSuccess) {
                if (s == VZ_SUCCESS) set_error(VZ_ERROR_HIP, "hipEventRecord failed");
                fail(VZ_ERROR_HIP);
                goto out;
            }
            progress = busy = true;
        }
        if (progress) continue;
        // 3. nothing to do: wait for a submission, or a moment for the GPU
        std::unique_lock<std::mutex> lk(mu);
        if (busy) {
            cv_work.wait_for(lk, std::chrono::microseconds(20));
        } else {
            if (pending.empty()) {
                cv_done.notify_all();
                if (stop) break;
                cv_work.wait(lk, [&] { return stop || !pending.empty(); });
            }
        }
    }
out:
    for (Flight& f : flights) (void)hipStreamSynchronize(f.stream);
}

extern "C" {

vzStatus vzServerCreate(vzContext ctx, const vzServeConfig* cfg, vzServer* out)
{
    if (!ctx || !cfg || !out) return set_error(VZ_ERROR_INVALID_VALUE, "NULL argument");
    *out = nullptr;
    VZ_HIP_TRY(hipSetDevice(ctx->device));
    vzServer s = new vzServer_st();
    s->ctx = ctx;
    s->cfg = *cfg;
    if (s->cfg.max_active == 0 || s->cfg.max_active > kMaxRequests) s->cfg.max_active = kMaxRequests;
    if (s->cfg.hbm_budget_bytes == 0) s->cfg.hbm_budget_bytes = ctx->hbm_bytes / 2;
    // Serving defaults: the memory of a 48M-ray queue (4.8 GB) over the
    // streams, 8x8 camera tiles
    vzTuning t = s->cfg.tuning;
    if (t.queue_capacity == 0) t.queue_capacity = 12u << 22;
    s->opt.tile_w = t.tile_w ? t.tile_w : 8u;
    s->opt.tile_h = t.tile_h ? t.tile_h : 8u;
    s->opt.refill = std::min<uint32_t>(t.refill_lanes, 65u);  // 0: the kernel variant's default
    const uint32_t n = std::min<uint32_t>(kServeStreams, s->cfg.max_active);
    s->slot_budget = tuning_budget(t) / kServeStreams;
    vzStatus rs;
    {
        std::lock_guard<std::mutex> lk(ctx->mu);
        rs = path_work(ctx, &s->work);
    }
    s->flights = std::vector<Flight>(n);
    for (Flight& f : s->flights) {
        if (rs == VZ_SUCCESS && !f.done.ok()) rs = set_error(VZ_ERROR_HIP, "hipEventCreate failed");
        if (rs == VZ_SUCCESS && hipStreamCreateWithFlags(&f.stream, hipStreamNonBlocking) != hipSuccess)
            rs = set_error(VZ_ERROR_HIP, "hipStreamCreateWithFlags failed");
        if (rs == VZ_SUCCESS) rs = f.slot.init(ctx, true);
        if (rs == VZ_SUCCESS) rs = slot_reserve(f.slot, s->slot_budget / kPathBytes);
    }
    if (rs != VZ_SUCCESS) {
        delete s;
        return rs;
    }
    s->t0 = std::chrono::steady_clock::now();
    s->worker = std::thread([s] { s->loop(); });
    ctx->live_servers++;
    *out = s;
    return VZ_SUCCESS;
}

vzStatus vzServerSubmit(vzServer srv, vzScene scene, const vzLaunchParams* params, uint64_t* request_id)
{
    if (!srv || !scene || !params || !request_id) return set_error(VZ_ERROR_INVALID_VALUE, "NULL argument");
    if (scene->ctx != srv->ctx) return set_error(VZ_ERROR_INVALID_VALUE, "scene belongs to another context");
    VZ_TRY(check_launch_params(params));
    if (params->flags & VZ_MEGAKERNEL) return set_error(VZ_ERROR_INVALID_VALUE, "VZ_MEGAKERNEL is not a serving mode");
    std::lock_guard<std::mutex> lk(srv->mu);
    if (srv->fatal != VZ_SUCCESS) return set_error(srv->fatal, "server stopped: " + srv->fatal_msg);
    Pending p;
    p.id = srv->next_id++;
    p.scene = scene;
    scene->server_refs.fetch_add(1);  // vzSceneDestroy refuses until the request is done
    p.params = *params;
    p.bytes = request_bytes(*params);
    p.submit_ms = srv->now_ms();
    srv->pending.push_back(p);
    *request_id = p.id;
    srv->cv_work.notify_one();
    return VZ_SUCCESS;
}

vzStatus vzServerPoll(vzServer srv, uint64_t request_id, vzRequestResult* out)
{
    if (!srv || !out) return set_error(VZ_ERROR_INVALID_VALUE, "NULL argument");
    std::lock_guard<std::mutex> lk(srv->mu);
    auto it = srv->results.find(request_id);
    if (it == srv->results.end()) {
        if (request_id == 0 || request_id >= srv->next_id) return set_error(VZ_ERROR_INVALID_VALUE, "unknown request id");
        if (srv->fatal != VZ_SUCCESS) return set_error(srv->fatal, "server stopped: " + srv->fatal_msg);
        return VZ_ERROR_NOT_READY;
    }
    *out = it->second;
    return VZ_SUCCESS;
}

vzStatus vzServerDrain(vzServer srv)
{
    if (!srv) return set_error(VZ_ERROR_INVALID_VALUE, "NULL argument");
    std::unique_lock<std::mutex> lk(srv->mu);
    srv->cv_done.wait(lk, [&] {
        return srv->fatal != VZ_SUCCESS || (srv->pending.empty() && srv->n_active == 0);
    });
    if (srv->fatal != VZ_SUCCESS) return set_error(srv->fatal, "server stopped: " + srv->fatal_msg);
    return VZ_SUCCESS;
}

vzStatus vzServerDestroy(vzServer srv)
{
    if (!srv) return set_error(VZ_ERROR_INVALID_VALUE, "NULL argument");
    {
        std::lock_guard<std::mutex> lk(srv->mu);
        srv->stop = true;
        srv->cv_work.notify_all();
    }
    if (srv->worker.joinable()) srv->worker.join();
    // after a fatal error requests may remain; they will never run
    for (const Pending& p : srv->pending) vzServer_st::release_scene(p.scene);
    for (const Flight& f : srv->flights)
        for (const Active& a : f.active) vzServer_st::release_scene(a.scene);
    srv->ctx->live_servers--;
    delete srv;
    return VZ_SUCCESS;
}

vzStatus vzAutotune(vzContext ctx, const vzBatchItem* items, uint32_t n, vzStream stream, vzTuning* out)
{
    if (!ctx || !items || n == 0 || !out) return set_error(VZ_ERROR_INVALID_VALUE, "NULL argument or empty batch");
    // Times the batch itself, twice per candidate, and keeps each
    // candidate's faster run: the candidates are often within a few percent,
    // and a single run let the noise pick.  The render time starts after the
    // buffers are allocated, so no warm-up run is needed.
    std::vector<vzBatchItem> probe(items, items + n);
    for (auto& it : probe) it.params.flags &= ~(uint32_t)(VZ_COUNT_VISITS | VZ_TIME_STAGES);
    vzTuning best{};
    double best_rate = -1.0;
    auto time = [&](const vzTuning& cand) -> vzStatus {
        double rate = 0.0;
        for (int rep = 0; rep < 2; rep++) {
            vzStats st{};
            VZ_TRY(vzBatchLaunch(ctx, probe.data(), n, &cand, stream, &st));
            if (st.render_ms > 0.0) rate = std::max(rate, (double)st.segments / st.render_ms);
        }
        if (rate > best_rate) {
            best_rate = rate;
            best = cand;
        }
        return VZ_SUCCESS;
    };
    // stage 1: buffer size x camera tile at the default refill
    const uint32_t caps[] = {1u << 22, 1u << 23, 3u << 22, 6u << 22, 8u << 22, 12u << 22};
    const uint32_t tiles[][2] = {{32, 2}, {16, 4}, {8, 8}};
    for (uint32_t cap : caps)
        for (auto& t : tiles) {
            vzTuning cand{};
            cand.queue_capacity = cap;
            cand.tile_w = t[0];
            cand.tile_h = t[1];
            cand.iters_per_graph = 16;
            cand.refill_lanes = 0;
            cand.slice_split = 4;
            VZ_TRY(time(cand));
        }
    // stage 2: at the best of those, the refill threshold
    const vzTuning base = best;
    for (uint32_t refill : {25u, 33u, 49u, 57u}) {
        vzTuning cand = base;
        cand.refill_lanes = refill;
        VZ_TRY(time(cand));
    }
    {
        std::lock_guard<std::mutex> lk(ctx->mu);
        ctx->tuning = best;
        ctx->tuned = true;
    }
    tuning_cache_store(ctx, best);
    *out = best;
    return VZ_SUCCESS;
}

}  // extern "C"
