// vz_serve.cpp -- the serving form and the autotuner.
//
// Serving: a host thread owns a few streams, each with the buffers of its
// launches (a slot).  Requests are queued FIFO by vzServerSubmit and admitted
// while they fit the HBM budget.  Whenever a slot is idle the admitted requests
// next in turn are rendered as one launch on its stream, at once and beside the
// launches of the other slots, which the GPU works through in the order they
// came: new work overlaps with requests already on the GPU (continuous
// batching) and takes over the CUs that finishing launches leave.  A request of
// more paths than a launch takes is rendered a slice of its passes at a time
// and goes to the end of the queue between them, so that no request waits for
// another to finish.  BVHs stay resident (vzScene objects owned by the caller)
// and the slots' buffers are kept, so admission and release never synchronise
// the device.  The nearest reference analogue is the interactive loop that
// keeps the GAS and accumulator resident across frames (Core/Core.cpp:358-430,
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
#include <memory>
#include <thread>
#include <unordered_map>

#include "vz_internal.h"
#include "vz_path.h"

using namespace vz;

namespace {

struct Request {
    uint64_t id;
    PathItem item;
    size_t bytes;               // counted against the budget
    uint64_t npad;              // its pixels, padded
    double submit_ms, admit_ms = 0.0;
    uint32_t done = 0;          // passes rendered or in flight
    char* carry = nullptr;      // what its slices hand on
    size_t carry_size = 0;
    unsigned long long segments = 0;

    uint32_t left() const { return item.params.samples_per_pixel - done; }
};
using RequestPtr = std::unique_ptr<Request>;

struct Share {                  // of a request, in a launch
    RequestPtr r;
    uint32_t s0, ns;
};

// One launch.
struct Flight {
    PathSlot slot;
    hipStream_t stream = nullptr;
    Event done{hipEventDisableTiming};
    std::vector<Share> shares;  // empty: idle
};

// Launches side by side: the second takes over the CUs that the first one's
// last paths leave.  A burst of 20 requests (1k to 200k spheres, 256 to 1024
// pixels square, 4 to 64 samples, one of 1088) takes 153.6 ms with 1, 141.1 with
// 2 and 144.2 with 3.
constexpr uint32_t kServeStreams = 2;

}  // namespace

struct vzServer_st {
    vzContext ctx = nullptr;
    vzServeConfig cfg{};
    PathWork* work = nullptr;
    PathOptions opt;
    uint64_t footprint_slice = kServeSlicePaths;  // by the tuning
    // paths of a launch of several requests, of a slice, and of a slice of a
    // request that has the server to itself: its slices follow one another, so
    // it takes as many as the tuning's memory holds (1080p at 512 samples: 474
    // ms in launches of 150M, 493 of 64M).  Lower where memory is short (the
    // worker's)
    uint64_t launch_paths = kServePaths, slice_paths = kServeSlicePaths, alone_paths = kServeSlicePaths;
    bool trimmed = false;              // idle slots have made room for the next launch (the worker's)
    std::vector<Flight> flights;
    std::thread worker;
    std::mutex mu;
    std::condition_variable cv_work, cv_done;
    std::deque<RequestPtr> pending;    // in arrival order
    std::deque<RequestPtr> ready;      // admitted, in turn (the worker's)
    std::unordered_map<uint64_t, vzRequestResult> results;
    size_t n_active = 0;
    uint64_t next_id = 1;
    size_t used_bytes = 0;             // footprints of the admitted
    size_t carried = 0;                // allocated for slices (the worker's)
    bool stop = false;
    vzStatus fatal = VZ_SUCCESS;
    std::string fatal_msg;
    std::chrono::steady_clock::time_point t0;

    double now_ms() const
    {
        return std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    }
    void loop();
    void admit();
    uint64_t pick(Flight& f, uint64_t most, uint64_t slice);
    bool make_room(Flight& f, size_t slot, size_t carry);
    void free_carry(Request& r, hipStream_t st)
    {
        if (!r.carry) return;
        (void)hipFreeAsync(r.carry, st);
        carried -= r.carry_size;
        r.carry = nullptr;
    }
    vzStatus start(Flight& f);
    void put_back(Flight& f);
    void harvest(Flight& f);
    bool others_busy(const Flight& f) const
    {
        for (const Flight& o : flights)
            if (&o != &f && !o.shares.empty()) return true;
        return false;
    }
    // A request no longer needs its scene (finished, rejected or dropped).
    static void release_scene(const Request& r)
    {
        const_cast<vzScene_st*>(r.item.scene)->server_refs.fetch_sub(1);
    }
    // A request is over (mu held).
    void finish(const Request& r, vzStatus status)
    {
        release_scene(r);
        vzRequestResult out{};
        out.request_id = r.id;
        out.submit_ms = r.submit_ms;
        out.finish_ms = now_ms();
        out.admit_ms = r.admit_ms > 0.0 ? r.admit_ms : out.finish_ms;
        out.segments = r.segments;
        out.status = status;
        results[r.id] = out;
    }
    ~vzServer_st()
    {
        // after a fatal error requests may remain; they will never run
        for (const RequestPtr& r : pending) release_scene(*r);
        for (const RequestPtr& r : ready) drop(*r);
        for (Flight& f : flights)
            for (const Share& s : f.shares) drop(*s.r);
        for (Flight& f : flights) {
            f.slot.free();
            if (f.stream) (void)hipStreamDestroy(f.stream);
        }
    }
    void drop(Request& r)
    {
        release_scene(r);
        free_carry(r, flights.front().stream);
    }
};

// Queued requests, in arrival order, while they fit the budget.
void vzServer_st::admit()
{
    std::lock_guard<std::mutex> lk(mu);
    while (!pending.empty() && n_active < cfg.max_active) {
        Request& p = *pending.front();
        if (p.bytes > cfg.hbm_budget_bytes || p.npad > kMaxLaunchPaths) {  // can never fit
            finish(p, VZ_ERROR_CAPACITY);
            pending.pop_front();
            cv_done.notify_all();
            continue;
        }
        if (used_bytes + p.bytes > cfg.hbm_budget_bytes) break;  // wait for memory
        p.admit_ms = now_ms();
        used_bytes += p.bytes;
        n_active++;
        ready.push_back(std::move(pending.front()));
        pending.pop_front();
    }
}

// The requests next in turn, as many as a launch of `most` paths takes; returns
// their paths.  A request of more has a launch to itself, whole or, above `slice`
// paths, one of as few equal slices as there can be.
uint64_t vzServer_st::pick(Flight& f, uint64_t most, uint64_t slice)
{
    uint64_t paths = 0;
    while (!ready.empty() && f.shares.size() < kMaxRequests) {
        Request& r = *ready.front();
        const uint64_t left = r.left();
        uint64_t take = left;
        if (paths + r.npad * left > most) {
            if (!f.shares.empty()) break;
            take = slice_passes(left, r.npad, slice);
        }
        paths += r.npad * take;
        f.shares.push_back(Share{std::move(ready.front()), r.done, (uint32_t)take});
        ready.pop_front();
        if (take < left) break;
    }
    return paths;
}

void vzServer_st::put_back(Flight& f)
{
    while (!f.shares.empty()) {
        ready.push_front(std::move(f.shares.back().r));
        f.shares.pop_back();
    }
}

// Whether the budget has room for a flight's slot of `slot` bytes and `carry`
// more for slices.  Slots keep the size of their largest launch; where that
// leaves no room, those of idle flights go.
bool vzServer_st::make_room(Flight& f, size_t slot, size_t carry)
{
    for (;;) {
        size_t total = carried + carry + std::max(slot, f.slot.paths_bytes);
        Flight* idle = f.slot.paths_bytes > slot ? &f : nullptr;
        for (Flight& o : flights) {
            if (&o == &f) continue;
            total += o.slot.paths_bytes;
            if (o.shares.empty() && o.slot.paths_bytes) idle = &o;
        }
        if (total <= cfg.hbm_budget_bytes) return true;
        if (!idle) return false;
        slot_drop(idle->slot);
    }
}

// Renders the requests next in turn on an idle flight.  VZ_ERROR_OUT_OF_MEMORY:
// they are back in the queue.
vzStatus vzServer_st::start(Flight& f)
{
    bool alone;
    {
        std::lock_guard<std::mutex> lk(mu);
        alone = ready.size() == 1 && pending.empty() && !others_busy(f);
    }
    uint64_t paths = 0;
    size_t carry = 0;
    vzStatus rs = VZ_SUCCESS;
    for (;;) {
        paths = alone ? pick(f, alone_paths, alone_paths) : pick(f, launch_paths, slice_paths);
        const Share& s = f.shares.front();
        carry = !s.r->carry && s.ns < s.r->item.params.samples_per_pixel ? carry_bytes(s.r->item.params, s.r->npad) : 0;
        if (make_room(f, slot_bytes(paths), carry)) break;
        put_back(f);
        if (!alone) return set_error(VZ_ERROR_OUT_OF_MEMORY, "the budget has no room for a launch");
        alone = false;
    }
    Request& first = *f.shares.front().r;
    rs = slot_reserve(f.slot, paths);
    if (rs == VZ_SUCCESS && carry) {
        if (hipMallocAsync((void**)&first.carry, carry, f.stream) == hipSuccess) {
            first.carry_size = carry;
            carried += carry;
        } else {
            (void)hipGetLastError();
            first.carry = nullptr;
            ctx->scene_blocks.trim();
            rs = set_error(VZ_ERROR_OUT_OF_MEMORY, "no memory for the sums of a request");
        }
    }
    if (rs == VZ_SUCCESS) {
        std::vector<PathSlice> slices;
        for (const Share& s : f.shares) slices.push_back(PathSlice{&s.r->item, s.s0, s.ns, s.r->carry});
        PathOptions o = opt;
        for (const Share& s : f.shares) o.count |= !ordered_paths(s.r->item);
        f.slot.used = 0;
        rs = path_enqueue_many(work, f.slot, slices.data(), (uint32_t)slices.size(), o, false, f.stream);
    }
    if (rs == VZ_ERROR_OUT_OF_MEMORY) {
        put_back(f);
        return rs;
    }
    if (rs == VZ_SUCCESS && hipEventRecord(f.done.e, f.stream) != hipSuccess)
        rs = set_error(VZ_ERROR_HIP, "hipEventRecord failed");
    for (Share& s : f.shares) s.r->done += s.ns;
    return rs;
}

// A flight's launch has finished.
void vzServer_st::harvest(Flight& f)
{
    std::lock_guard<std::mutex> lk(mu);
    const uint32_t n = (uint32_t)f.shares.size();
    for (uint32_t i = 0; i < n; i++) {
        RequestPtr r = std::move(f.shares[i].r);
        r->segments += slice_segments(f.slot, n, i);
        if (r->left()) {
            ready.push_back(std::move(r));
            continue;
        }
        free_carry(*r, f.stream);
        used_bytes -= r->bytes;
        n_active--;
        finish(*r, VZ_SUCCESS);
    }
    f.shares.clear();
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
        // 1. finished launches; requests that came meanwhile go before those
        // whose turn ends
        admit();
        for (Flight& f : flights) {
            if (f.shares.empty()) continue;
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
        if (progress) admit();
        // 2. the next launches onto idle slots
        for (Flight& f : flights) {
            if (!f.shares.empty() || ready.empty()) continue;
            const vzStatus s = start(f);
            if (s == VZ_ERROR_OUT_OF_MEMORY) {
                if (others_busy(f)) break;  // until one of them has finished
                // even an idle device does not hold the launch beside the slots:
                // without them, then fewer paths at a time, down to one pass of
                // one request
                for (Flight& o : flights) slot_drop(o.slot);
                if (!trimmed) {
                    trimmed = true;
                } else if (alone_paths > slice_paths) {
                    alone_paths = slice_paths;
                } else if (slice_paths > ready.front()->npad) {
                    launch_paths = std::max<uint64_t>(launch_paths / 2, 1);
                    alone_paths = slice_paths = slice_paths / 2;
                } else {
                    std::lock_guard<std::mutex> lk(mu);
                    Request& r = *ready.front();
                    free_carry(r, f.stream);
                    used_bytes -= r.bytes;
                    n_active--;
                    finish(r, s);
                    ready.pop_front();
                    cv_done.notify_all();
                }
                progress = true;
                break;
            }
            if (s != VZ_SUCCESS) {
                fail(s);
                goto out;
            }
            trimmed = false;
            progress = busy = true;
        }
        if (progress) continue;
        // 3. nothing to do: wait for a submission, or a moment for the GPU
        std::unique_lock<std::mutex> lk(mu);
        if (busy) {
            cv_work.wait_for(lk, std::chrono::microseconds(20));
        } else if (pending.empty()) {
            cv_done.notify_all();
            if (stop) break;
            cv_work.wait(lk, [&] { return stop || !pending.empty(); });
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
    const uint64_t slot_paths = std::max<uint64_t>(tuning_budget(t) / kServeStreams / kPathBytes, 1);
    s->launch_paths = std::min(kServePaths, slot_paths);
    s->footprint_slice = s->slice_paths = std::min(kServeSlicePaths, slot_paths);
    s->alone_paths = slot_paths;
    // what a flight starts with; larger ones as launches need them
    const uint64_t share = s->cfg.hbm_budget_bytes / kServeStreams;
    const uint64_t first = std::min(s->slice_paths, share > slot_bytes(0) ? (share - slot_bytes(0)) / kPathBytes : 0);
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
        if (rs == VZ_SUCCESS) rs = slot_reserve(f.slot, first);
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
    RequestPtr p(new Request());
    p->id = srv->next_id++;
    p->item = PathItem{scene, *params};
    scene->server_refs.fetch_add(1);  // vzSceneDestroy refuses until the request is done
    p->bytes = request_bytes(*params, srv->opt, srv->footprint_slice);
    p->npad = padded_pixels(*params, srv->opt);
    p->submit_ms = srv->now_ms();
    *request_id = p->id;
    srv->pending.push_back(std::move(p));
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
    vzContext ctx = srv->ctx;
    delete srv;
    ctx->live_servers--;
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
