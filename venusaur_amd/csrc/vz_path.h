// vz_path.h -- rendering as persistent path tracing, shared by the plain
// launch (vzLaunch), the batched form (vzBatchLaunch) and the serving loop.
// vz_path.hip says how a launch works and why; this file is its host side.
//
// A slot holds the buffers of the launches that are enqueued on one stream:
// each launch uses them after the one before it on that stream, so a slot
// belongs to one stream at a time.
#pragma once
#include <vector>

#include "vz_device.h"
#include "vz_internal.h"

namespace vz {

constexpr int kPathStats = 4;         // segments, hits, node visits, sphere tests
// Device memory per path of a launch: its camera seed and its radiance.
constexpr uint64_t kPathBytes = 16;
// vzTuning.queue_capacity counts rays in flight at 96 bytes each; a batch or
// a server keeps the paths of its launches in as much memory.
constexpr uint64_t kRayBytes = 96;
// A plain launch: 4 GiB hold 129 passes of a 1080p frame.
constexpr uint64_t kPlainBudget = 4ull << 30;
// The most a slot is used for, beyond one pass of a large image.
constexpr uint64_t kMaxSlotBudget = 16ull << 30;
constexpr uint64_t kMaxLaunchPaths = 0xFFFFFF00ull;  // a path's index has 32 bits

// Paths of a server's launch of several requests, and of a slice of one request,
// at most.  A launch's requests finish together and the next in turn start after
// it; each launch's end leaves part of the GPU idle.  Launches and slices of up
// to 16M, 32M, 48M, 64M and 128M: a burst of 20 requests (vz_serve.cpp) takes
// 147.9, 143.6, 140.8, 139.5 and 139.4 ms, 600 such requests at 0.8 of the
// capacity have a p50 of 102, 174, 234, 292 and 489 ms, and 256x256 at 4 samples
// behind two 1080p frames at 512 samples takes 11, 25, 24, 10 to 39 and 38 to 165
// ms.  With 48M and 72M 139.6, 287 and 12 to 79, and bursts of 2 to 5 requests,
// one of 71M paths, take 2 to 4% less than with 48M for both.  (Requests up to
// 150M paths whole, in order of arrival: 141.2, 923 and 724 ms.)
constexpr uint64_t kServePaths = 48u << 20;
constexpr uint64_t kServeSlicePaths = kServePaths + kServePaths / 2;

struct PathReq {               // one request of a launch, read by scalar loads
    Cam cam;
    uint32_t subframe, max_depth, spp, fp64;
    uint32_t lw;               // camera tiles are 2^lw x 2^(6 - lw) pixels
    uint32_t tiles_x, npad;    // npad: pixels of all tiles
    uint32_t s0, ns;           // the launch's passes [s0, s0 + ns)
    uint32_t spu, groups;      // passes per unit, units per tile
    uint32_t parts;            // log2 of the units that share a pass of a tile (spu 1)
    uint32_t unit0, pix0, slot0;  // its first unit, padded pixel and path in the launch
    uint32_t* camseed;         // npad: camera seed of the next launch's first pass (ns < spp)
    void* sums;                // 3 * npad float or double, carried between launches (ns < spp)
    void* accum;
    uint32_t* image;
    SceneView sc;
};

struct PathSlot {
    vzContext ctx = nullptr;
    char* paths = nullptr;     // seeds and radiances
    size_t paths_bytes = 0;
    char* pixels = nullptr;    // camera seeds and sums carried between the launches of one request
    size_t pixels_bytes = 0;
    unsigned long long* stats = nullptr;     // per workgroup, the unit counters, segments per request
    unsigned long long* h_totals = nullptr;  // pinned: kPathStats, then segments per request
    PathReq* reqs = nullptr;   // request table (many requests in one launch)
    PathReq* h_reqs = nullptr; // pinned staging of it
    uint32_t used = 0;         // its entries given to launches not yet waited for

    vzStatus init(vzContext c, bool table);
    void free();
};

struct PathItem {
    const vzScene_st* scene;
    vzLaunchParams params;
};

// Passes [s0, s0 + ns) of a request: one launch's share of it.  carry holds
// its sums and camera seeds from slice to slice (carry_bytes), and may be null
// for a slice of all passes.
struct PathSlice {
    const PathItem* item;
    uint32_t s0, ns;
    char* carry;
};

struct PathOptions {
    uint32_t refill = 0;       // 0: the kernel variant's default
    uint32_t tile_w = 8, tile_h = 8;
    bool count = false;        // count node visits and sphere tests; test spheres in the one order
    std::vector<Event>* events = nullptr;  // appended to: a pair around every k_path launch
};

struct RunResult {
    unsigned long long segments = 0, hits = 0, node_visits = 0, sphere_tests = 0, paths = 0;
    double render_ms = 0.0, trace_ms = 0.0;
    uint32_t trace_launches = 0, iterations = 0;
};

struct PathWork {              // what a context keeps between launches
    PathSlot plain, batch;
    Event t0, t1;
    uint32_t grid_lds = 0, grid_mem = 0;  // resident k_path workgroups by variant
    ~PathWork() { path_trim(this); }
};

vzStatus path_work(vzContext ctx, PathWork** out);

Cam make_cam(const vzLaunchParams& p);
// Whether a request may go through the traversals that do not count.
bool ordered_paths(const PathItem& item);
// Pixels of a request with its tiles' padding, and its paths.
uint64_t padded_pixels(const vzLaunchParams& p, const PathOptions& opt);
uint64_t path_count(const vzLaunchParams& p, const PathOptions& opt);
// Device memory that a request of several launches carries between them.
uint64_t carry_bytes(const vzLaunchParams& p, uint64_t npad);
// Bytes of a slot for launches of up to `paths` paths.
inline uint64_t slot_bytes(uint64_t paths) { return paths * kPathBytes + 256; }
// Passes of the next slice of `passes` that are left, where a launch takes at
// most `most` paths: of as few equal slices as there can be.
uint64_t slice_passes(uint64_t passes, uint64_t npad, uint64_t most);
// The device memory a served request is admitted by: the paths of one of its
// slices, and what they carry if there are several.
size_t request_bytes(const vzLaunchParams& p, const PathOptions& opt, uint64_t most);
// Makes room in the slot for launches of up to `paths` paths; nothing on its
// stream may still run.
vzStatus slot_reserve(PathSlot& s, uint64_t paths);
// Gives the buffer back (likewise).
void slot_drop(PathSlot& s);
// Makes room for a request's launches, of *passes passes each: as many as fit
// *budget bytes, fewer where the memory is not there (*budget is then what
// they take), with room for at least `least` paths.  Nothing on the slot's
// stream may still run.
vzStatus path_reserve_one(PathSlot& s, const PathItem& item, const PathOptions& opt, uint64_t* budget, uint64_t least,
                          uint32_t* passes);
// Enqueues one request in launches of `passes` passes.  add: its totals add to
// those of the slot's launch before.
vzStatus path_enqueue_one(PathWork* w, PathSlot& s, const PathItem& item, const PathOptions& opt, uint32_t passes,
                          bool add, hipStream_t st, uint32_t* launches);
// Enqueues n slices of different requests as one launch (their paths fit the slot).
vzStatus path_enqueue_many(PathWork* w, PathSlot& s, const PathSlice* slices, uint32_t n, const PathOptions& opt,
                           bool add, hipStream_t st);
// Segments of slice i of the slot's last launch, of n slices, once it is done.
unsigned long long slice_segments(const PathSlot& s, uint32_t n, uint32_t i);

// Renders one frame and waits for it.
vzStatus path_launch(vzContext ctx, const PathItem& item, hipStream_t st, RunResult* res);
// Renders every item and waits for them.
vzStatus path_batch(vzContext ctx, const std::vector<PathItem>& items, const vzTuning& t, hipStream_t st,
                    RunResult* res);
// Memory of a tuning's paths.
uint64_t tuning_budget(const vzTuning& t);

}  // namespace vz
