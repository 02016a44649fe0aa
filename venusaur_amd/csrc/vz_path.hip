// vz_path.hip -- rendering as persistent path tracing: plain launches
// (vzLaunch), batches (vzBatchLaunch) and the launches of a server.  Replaces
// the recursive optixTrace chain of the reference's OptiX programs
// (Core/RayTracer.cu:163-450).
//
// A launch renders one request, or a table of requests of any scenes and
// sizes, in three kernels (a pass is sample s of every pixel of a request):
//   k_path_seeds    per pixel, the camera seed of every pass.  The seed of
//                   pass s + 1 follows from the camera draws of pass s alone
//                   (RayTracer.cu:163-204), so with the seeds known every
//                   path is independent.
//   k_path          persistent waves.  A lane traces one path from its
//                   camera ray to its end and then takes the next (path
//                   regeneration, Novak, Havran and Dachsbacher 2010), so a
//                   wave stays full until the launch runs out of paths; its
//                   radiance goes to the path's own slot of a buffer.
//   k_path_resolve  adds the radiances to the per-pixel sums in sample order
//                   and writes accum and image.  The sums are the sequential
//                   ones whatever order the paths finished in.
// A request with more paths than the buffer holds takes several launches, a
// chunk of its passes each; its sums and camera seeds carry over.
//
// Why.  The queue-driven wavefront this replaces spent a launch per bounce: 304
// rounds of three kernels for the 1080p book frame at 256 samples, each as
// long as its slowest workgroup, its path records written and read back from
// HBM between them, and no fewer rounds for a small frame.  Tracing whole
// paths needs one launch, keeps a path in its lane's registers and reads
// nothing but the scene.  Same box, both sides in turn, as first built: 1080p
// at 256 samples 115.2 -> 78.6 ms, a million spheres at 1080p and 64 samples
// 241 -> 187 ms, 512x512 at 2048 samples in double 355 -> 135 ms, 400x225 at 16
// samples 2.80 -> 1.12 ms; with the traversals of vz_traverse_lds.h and
// vz_traverse_mem.h, queued sphere tests, shared shading and the counters below
// 53.8 ms, 134 ms, 106 ms and 0.66 ms; images bit for bit the same.  What bounds it is VALU
// issue at half the lanes with the scene in LDS, the L1 and the latency of
// node loads as well with it in memory, and the longest path at the end of a
// small frame.  k_path_seeds and k_path_resolve are under 1% each of the
// 1080p frame (0.27 and 0.60 ms per 128 passes, the latter reading 3.2 GB at
// 5.3 TB/s).
#include <algorithm>
#include <cstring>
#include <string>
#include <type_traits>
#include <vector>

#include "vz_path.h"
#include "vz_traverse_lds.h"
#include "vz_traverse_mem.h"

namespace vz {
namespace {

// k_path workgroups: with the scene in LDS two of 12 waves per CU, so that
// 160 KB hold it twice and not three times; with the nodes in memory seven of 4
// waves (vz_traverse_mem.h).
constexpr int kMemBlk = kMemThreads;
constexpr int kLdsBlk = 768;
constexpr int kStackS = kWideStackS;  // LDS stack slots per lane
constexpr int kBlk = 256;
constexpr uint32_t kMaxPathBlocks = 8192;
// A wave leaves the traversal to shade and take new paths once fewer than
// this many of its lanes still trace.  Nodes in LDS, 1080p book frame: 54.1
// ms at 5, 53.8 at 9, 54.6 at 17 (66.2, 61.3 and 64.6 at 1, 9 and 25 as first
// built).  Nodes in memory: a million spheres 136.4 ms at 33, 134.0 at 41,
// 134.3 at 49, a 24-scene batch 90.5, 90.5 and 90.3 (141, 128 and 115 at 9, 17
// and 41 as first built).
constexpr uint32_t kRefillLds = 9;
constexpr uint32_t kRefillGlobal = 41;
// Queued sphere tests run once two thirds of the tracing lanes hold some:
// 1080p book frame 53.8 ms, 53.9 at a half and 53.6 when all of them do, a
// million spheres 134.0, 135.6 and 133.4 (tested at once as first built 65.8
// against 61.1 for the book frame).
constexpr uint32_t kFlushNum = 2, kFlushDen = 3;
constexpr uint32_t kTile = 64;        // pixels of a camera tile: one wave of camera rays
// A unit is what a wave claims at a time: up to kUnitPasses passes of one
// tile, fewer while the units would not go round the waves kUnitRounds times.
// 1200x800 at 16 samples depth 4: 1377 us at 8 rounds, 1354 at 16, 1398 at 32;
// a million spheres 133.9, 134.0 and 133.9 ms.  With up to 4, 8 and 16 passes a
// million spheres 132.9, 134.0 and 136.5 ms, the 1080p book frame 54.0, 53.8 and
// 54.2.
constexpr uint32_t kUnitPasses = 8;
constexpr uint32_t kUnitRounds = 16;
// Units beyond the first ones are dealt out to up to 2^kLogCounters counters
// (128 bytes apart), each of which serves every so-many-th workgroup alone.  One
// counter for all waves served a unit every 12 ns and no more: 400x225 at 16
// samples 775 us with one and 680 with 8 as first built; 656 with 8, 657 with
// 16 and 652 with 32 now.
constexpr uint32_t kLogCounters = 4;
constexpr uint32_t kCounterStride = 32;
constexpr uint32_t kCounterWords = (kCounterStride << kLogCounters) / 2;  // in 8 bytes

// Where k_path's requests and scenes come from.
enum PathSrc {
    kOneLds,    // one request, its scene's nodes staged in LDS
    kOneMem,    // one request, its scene's nodes in memory
    kManyLds,   // a table of requests of one scene, staged in LDS
    kManyMem    // a table of requests of any scenes
};

constexpr int path_threads(PathSrc src) { return src == kOneLds || src == kManyLds ? kLdsBlk : kMemBlk; }

// One launch of the three kernels: a request of its own (`one`, by value) or
// the requests of a table.
struct PathGroup {
    const PathReq* reqs;       // table (many)
    uint32_t n;                // its requests
    uint32_t units, pixels;    // of all requests
    uint32_t refill;
    uint32_t grid;             // k_path workgroups
    uint32_t add;              // the totals add to those of the launch before
    uint32_t log_counters;
    uint32_t* counters;        // units claimed beyond every wave's first
    uint32_t* seeds;           // per path: camera seed
    float* rad;                // per path: radiance
    unsigned long long* stats; // kPathStats per k_path workgroup
    unsigned long long* segs;  // per request of the table: segments
    unsigned long long* totals;  // pinned host memory: kPathStats, then segs
};

__device__ __forceinline__ uint32_t mbcnt(uint64_t m)
{
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}
__device__ __forceinline__ unsigned long long wave_sum(unsigned long long v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
    return v;
}

// Pixel i of the padded, tile by tile numbering.
__device__ __forceinline__ void pixel_of(const PathReq& P, uint32_t i, uint32_t& x, uint32_t& y)
{
    const uint32_t t = i / kTile, w = i % kTile;
    const uint32_t ty = t / P.tiles_x, tx = t - ty * P.tiles_x;
    x = (tx << P.lw) + (w & ((1u << P.lw) - 1u));
    y = (ty << (6u - P.lw)) + (w >> P.lw);
}

// The last request of the table whose first unit / first pixel is at or
// below v (wave-uniform, so the table is read by scalar loads).
__device__ __forceinline__ uint32_t request_of_unit(const PathReq* __restrict__ reqs, uint32_t n, uint32_t v)
{
    uint32_t lo = 0, hi = n;
    while (hi - lo > 1u) {
        const uint32_t mid = (lo + hi) >> 1;
        if (reqs[mid].unit0 <= v) lo = mid; else hi = mid;
    }
    return lo;
}
__device__ __forceinline__ uint32_t request_of_pixel(const PathReq* __restrict__ reqs, uint32_t n, uint32_t v)
{
    uint32_t lo = 0, hi = n;
    while (hi - lo > 1u) {
        const uint32_t mid = (lo + hi) >> 1;
        if (reqs[mid].pix0 <= v) lo = mid; else hi = mid;
    }
    return lo;
}

// The camera seed of every pass, one thread per pixel: only the draws of
// camera_ray, so the walk is a few LCG steps a pass.
__device__ __forceinline__ void seed_pixel(const PathReq& P, uint32_t i, uint32_t* __restrict__ seeds)
{
    uint32_t x, y;
    pixel_of(P, i, x, y);
    if (x >= P.cam.width || y >= P.cam.height) return;
    uint32_t seed = P.s0 == 0u ? tea4(y * P.cam.width + x, P.subframe) : P.camseed[i];
    for (uint32_t s = 0; s < P.ns; s++) {
        seeds[P.slot0 + (size_t)s * P.npad + i] = seed;
        skip_camera(seed);
    }
    if (P.s0 + P.ns < P.spp) P.camseed[i] = seed;
}
template <bool MANY>
__global__ void __launch_bounds__(kBlk) k_path_seeds(PathGroup G, PathReq one)
{
    const uint32_t j = blockIdx.x * kBlk + threadIdx.x;
    if (j < 1u << G.log_counters) G.counters[j * kCounterStride] = 0u;
    if (MANY)
        for (uint32_t r = j; r < G.n; r += gridDim.x * kBlk) G.segs[r] = 0ull;
    if (j >= G.pixels) return;
    if (MANY) {
        // requests have whole tiles, so a wave's pixels belong to one
        const PathReq& P = G.reqs[request_of_pixel(G.reqs, G.n, (uint32_t)__builtin_amdgcn_readfirstlane(j))];
        seed_pixel(P, j - P.pix0, G.seeds);
    } else {
        seed_pixel(one, j, G.seeds);
    }
}

// LDS of a workgroup whose nodes are in memory, where visits are counted.
struct CountScene {
    uint32_t node[kStackS * kMemBlk];
    float t[kStackS * kMemBlk];
};
struct NoBound {
    __device__ explicit NoBound(const SceneView&) {}
};

// What a lane of a many-scene launch keeps of its scene: the two arrays the
// traversal reads (as SceneArrays).  The others are looked up in the request
// table where a hit is shaded.
template <bool COUNT>
struct LaneScene {
    const uint4* nodes;
    const float4* spheres;
    const PathReq* req;
    __device__ __forceinline__ const uint4* node_array() const { return nodes; }
    __device__ __forceinline__ const float4* sphere_array() const { return spheres; }
    __device__ __forceinline__ const uint32_t* info_array() const { return COUNT ? req->sc.leaf_info : req->sc.tinfo; }
    __device__ __forceinline__ const float4* mat_array() const { return COUNT ? req->sc.mats : req->sc.tmats; }
};

// Every wave takes units until none is left: the first by its place (so a
// small frame spreads over the CUs), the others from its workgroup's counter
// (a device-wide atomic per unit of up to 512 paths).  Lanes without a path
// take the next ones of the wave's unit, all lanes with a ray walk the tree
// until fewer than `refill` of them still do, and the finished ones shade: a
// path that goes on starts its next segment in place.  A wave never waits for its lanes to finish one
// request before it starts the next: with kManyMem each lane carries its own
// scene.
// COUNT: node visits and sphere tests are counted, with the nodes in memory,
// and tests run at once so that the counts follow each ray alone.
template <bool COUNT, PathSrc SRC>
__global__ void __launch_bounds__(path_threads(SRC)) __attribute__((amdgpu_waves_per_eu(SRC == kOneLds || SRC == kManyLds || COUNT ? 6 : kMemWaves))) k_path(PathGroup G, PathReq one)
{
    constexpr bool LDSN = SRC == kOneLds || SRC == kManyLds, MANY = SRC == kManyLds || SRC == kManyMem;
    static_assert(!(COUNT && LDSN), "node visits are counted with the nodes in memory");
    constexpr uint32_t NT = path_threads(SRC), kWaves = NT / 64;
    __shared__ typename std::conditional<LDSN, LdsScene<NT>,
                                         typename std::conditional<COUNT, CountScene, MemScene<NT>>::type>::type sh;
    __shared__ unsigned long long s_red[kPathStats][kWaves];
    const uint32_t tid = threadIdx.x, lane = __lane_id();
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane(tid >> 6);
    // many requests of many scenes: the lane's own, filled in with its path
    typename std::conditional<SRC == kManyMem, LaneScene<COUNT>, SceneArrays>::type sc;
    const SceneView& view = MANY ? G.reqs[0].sc : one.sc;
    if constexpr (SRC == kManyMem) sc = LaneScene<COUNT>{nullptr, nullptr, nullptr};
    else sc = scene_arrays<COUNT>(view);
    typename std::conditional<LDSN, PlaneBound, NoBound>::type pb(view);
    if constexpr (LDSN) {
        stage_scene(view, sh);
        __syncthreads();
    }
    typename std::conditional<LDSN, LdsTraversal<NT>,
                              typename std::conditional<COUNT, Traversal<kStackS, true>, MemTraversal<NT>>::type>::type tr;
    typename std::conditional<LDSN, LdsOverflow,
                              typename std::conditional<COUNT, Overflow, MemOverflow>::type>::type ov;
    if constexpr (!COUNT) tr.npend = 0;
    uint32_t nv = 0, ns = 0;
    uint32_t n_seg = 0, n_hit = 0;    // of the wave
    bool active = false, tdone = false, exhausted = false, fresh = true;
    uint32_t unit = wave * gridDim.x + blockIdx.x;
    uint32_t cur = 0, end = 0;        // the wave's unit: its next path and their number
    uint32_t u_req = 0, u_tile = 0, u_x = 0, u_y = 0, u_s = 0;
    // segments of the unit's request and of the one before it, not yet added
    // to G.segs: an atomic per change of request, since one per segment on a
    // request's counter made a 24-scene batch 1.4 times slower
    uint32_t r_seg = 0, o_req = 0, o_seg = 0;
    v3 thr = mk(0.0f, 0.0f, 0.0f);    // the lane's path
    uint32_t seed = 0, slot = 0, depth = 0, my_req = 0;
    bool start = false;               // its next segment has not been set up
    for (;;) {
        const uint64_t m = __ballot(!active);
        if (m && !exhausted) {
            if (cur == end) {
                if (!fresh) {
                    uint32_t u = 0;
                    const uint32_t h = blockIdx.x & ((1u << G.log_counters) - 1u);
                    if (lane == 0) u = atomicAdd(G.counters + h * kCounterStride, 1u);
                    unit = kWaves * gridDim.x + ((uint32_t)__builtin_amdgcn_readfirstlane(u) << G.log_counters) + h;
                }
                fresh = false;
                cur = end = 0;
                if (unit >= G.units) {
                    exhausted = true;
                } else {
                    if (MANY) {
                        const uint32_t r = request_of_unit(G.reqs, G.n, unit);
                        if (r != u_req) {
                            if (o_seg && lane == 0) atomicAdd(&G.segs[o_req], (unsigned long long)o_seg);
                            o_req = u_req;
                            o_seg = r_seg;
                            r_seg = 0;
                            u_req = r;
                        }
                    }
                    const PathReq& P = MANY ? G.reqs[u_req] : one;
                    // all passes of a tile follow one another: the waves
                    // work on one part of the image at a time
                    const uint32_t u = unit - P.unit0;
                    u_tile = u / P.groups;
                    const uint32_t g = u - u_tile * P.groups;
                    u_s = (g >> P.parts) * P.spu;
                    const uint32_t ty = u_tile / P.tiles_x;
                    u_x = (u_tile - ty * P.tiles_x) << P.lw;
                    u_y = ty << (6u - P.lw);
                    cur = (g & ((1u << P.parts) - 1u)) * (kTile >> P.parts);
                    end = P.parts ? cur + (kTile >> P.parts) : min(P.spu, P.ns - u_s) * kTile;
                }
            }
            const uint32_t take = min((uint32_t)__popcll(m), end - cur);
            const uint32_t rk = mbcnt(m);
            if (!active && rk < take) {
                const PathReq& P = MANY ? G.reqs[u_req] : one;
                const uint32_t p = cur + rk, w = p % kTile;
                const uint32_t x = u_x + (w & ((1u << P.lw) - 1u)), y = u_y + (w >> P.lw);
                if (x < P.cam.width && y < P.cam.height) {
                    slot = P.slot0 + (u_s + p / kTile) * P.npad + u_tile * kTile + w;
                    seed = ldg(G.seeds + slot);
                    camera_ray(P.cam, x, y, seed, tr.o, tr.d);
                    thr = mk(1.0f, 1.0f, 1.0f);
                    depth = P.max_depth - 1u;
                    if (MANY) my_req = u_req;
                    if constexpr (SRC == kManyMem) {
                        const SceneArrays v = scene_arrays<COUNT>(P.sc);
                        sc = LaneScene<COUNT>{v.nodes, v.spheres, G.reqs + u_req};
                    }
                    active = start = true;
                }
            }
            cur += take;
        }
        if (__ballot(active) == 0ull) {
            if (exhausted) break;
            continue;
        }
        if (start) {  // new paths and scattered ones alike
            if constexpr (LDSN) tr.begin(tr.o, tr.d, 0.001f, 1e16f);
            else if constexpr (COUNT) tdone = tr.init(sc, tr.o, tr.d, 0.001f, 1e16f, ns);
            else tdone = tr.begin(sc, sh, tr.o, tr.d, 0.001f, 1e16f);
            if (LDSN) tdone = false;
            start = false;
        }
        // for the lanes still tracing as well: the wave executes this for the
        // new rays anyway, and need not keep the others' through the shading
        if constexpr (LDSN) tr.derive(pb);
        else if constexpr (!COUNT) tr.derive();
        uint64_t busy = __ballot(active && !tdone);
        while (busy) {
            if (active && !tdone) {
                if constexpr (LDSN)
                    tdone = tr.step(sh, ov);
                else if constexpr (COUNT)
                    tdone = tr.step(sc, sh.node + tid, sh.t + tid, NT, ov, nv, ns);
                else
                    tdone = tr.step(sc, sh, ov);
            }
            busy = __ballot(active && !tdone);
            if constexpr (!COUNT) {
                // flush once enough lanes hold queued tests, relative to the
                // lanes still tracing, or before a queue could overflow (a
                // visit queues one entry)
                const uint64_t pm = __ballot(tr.npend != 0u);
                if (pm && (__ballot(tr.npend == (LDSN ? kLdsPend : kMemPend)) != 0ull ||
                           kFlushDen * (uint32_t)__popcll(pm) >= kFlushNum * (uint32_t)__popcll(busy))) {
                    tr.flush(sc, sh);
                }
            }
            // with no paths left to take, the wave finishes its rays first:
            // leaving at every step made the last paths of a launch slower
            // (400x225 at 16 samples 1005 us against 812)
            if (!exhausted && (uint32_t)__popcll(busy) < G.refill) break;
        }
        // every queued test has run before a lane's hit is shaded
        if constexpr (!COUNT) tr.flush(sc, sh);
        const bool fin = active && tdone;
        const uint64_t fm = __ballot(fin);
        if (fm == 0ull) continue;
        n_seg += (uint32_t)__popcll(fm);
        n_hit += (uint32_t)__popcll(__ballot(fin && tr.bleaf != 0xFFFFFFFFu));
        if (MANY) {
            // nearly always the unit's request; after a change of request
            // some lanes still trace the one before
            const uint64_t same = __ballot(fin && my_req == u_req);
            r_seg += (uint32_t)__popcll(same);
            if (fm & ~same) {
                const uint64_t prev = __ballot(fin && my_req != u_req && my_req == o_req);
                o_seg += (uint32_t)__popcll(prev);
                if (fin && my_req != u_req && my_req != o_req) atomicAdd(&G.segs[my_req], 1ull);
            }
        }
        if (fin) {
            v3 L = mk(0.0f, 0.0f, 0.0f);
            bool ended = true;
            // shade (RayTracer.cu:272-440) or miss (RayTracer.cu:442-450); a
            // wave with both normalises once
            const bool miss = tr.bleaf == 0xFFFFFFFFu, shade = !miss && depth > 0u;
            uint32_t type = 0;
            float param = 0.0f;
            bool front = false;
            v3 n = mk(0.0f, 0.0f, 0.0f), p = n, u = tr.d;
            if (shade) {
                float4 s;
                if constexpr (LDSN) s = sh.spheres[tr.bleaf];
                else s = ldg(sc.sphere_array() + tr.bleaf);
                type = ldg(sc.info_array() + tr.bleaf) >> 30;
                const float4 mat = ldg(sc.mat_array() + tr.bleaf);
                tr.o = add(tr.o, scl(tr.d, tr.best));
                n = scl(sub(tr.o, mk(s.x, s.y, s.z)), recip_rn(s.w));
                front = dot(tr.d, n) < 0.0f;
                if (!front) n = neg(n);
                thr = mul(thr, attenuation(type, mat));  // (of no use to a path that ends here)
                param = mat.w;
                p = scatter_point(type, seed);
                if (type == 0u) u = p;
            }
            u = normalize(u);
            if (miss) {
                L = mul(thr, sky(u));
            } else if (shade && scatter(type, param, u, p, n, front, seed, tr.d)) {
                depth--;
                ended = false;
                start = true;
            }
            if (ended) {
                float* q = G.rad + 3 * (size_t)slot;
                q[0] = L.x;
                q[1] = L.y;
                q[2] = L.z;
                active = false;
            }
        }
    }
    if (MANY && lane == 0) {
        if (r_seg) atomicAdd(&G.segs[u_req], (unsigned long long)r_seg);
        if (o_seg) atomicAdd(&G.segs[o_req], (unsigned long long)o_seg);
    }
    const unsigned long long w_nv = COUNT ? wave_sum((unsigned long long)nv) : 0ull;
    const unsigned long long w_ns = COUNT ? wave_sum((unsigned long long)ns) : 0ull;
    if (lane == 0) {
        s_red[0][wave] = n_seg;
        s_red[1][wave] = n_hit;
        s_red[2][wave] = w_nv;
        s_red[3][wave] = w_ns;
    }
    __syncthreads();
    if (tid < (uint32_t)kPathStats) {
        unsigned long long a = 0;
        for (uint32_t w = 0; w < kWaves; w++) a += s_red[tid][w];
        G.stats[(size_t)blockIdx.x * kPathStats + tid] = a;
    }
}

// Adds the radiances of pixel i to its sums in sample order; on the last
// chunk blends the average into accum and encodes the image (RayTracer.cu:
// 16-47, 203-216).
template <bool FP64>
__device__ __forceinline__ void resolve_pixel(const PathReq& P, uint32_t i, const float* __restrict__ rad)
{
    using T = typename std::conditional<FP64, double, float>::type;
    uint32_t x, y;
    pixel_of(P, i, x, y);
    if (x >= P.cam.width || y >= P.cam.height) return;
    T* sums = (T*)P.sums;
    T s[3] = {T(0), T(0), T(0)};
    if (P.s0)
        for (int k = 0; k < 3; k++) s[k] = sums[(size_t)k * P.npad + i];
    const float* q = rad + 3 * ((size_t)P.slot0 + i);
#pragma unroll 8
    for (uint32_t p = 0; p < P.ns; p++, q += 3 * (size_t)P.npad)
        for (int k = 0; k < 3; k++) s[k] = s[k] + (T)q[k];
    if (P.s0 + P.ns != P.spp) {
        for (int k = 0; k < 3; k++) sums[(size_t)k * P.npad + i] = s[k];
        return;
    }
    const size_t px = (size_t)y * P.cam.width + x;
    float oc[3];
    if (FP64) {
        double* acc = (double*)P.accum + 4 * px;
        double avg[3];
        for (int k = 0; k < 3; k++) avg[k] = (double)s[k] / (double)P.spp;
        if (P.subframe > 1u) {
            const double a = 1.0 / (double)P.subframe;
            for (int k = 0; k < 3; k++) avg[k] = acc[k] + a * (avg[k] - acc[k]);
        }
        reinterpret_cast<double2*>(acc)[0] = make_double2(avg[0], avg[1]);
        reinterpret_cast<double2*>(acc)[1] = make_double2(avg[2], 1.0);
        for (int k = 0; k < 3; k++) oc[k] = (float)avg[k];
    } else {
        float4* acc = (float4*)P.accum + px;
        const float inv = 1.0f / (float)P.spp;
        float avg[3] = {(float)s[0] * inv, (float)s[1] * inv, (float)s[2] * inv};
        if (P.subframe > 1u) {
            const float4 prev = *acc;
            const float a = 1.0f / (float)P.subframe;
            avg[0] = prev.x + a * (avg[0] - prev.x);
            avg[1] = prev.y + a * (avg[1] - prev.y);
            avg[2] = prev.z + a * (avg[2] - prev.z);
        }
        *acc = make_float4(avg[0], avg[1], avg[2], 1.0f);
        for (int k = 0; k < 3; k++) oc[k] = avg[k];
    }
    if (P.image) P.image[px] = make_color(oc[0], oc[1], oc[2]);
}

// The first workgroup also adds the k_path workgroups' counters to the
// totals in host memory, which saves a copy.
template <bool MANY>
__global__ void __launch_bounds__(kBlk) k_path_resolve(PathGroup G, PathReq one)
{
    if (blockIdx.x == 0) {
        static_assert(kBlk == 64 * kPathStats, "a wave per counter");
        const uint32_t k = threadIdx.x >> 6;
        unsigned long long a = 0;
        for (uint32_t b = threadIdx.x & 63u; b < G.grid; b += 64u) a += G.stats[(size_t)b * kPathStats + k];
        a = wave_sum(a);
        if (__lane_id() == 0) G.totals[k] = (G.add ? G.totals[k] : 0ull) + a;
        if (MANY)
            for (uint32_t r = threadIdx.x; r < G.n; r += kBlk) G.totals[kPathStats + r] = G.segs[r];
    }
    const uint32_t j = blockIdx.x * kBlk + threadIdx.x;
    if (j >= G.pixels) return;
    if (MANY) {
        const PathReq& P = G.reqs[request_of_pixel(G.reqs, G.n, (uint32_t)__builtin_amdgcn_readfirstlane(j))];
        if (P.fp64) resolve_pixel<true>(P, j - P.pix0, G.rad);
        else resolve_pixel<false>(P, j - P.pix0, G.rad);
    } else {
        if (one.fp64) resolve_pixel<true>(one, j, G.rad);
        else resolve_pixel<false>(one, j, G.rad);
    }
}

inline uint64_t align256(uint64_t v) { return (v + 255) & ~255ull; }

// What a request's launches carry from one to the next: the sums of every
// padded pixel, then the camera seeds.
uint64_t sum_bytes(const vzLaunchParams& p, uint64_t npad)
{
    return align256(((p.flags & VZ_ACCUM_FP64) ? 24ull : 12ull) * npad);
}
// Gives back a buffer that nothing in flight uses.
void drop(char** p, size_t* have)
{
    if (*p) (void)hipFree(*p);
    *p = nullptr;
    *have = 0;
}

// Grows a buffer that nothing in flight uses.
bool grow(vzContext ctx, char** p, size_t* have, size_t need)
{
    if (*have >= need) return true;
    drop(p, have);
    if (!device_alloc(ctx, (void**)p, need)) return false;
    *have = need;
    return true;
}

uint32_t resident_blocks(const void* kernel, int threads, uint32_t cus)
{
    int occ = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, kernel, threads, 0) != hipSuccess || occ < 1) occ = 1;
    return std::min<uint32_t>(kMaxPathBlocks, cus * (uint32_t)occ);
}

bool fits_lds(const vzScene_st* s) { return s->n >= 2 && s->nw <= kLdsNodes && s->n <= kLdsSpheres; }

// Tile shape of a request: the options' where it is 64 pixels of powers of
// two, 8x8 otherwise; images less than 8 pixels high or wide get tiles of
// their shape (2x2 takes a tile of 64 all the same; from a tile's pixels on
// padding less than quadruples them).
uint32_t tile_lw(const vzLaunchParams& p, const PathOptions& opt)
{
    if (p.height < 8u) return 5u;
    if (p.width < 8u) return 1u;
    for (uint32_t lw = 0; lw <= 6u; lw++)
        if (opt.tile_w == (1u << lw) && opt.tile_h == (kTile >> lw)) return lw;
    return 3u;
}

uint64_t tile_count(const vzLaunchParams& p, uint32_t lw)
{
    const uint64_t tw = 1u << lw, th = kTile >> lw;
    return ((p.width + tw - 1) / tw) * ((p.height + th - 1) / th);
}

// The request's fields that do not depend on its place in the launch.
void fill_request(PathReq& A, const PathItem& item, const PathOptions& opt)
{
    const vzLaunchParams& p = item.params;
    std::memset((void*)&A, 0, sizeof(A));
    A.cam = make_cam(p);
    A.subframe = p.subframe_index;
    A.max_depth = p.max_depth;
    A.spp = p.samples_per_pixel;
    A.fp64 = (p.flags & VZ_ACCUM_FP64) ? 1u : 0u;
    A.lw = tile_lw(p, opt);
    A.tiles_x = (p.width + (1u << A.lw) - 1) >> A.lw;
    A.npad = (uint32_t)(tile_count(p, A.lw) * kTile);
    A.accum = p.accum;
    A.image = (uint32_t*)p.image;
    A.sc = item.scene->view();
}

// Passes per unit, so that the units go round the resident waves.
uint32_t unit_passes(uint64_t tile_passes, uint32_t waves)
{
    uint32_t spu = kUnitPasses;
    while (spu > 1u && tile_passes / spu < (uint64_t)kUnitRounds * waves) spu >>= 1;
    return spu;
}

// Every counter has a workgroup.
uint32_t log_counters(uint32_t grid)
{
    uint32_t l = 0;
    while (l < kLogCounters && (2u << l) <= grid) l++;
    return l;
}

// Units to a pass of a tile, as a power of two, as long as every one has a
// resident wave: a wave of fewer paths waits for a less slow ray at every
// segment.  64x36 at 2 samples depth 8: 103 us whole, 86 with up to 1200 waves,
// 85 with 2400, 80 with 4800 (of 6144); 100x60 at 4 samples depth 50 337, 347,
// 309 and 296 us.
uint32_t unit_parts(uint64_t tile_passes, uint32_t waves)
{
    uint32_t l = 0;
    while (l < 6u && (tile_passes << (l + 1u)) <= waves) l++;
    return l;
}

void fill_group(PathGroup& G, PathSlot& s, bool add)
{
    std::memset((void*)&G, 0, sizeof(G));
    G.add = add ? 1u : 0u;
    G.stats = s.stats;
    G.counters = (uint32_t*)(s.stats + kMaxPathBlocks * kPathStats);
    G.segs = s.stats + kMaxPathBlocks * kPathStats + kCounterWords;
    G.totals = s.h_totals;
}

// The three kernels of one launch.
template <bool MANY>
vzStatus launch_group(const PathGroup& G, const PathReq& one, bool lds, const PathOptions& opt, hipStream_t st)
{
    const dim3 pix_grid((G.pixels + kBlk - 1) / kBlk), grid(G.grid), blk(lds ? kLdsBlk : kMemBlk);
    constexpr PathSrc L = MANY ? kManyLds : kOneLds, M = MANY ? kManyMem : kOneMem;
    hipLaunchKernelGGL(k_path_seeds<MANY>, pix_grid, dim3(kBlk), 0, st, G, one);
    if (opt.events) {
        for (int k = 0; k < 2; k++) {
            opt.events->emplace_back();
            VZ_EVENT_TRY(opt.events->back());
        }
        VZ_HIP_TRY(hipEventRecord((*opt.events)[opt.events->size() - 2].e, st));
    }
    if (opt.count) hipLaunchKernelGGL((k_path<true, M>), grid, blk, 0, st, G, one);
    else if (lds) hipLaunchKernelGGL((k_path<false, L>), grid, blk, 0, st, G, one);
    else hipLaunchKernelGGL((k_path<false, M>), grid, blk, 0, st, G, one);
    if (opt.events) VZ_HIP_TRY(hipEventRecord(opt.events->back().e, st));
    hipLaunchKernelGGL(k_path_resolve<MANY>, pix_grid, dim3(kBlk), 0, st, G, one);
    VZ_HIP_TRY(hipGetLastError());
    return VZ_SUCCESS;
}

uint32_t refill_of(const PathOptions& opt, uint32_t dflt)
{
    return opt.refill ? std::min<uint32_t>(opt.refill, 65u) : dflt;
}

}  // namespace

uint64_t carry_bytes(const vzLaunchParams& p, uint64_t npad) { return sum_bytes(p, npad) + 4ull * npad; }

// Whether the closest hits of a request's paths are free of the order of the
// tests (vz_traverse.h, ordered): directions stay below 2^24 and distances
// below 2^28, so the product keeps far below 2^60.  Other requests go through
// the traversal that counts, which keeps the order.
bool ordered_paths(const PathItem& item)
{
    if (item.scene->n < 2) return true;
    const Cam c = make_cam(item.params);
    auto sum = [](v3 v) { return fabsf(v.x) + fabsf(v.y) + fabsf(v.z); };
    const float lens = 4.0f * fabsf(c.lr) * (sum(c.un) + sum(c.vn));  // NaN without a frame
    return item.scene->ordered && 2.0f * (sum(c.U) + sum(c.V) + sum(c.W)) + lens < 0x1p24f &&
           sum(c.O) + lens < kOrderedBound;
}

Cam make_cam(const vzLaunchParams& p)
{
    auto nrm = [](v3 v) {
        float inv = 1.0f / sqrtf(v.x * v.x + v.y * v.y + v.z * v.z);
        v3 r;
        r.x = v.x * inv;
        r.y = v.y * inv;
        r.z = v.z * inv;
        return r;
    };
    Cam c;
    c.O.x = p.origin[0]; c.O.y = p.origin[1]; c.O.z = p.origin[2];
    c.U.x = p.u[0]; c.U.y = p.u[1]; c.U.z = p.u[2];
    c.V.x = p.v[0]; c.V.y = p.v[1]; c.V.z = p.v[2];
    c.W.x = p.w[0]; c.W.y = p.w[1]; c.W.z = p.w[2];
    c.un = nrm(c.U);
    c.vn = nrm(c.V);
    c.lr = p.lens_radius;
    c.width = p.width;
    c.height = p.height;
    return c;
}

uint64_t slice_passes(uint64_t passes, uint64_t npad, uint64_t most)
{
    const uint64_t take = std::max<uint64_t>(most / npad, 1);
    const uint64_t slices = (passes + take - 1) / take;
    return (passes + slices - 1) / slices;
}

size_t request_bytes(const vzLaunchParams& p, const PathOptions& opt, uint64_t most)
{
    const uint64_t npad = padded_pixels(p, opt), passes = slice_passes(p.samples_per_pixel, npad, most);
    return slot_bytes(npad * passes) + (passes < p.samples_per_pixel ? carry_bytes(p, npad) : 0);
}

vzStatus PathSlot::init(vzContext c, bool table)
{
    ctx = c;
    bool ok = stats || device_alloc(ctx, (void**)&stats, (kMaxPathBlocks * kPathStats + kCounterWords + kMaxRequests) *
                                                             sizeof(unsigned long long));
    ok = ok && (h_totals || hipHostMalloc((void**)&h_totals, (kPathStats + kMaxRequests) *
                                                                 sizeof(unsigned long long)) == hipSuccess);
    if (table) {
        ok = ok && (reqs || device_alloc(ctx, (void**)&reqs, kMaxRequests * sizeof(PathReq)));
        ok = ok && (h_reqs || hipHostMalloc((void**)&h_reqs, kMaxRequests * sizeof(PathReq)) == hipSuccess);
    }
    if (!ok) {
        (void)hipGetLastError();
        free();
        return set_error(VZ_ERROR_OUT_OF_MEMORY, "launch table allocation failed");
    }
    return VZ_SUCCESS;
}

void PathSlot::free()
{
    void* dev[] = {paths, pixels, stats, reqs};
    for (void* p : dev)
        if (p) (void)hipFree(p);
    if (h_totals) (void)hipHostFree(h_totals);
    if (h_reqs) (void)hipHostFree(h_reqs);
    *this = PathSlot();
}

vzStatus path_work(vzContext ctx, PathWork** out)
{
    if (!ctx->path) {
        PathWork* w = new PathWork();
        if (!w->t0.ok() || !w->t1.ok()) {
            delete w;
            return set_error(VZ_ERROR_HIP, "hipEventCreate failed");
        }
        const uint32_t cus = ctx->num_cus ? ctx->num_cus : 256;
        w->grid_lds = resident_blocks(reinterpret_cast<const void*>(k_path<false, kOneLds>), kLdsBlk, cus);
        w->grid_mem = resident_blocks(reinterpret_cast<const void*>(k_path<false, kManyMem>), kMemBlk, cus);
        ctx->path = w;
    }
    *out = ctx->path;
    return VZ_SUCCESS;
}

void path_trim(PathWork* w)
{
    if (!w) return;
    w->plain.free();
    w->batch.free();
}

void path_free(PathWork* w) { delete w; }

uint64_t padded_pixels(const vzLaunchParams& p, const PathOptions& opt) { return tile_count(p, tile_lw(p, opt)) * kTile; }

uint64_t path_count(const vzLaunchParams& p, const PathOptions& opt)
{
    return padded_pixels(p, opt) * p.samples_per_pixel;
}

void slot_drop(PathSlot& s) { drop(&s.paths, &s.paths_bytes); }

vzStatus slot_reserve(PathSlot& s, uint64_t paths)
{
    const uint64_t need = slot_bytes(paths);
    if (!grow(s.ctx, &s.paths, &s.paths_bytes, need))
        return set_error(VZ_ERROR_OUT_OF_MEMORY, "launch buffers (" + std::to_string(need) + " bytes) do not fit");
    return VZ_SUCCESS;
}

vzStatus path_reserve_one(PathSlot& s, const PathItem& item, const PathOptions& opt, uint64_t* budget, uint64_t least,
                          uint32_t* passes)
{
    const uint64_t ntiles = tile_count(item.params, tile_lw(item.params, opt));
    if (ntiles * kTile > kMaxLaunchPaths) return set_error(VZ_ERROR_CAPACITY, "image too large");
    const uint64_t npad = ntiles * kTile, spp = item.params.samples_per_pixel;
    // the passes in as few equal chunks as the budget allows; less memory
    // than that makes more chunks
    auto split = [&](uint64_t most) {
        const uint64_t chunks = (spp + most - 1) / most;
        return (spp + chunks - 1) / chunks;
    };
    *budget = std::min(*budget, kMaxSlotBudget);
    uint64_t chunk = split(std::max<uint64_t>(1, std::min<uint64_t>(spp, *budget / (kPathBytes * npad))));
    for (;;) {
        const uint64_t pix = chunk < spp ? carry_bytes(item.params, npad) : 0ull;
        const vzStatus rs = slot_reserve(s, std::max(npad * chunk, least));
        if (rs == VZ_SUCCESS && grow(s.ctx, &s.pixels, &s.pixels_bytes, pix)) break;
        if (chunk == 1u) return rs != VZ_SUCCESS ? rs : set_error(VZ_ERROR_OUT_OF_MEMORY, "launch buffers do not fit");
        chunk = split((chunk + 1) / 2);
        *budget = chunk * npad * kPathBytes;
        // neither buffer is kept larger than the smaller chunk needs: the one
        // that fitted would go on taking the room of the one that did not
        drop(&s.paths, &s.paths_bytes);
        drop(&s.pixels, &s.pixels_bytes);
    }
    *passes = (uint32_t)chunk;
    return VZ_SUCCESS;
}

vzStatus path_enqueue_one(PathWork* w, PathSlot& s, const PathItem& item, const PathOptions& opt, uint32_t passes,
                          bool add, hipStream_t st, uint32_t* launches)
{
    PathReq A;
    fill_request(A, item, opt);
    const uint64_t ntiles = A.npad / kTile;
    if (slot_bytes((uint64_t)A.npad * passes) > s.paths_bytes)
        return set_error(VZ_ERROR_INTERNAL, "launch larger than its slot");
    const bool lds = fits_lds(item.scene) && !opt.count;
    const uint32_t resident = lds ? w->grid_lds : w->grid_mem;
    const uint32_t waves = resident * (lds ? kLdsBlk : kMemBlk) / 64;
    PathGroup G;
    fill_group(G, s, add);
    G.seeds = (uint32_t*)s.paths;
    G.rad = (float*)(s.paths + align256(4ull * A.npad * passes));
    G.pixels = A.npad;
    G.refill = refill_of(opt, lds ? kRefillLds : kRefillGlobal);
    A.sums = s.pixels;
    A.camseed = (uint32_t*)(s.pixels + sum_bytes(item.params, A.npad));
    for (A.s0 = 0; A.s0 < A.spp; A.s0 += passes) {
        A.ns = std::min(passes, A.spp - A.s0);
        A.spu = unit_passes(ntiles * A.ns, waves);
        A.parts = unit_parts(ntiles * A.ns, waves);
        A.groups = ((A.ns + A.spu - 1) / A.spu) << A.parts;
        G.units = (uint32_t)(ntiles * A.groups);
        G.grid = std::min(resident, G.units);
        G.log_counters = log_counters(G.grid);
        VZ_TRY(launch_group<false>(G, A, lds, opt, st));
        G.add = 1u;
        if (launches) ++*launches;
    }
    return VZ_SUCCESS;
}

vzStatus path_enqueue_many(PathWork* w, PathSlot& s, const PathSlice* slices, uint32_t n, const PathOptions& opt,
                           bool add, hipStream_t st)
{
    if (s.used + n > kMaxRequests) return set_error(VZ_ERROR_INTERNAL, "request table overrun");
    PathReq* const h = s.h_reqs + s.used;
    PathReq* const d = s.reqs + s.used;
    bool lds = fits_lds(slices[0].item->scene) && !opt.count;
    uint64_t tile_passes = 0, paths = 0;
    for (uint32_t i = 0; i < n; i++) {
        const PathSlice& sl = slices[i];
        fill_request(h[i], *sl.item, opt);
        h[i].s0 = sl.s0;
        h[i].ns = sl.ns;
        if (sl.carry) {
            h[i].sums = sl.carry;
            h[i].camseed = (uint32_t*)(sl.carry + sum_bytes(sl.item->params, h[i].npad));
        } else if (sl.ns != h[i].spp) {
            return set_error(VZ_ERROR_INTERNAL, "a slice of a request without its sums");
        }
        lds = lds && sl.item->scene == slices[0].item->scene;
        tile_passes += (uint64_t)h[i].npad / kTile * sl.ns;
        paths += (uint64_t)h[i].npad * sl.ns;
    }
    if (slot_bytes(paths) > s.paths_bytes || paths > kMaxLaunchPaths)
        return set_error(VZ_ERROR_INTERNAL, "launch larger than its slot");
    const uint32_t resident = lds ? w->grid_lds : w->grid_mem;
    const uint32_t waves = resident * (lds ? kLdsBlk : kMemBlk) / 64;
    const uint32_t spu = unit_passes(tile_passes, waves), parts = unit_parts(tile_passes, waves);
    PathGroup G;
    fill_group(G, s, add);
    uint32_t slot0 = 0;
    for (uint32_t i = 0; i < n; i++) {
        PathReq& A = h[i];
        A.spu = std::min(spu, A.ns);
        A.parts = parts;
        A.groups = ((A.ns + A.spu - 1) / A.spu) << parts;
        A.unit0 = G.units;
        A.pix0 = G.pixels;
        A.slot0 = slot0;
        G.units += A.npad / kTile * A.groups;
        G.pixels += A.npad;
        slot0 += A.npad * A.ns;
    }
    G.seeds = (uint32_t*)s.paths;
    G.rad = (float*)(s.paths + align256(4ull * paths));
    G.refill = refill_of(opt, lds ? kRefillLds : kRefillGlobal);
    G.grid = std::min(resident, G.units);
    G.log_counters = log_counters(G.grid);
    if (n == 1) return launch_group<false>(G, h[0], lds, opt, st);  // by value: no table
    G.reqs = d;
    G.n = n;
    VZ_HIP_TRY(hipMemcpyAsync(d, h, n * sizeof(PathReq), hipMemcpyHostToDevice, st));
    s.used += n;
    return launch_group<true>(G, PathReq{}, lds, opt, st);
}

unsigned long long slice_segments(const PathSlot& s, uint32_t n, uint32_t i)
{
    return n == 1 ? s.h_totals[0] : s.h_totals[kPathStats + i];
}

// Waits for the launches of a slot, whose buffers are then free for the next
// ones on any stream, and reads their counters and times.
static vzStatus finish(PathWork* w, PathSlot& s, vzStatus rs, bool visits, const std::vector<Event>& ev, hipStream_t st,
                       RunResult* res)
{
    if (hipStreamSynchronize(st) != hipSuccess && rs == VZ_SUCCESS)
        rs = set_error(VZ_ERROR_HIP, "hipStreamSynchronize failed");
    VZ_TRY(rs);
    res->segments = s.h_totals[0];
    res->hits = s.h_totals[1];
    if (visits) {  // (others may have been counted on the way)
        res->node_visits = s.h_totals[2];
        res->sphere_tests = s.h_totals[3];
    }
    float ms = 0.0f;
    VZ_HIP_TRY(hipEventElapsedTime(&ms, w->t0.e, w->t1.e));
    res->render_ms = ms;
    for (size_t k = 0; k + 1 < ev.size(); k += 2) {
        VZ_HIP_TRY(hipEventElapsedTime(&ms, ev[k].e, ev[k + 1].e));
        res->trace_ms += ms;
    }
    res->trace_launches = res->iterations;
    return VZ_SUCCESS;
}

vzStatus path_launch(vzContext ctx, const PathItem& item, hipStream_t st, RunResult* res)
{
    PathWork* w = nullptr;
    VZ_TRY(path_work(ctx, &w));
    VZ_TRY(w->plain.init(ctx, false));
    std::vector<Event> ev;
    PathOptions opt;
    const bool asked = (item.params.flags & VZ_COUNT_VISITS) != 0;
    opt.count = asked || !ordered_paths(item);
    if (item.params.flags & VZ_TIME_STAGES) opt.events = &ev;
    *res = RunResult();
    res->paths = (unsigned long long)item.params.width * item.params.height * item.params.samples_per_pixel;
    uint64_t budget = kPlainBudget;
    uint32_t passes = 0;
    VZ_TRY(path_reserve_one(w->plain, item, opt, &budget, 0, &passes));
    auto enqueue = [&]() -> vzStatus {
        VZ_HIP_TRY(hipEventRecord(w->t0.e, st));
        VZ_TRY(path_enqueue_one(w, w->plain, item, opt, passes, false, st, &res->iterations));
        VZ_HIP_TRY(hipEventRecord(w->t1.e, st));
        return VZ_SUCCESS;
    };
    return finish(w, w->plain, enqueue(), asked, ev, st, res);
}

uint64_t tuning_budget(const vzTuning& t)
{
    return std::min(std::max<uint64_t>((uint64_t)t.queue_capacity * kRayBytes, 256ull << 20), kMaxSlotBudget);
}

// A batch: its items in groups as large as the slot holds, each group one
// launch; an item too large for the slot renders by itself, a chunk of passes
// at a time.  One stream: with the groups side by side on 2, 4 and 8 streams,
// so that a group takes over the CUs another's last paths leave, a 24-scene
// batch took 139-143 ms when one stream took 121 (groups that share the GPU
// also share its caches).
vzStatus path_batch(vzContext ctx, const std::vector<PathItem>& items, const vzTuning& t, hipStream_t st, RunResult* res)
{
    *res = RunResult();
    if (items.empty()) return VZ_SUCCESS;
    PathWork* w = nullptr;
    VZ_TRY(path_work(ctx, &w));
    PathSlot& slot = w->batch;
    std::vector<Event> ev;
    PathOptions opt;
    opt.refill = t.refill_lanes;
    opt.tile_w = t.tile_w;
    opt.tile_h = t.tile_h;
    bool asked = false;
    for (const PathItem& it : items) {
        asked |= (it.params.flags & VZ_COUNT_VISITS) != 0;
        opt.count |= asked || !ordered_paths(it);
        if (it.params.flags & VZ_TIME_STAGES) opt.events = &ev;
        res->paths += (unsigned long long)it.params.width * it.params.height * it.params.samples_per_pixel;
    }
    const uint64_t budget = tuning_budget(t);
    if (slot.paths_bytes > budget + 256) slot.free();  // a smaller tuning gives memory back
    VZ_TRY(slot.init(ctx, true));
    slot.used = 0;
    std::vector<std::vector<PathSlice>> groups(1);
    std::vector<const PathItem*> large;
    uint64_t open = 0, need = 0;
    for (const PathItem& it : items) {
        const uint64_t n = path_count(it.params, opt);
        if (n * kPathBytes > budget) {
            large.push_back(&it);
            continue;
        }
        if ((open + n) * kPathBytes > budget) {
            groups.emplace_back();
            open = 0;
        }
        groups.back().push_back(PathSlice{&it, 0u, it.params.samples_per_pixel, nullptr});
        open += n;
        need = std::max(need, open);
    }
    // the buffers before anything runs; an item that has to make do with less
    // leaves no more to the others
    if (need) VZ_TRY(slot_reserve(slot, need));
    std::vector<uint32_t> passes(large.size());
    for (uint64_t most = budget, before = 0; most != before;) {
        before = most;
        for (size_t i = 0; i < large.size(); i++)
            VZ_TRY(path_reserve_one(slot, *large[i], opt, &most, need, &passes[i]));
    }
    auto enqueue = [&]() -> vzStatus {
        VZ_HIP_TRY(hipEventRecord(w->t0.e, st));
        for (const auto& g : groups) {
            if (g.empty()) continue;
            VZ_TRY(path_enqueue_many(w, slot, g.data(), (uint32_t)g.size(), opt, res->iterations != 0, st));
            res->iterations++;
        }
        for (size_t i = 0; i < large.size(); i++)
            VZ_TRY(path_enqueue_one(w, slot, *large[i], opt, passes[i], res->iterations != 0, st, &res->iterations));
        VZ_HIP_TRY(hipEventRecord(w->t1.e, st));
        return VZ_SUCCESS;
    };
    VZ_TRY(finish(w, slot, enqueue(), asked, ev, st, res));
    return VZ_SUCCESS;
}

}  // namespace vz
