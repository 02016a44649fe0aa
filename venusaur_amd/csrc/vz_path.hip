// vz_path.hip -- plain launches (vzLaunch) as persistent path tracing.
// Replaces the recursive optixTrace chain of the reference's OptiX programs
// (Core/RayTracer.cu:163-450).
//
// A launch is three kernels per chunk of passes (a pass is sample s of every
// pixel):
//   k_path_seeds    per pixel, the camera seed of every pass of the chunk.
//                   The seed of pass s + 1 follows from the camera draws of
//                   pass s alone (RayTracer.cu:163-204), so with the seeds
//                   known every path of the chunk is independent.
//   k_path          persistent waves.  A lane traces one path from its
//                   camera ray to its end and then takes the next (path
//                   regeneration, Novak, Havran and Dachsbacher 2010), so a
//                   wave stays full until the chunk runs out; its radiance
//                   goes to the path's own slot of a buffer.
//   k_path_resolve  adds the chunk's radiances to the per-pixel sums in
//                   sample order and, after the last chunk, writes accum and
//                   image.  The sums are the sequential ones whatever order
//                   the paths finished in.
//
// Why.  The queue-driven wavefront this replaces for plain launches spent a
// launch per bounce: 304 rounds of three kernels for the 1080p book frame at
// 256 samples, each as long as its slowest workgroup, its path records
// written and read back from HBM between them, and no fewer rounds for a
// small frame.  Tracing whole paths needs one launch, keeps a path in its
// lane's registers and reads nothing but the scene.  Same box, both sides in
// turn: 64x36 at 2 samples 817 -> 143 us, 400x225 at 16 samples 2.80 -> 1.12
// ms, 1200x800 at 16 samples depth 4 3.43 -> 2.04 ms, 1080p at 256 samples
// 115.2 -> 78.6 ms, a million spheres at 1080p and 64 samples 241 -> 187 ms,
// 512x512 at 2048 samples in double 355 -> 135 ms; images bit for bit the
// same.  k_path is bound by VALU issue (traversal and sphere tests with part
// of the lanes idle); k_path_seeds and k_path_resolve are under 1% each of
// the 1080p frame (0.27 and 0.60 ms per 128 passes, the latter reading 3.2 GB
// at 5.3 TB/s).
#include <algorithm>
#include <cstring>
#include <string>
#include <type_traits>
#include <vector>

#include "vz_path.h"
#include "vz_traverse.h"

namespace vz {
namespace {

constexpr int kPathBlk = 512;         // k_path workgroup (8 waves)
constexpr int kWaves = kPathBlk / 64;
constexpr int kStackS = kWideStackS;  // LDS stack slots per lane
constexpr int kBlk = 256;
constexpr uint32_t kLdsNodes = 256;   // a scene of at most this many 4-wide nodes is staged in LDS (16 KB)
constexpr uint32_t kMaxPathBlocks = 8192;
// A wave leaves the traversal to shade and take new paths once fewer than
// this many of its lanes still trace.
constexpr uint32_t kRefillLds = 9;
constexpr uint32_t kRefillGlobal = 41;
constexpr uint32_t kFlushDen = 2;     // queued sphere tests run once 1/kFlushDen of the tracing lanes hold some
constexpr uint32_t kTile = 64;        // pixels of a camera tile: one wave of camera rays
// A unit is what a wave claims at a time: up to kUnitPasses passes of one
// tile, fewer while the units would not go round the waves kUnitRounds times.
constexpr uint32_t kUnitPasses = 8;
constexpr uint32_t kUnitRounds = 8;
// Radiance buffer of a chunk: 16 bytes a path (seed and radiance).  4 GiB
// holds 129 passes of a 1080p frame; every chunk ends with a fraction of a
// millisecond in which the last long paths run alone.
constexpr uint64_t kPathBudget = 4ull << 30;
constexpr int kPathStats = 4;         // segments, hits, node visits, sphere tests

struct PathArgs {
    Cam cam;
    uint32_t subframe, max_depth, spp;
    uint32_t lw;               // tiles are 2^lw x 2^(6 - lw) pixels
    uint32_t tiles_x, npad;    // npad: pixels of all tiles
    uint32_t s0, ns;           // the chunk's passes [s0, s0 + ns)
    uint32_t spu, groups;      // passes per unit, units per tile
    uint32_t units;
    uint32_t refill;
    uint32_t* counter;         // units claimed beyond every wave's first
    uint32_t* seeds;           // ns * npad: camera seed of the pass
    uint32_t* camseed;         // npad: camera seed of the next chunk's first pass
    float* rad;                // 3 * ns * npad: radiance of each path
    unsigned long long* stats; // kPathStats per workgroup
    void* sums;                // 3 * npad float or double, carried between chunks
    void* accum;
    uint32_t* image;
    uint32_t grid;             // k_path workgroups of the chunk
    unsigned long long* totals;  // pinned host memory, kPathStats
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
__device__ __forceinline__ void pixel_of(const PathArgs& P, uint32_t i, uint32_t& x, uint32_t& y)
{
    const uint32_t t = i / kTile, w = i % kTile;
    const uint32_t ty = t / P.tiles_x, tx = t - ty * P.tiles_x;
    x = (tx << P.lw) + (w & ((1u << P.lw) - 1u));
    y = (ty << (6u - P.lw)) + (w >> P.lw);
}

// The camera seed of every pass of the chunk, one thread per pixel: only the
// draws of camera_ray, so the walk is a few LCG steps a pass.
__global__ void __launch_bounds__(kBlk) k_path_seeds(PathArgs P)
{
    const uint32_t i = blockIdx.x * kBlk + threadIdx.x;
    if (i == 0) *P.counter = 0u;
    if (i >= P.npad) return;
    uint32_t x, y;
    pixel_of(P, i, x, y);
    if (x >= P.cam.width || y >= P.cam.height) return;
    uint32_t seed = P.s0 == 0u ? tea4(y * P.cam.width + x, P.subframe) : P.camseed[i];
    for (uint32_t s = 0; s < P.ns; s++) {
        P.seeds[(size_t)s * P.npad + i] = seed;
        skip_camera(seed);
    }
    if (P.s0 + P.ns < P.spp) P.camseed[i] = seed;
}

// Every wave takes units until none is left: the first by its place (so a
// small frame spreads over the CUs), the others from one counter (one
// device-wide atomic per unit of up to 512 paths; per path they would
// serialise across the XCDs).  Lanes without a path take the next ones of the
// wave's unit, all lanes with a ray walk the tree until fewer than `refill`
// of them still do, and the finished ones shade: a path that goes on starts
// its next segment in place.  LDSN: the scene's nodes are staged in LDS.
// COUNT: node visits and sphere tests are counted, and tests run at once so
// that the counts follow each ray alone.
template <bool COUNT, bool LDSN>
__global__ void __launch_bounds__(kPathBlk) __attribute__((amdgpu_waves_per_eu(6))) k_path(SceneView sc, PathArgs P)
{
    constexpr bool DEFER = !COUNT && !LDSN;
    __shared__ uint32_t s_node[kStackS * kPathBlk];
    __shared__ float s_t[kStackS * kPathBlk];
    __shared__ uint4 s_bvh[LDSN ? 4 * kLdsNodes : 1];
    __shared__ uint32_t s_pend[DEFER ? kPend * kPathBlk : 1];
    __shared__ unsigned long long s_red[kPathStats][kWaves];
    const uint32_t tid = threadIdx.x, lane = __lane_id();
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane(tid >> 6);
    if (LDSN) {
        const uint32_t nn = 4u * sc.nw;
        for (uint32_t i = tid; i < nn; i += kPathBlk) s_bvh[i] = ldg(sc.nodes + i);
        __syncthreads();
    }
    Traversal<kStackS, COUNT, DEFER> tr;
    Overflow ov;
    uint32_t nv = 0, ns = 0;
    uint32_t n_seg = 0, n_hit = 0;    // of the wave
    bool active = false, tdone = false, exhausted = false;
    uint32_t unit = wave * gridDim.x + blockIdx.x;
    uint32_t cur = 0, end = 0;        // the wave's unit: its next path and their number
    uint32_t u_tile = 0, u_x = 0, u_y = 0, u_s = 0;
    v3 thr = mk(0.0f, 0.0f, 0.0f);    // the lane's path
    uint32_t seed = 0, slot = 0, depth = 0;
    bool fresh = true;
    for (;;) {
        const uint64_t m = __ballot(!active);
        if (m && !exhausted) {
            if (cur == end) {
                if (!fresh) {
                    uint32_t u = 0;
                    if (lane == 0) u = atomicAdd(P.counter, 1u);
                    unit = kWaves * gridDim.x + (uint32_t)__builtin_amdgcn_readfirstlane(u);
                }
                fresh = false;
                cur = end = 0;
                if (unit >= P.units) {
                    exhausted = true;
                } else {
                    // all passes of a tile follow one another: the waves
                    // work on one part of the image at a time
                    u_tile = unit / P.groups;
                    u_s = (unit - u_tile * P.groups) * P.spu;
                    const uint32_t ty = u_tile / P.tiles_x;
                    u_x = (u_tile - ty * P.tiles_x) << P.lw;
                    u_y = ty << (6u - P.lw);
                    end = min(P.spu, P.ns - u_s) * kTile;
                }
            }
            const uint32_t take = min((uint32_t)__popcll(m), end - cur);
            const uint32_t rk = mbcnt(m);
            if (!active && rk < take) {
                const uint32_t p = cur + rk, w = p % kTile;
                const uint32_t x = u_x + (w & ((1u << P.lw) - 1u)), y = u_y + (w >> P.lw);
                if (x < P.cam.width && y < P.cam.height) {
                    slot = (u_s + p / kTile) * P.npad + u_tile * kTile + w;
                    seed = ldg(P.seeds + slot);
                    v3 o, d;
                    camera_ray(P.cam, x, y, seed, o, d);
                    thr = mk(1.0f, 1.0f, 1.0f);
                    depth = P.max_depth - 1u;
                    tdone = tr.init(sc, o, d, 0.001f, 1e16f, ns);
                    active = true;
                }
            }
            cur += take;
        }
        if (__ballot(active) == 0ull) {
            if (exhausted) break;
            continue;
        }
        uint64_t busy = __ballot(active && !tdone);
        while (busy) {
            if (active && !tdone) {
                if (LDSN)
                    tdone = tr.step(sc, LdsNodes{s_bvh}, s_node + tid, s_t + tid, kPathBlk, ov, nv, ns, s_pend + tid);
                else
                    tdone = tr.step(sc, GlobalNodes{sc.nodes}, s_node + tid, s_t + tid, kPathBlk, ov, nv, ns,
                                    s_pend + tid);
            }
            busy = __ballot(active && !tdone);
            if (DEFER) {
                // flush once enough lanes hold queued tests, relative to the
                // lanes still tracing, or before a queue could overflow (a
                // visit queues at most 4)
                const uint64_t pm = __ballot(tr.npend != 0u);
                if (pm && (__ballot(tr.npend + 4u > kPend) != 0ull ||
                           kFlushDen * (uint32_t)__popcll(pm) >= (uint32_t)__popcll(busy)))
                    tr.flush(sc, s_pend + tid, kPathBlk, ns);
            }
            if ((uint32_t)__popcll(busy) < P.refill) break;
        }
        // every queued test has run before a lane's hit is shaded
        if (DEFER) tr.flush(sc, s_pend + tid, kPathBlk, ns);
        const bool fin = active && tdone;
        const uint64_t fm = __ballot(fin);
        if (fm == 0ull) continue;
        n_seg += (uint32_t)__popcll(fm);
        n_hit += (uint32_t)__popcll(__ballot(fin && tr.bleaf != 0xFFFFFFFFu));
        if (fin) {
            v3 L = mk(0.0f, 0.0f, 0.0f);
            bool ended = true;
            if (tr.bleaf == 0xFFFFFFFFu) {
                // miss (RayTracer.cu:442-450)
                L = mul(thr, sky(tr.d));
            } else if (depth > 0u) {
                // shade (RayTracer.cu:272-440)
                const float4 s = ldg(sc.spheres + tr.bleaf);
                const uint32_t type = ldg(sc.leaf_info + tr.bleaf) >> 30;
                const float4 mat = ldg(sc.mats + tr.bleaf);
                const v3 pos = add(tr.o, scl(tr.d, tr.best));
                v3 n = scl(sub(pos, mk(s.x, s.y, s.z)), recip_rn(s.w));
                const bool front = dot(tr.d, n) < 0.0f;
                if (!front) n = neg(n);
                v3 att, nd;
                if (scatter(type, mat, tr.d, n, front, seed, nd, att)) {
                    thr = mul(thr, att);
                    depth--;
                    ended = false;
                    tdone = tr.init(sc, pos, nd, 0.001f, 1e16f, ns);
                }
            }
            if (ended) {
                float* q = P.rad + 3 * (size_t)slot;
                q[0] = L.x;
                q[1] = L.y;
                q[2] = L.z;
                active = false;
            }
        }
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
        for (int w = 0; w < kWaves; w++) a += s_red[tid][w];
        P.stats[(size_t)blockIdx.x * kPathStats + tid] = a;
    }
}

// Adds the chunk's radiances to the pixels' sums in sample order; on the last
// chunk blends the average into accum and encodes the image (RayTracer.cu:
// 16-47, 203-216).  Its first workgroup also adds the k_path workgroups'
// counters to the totals in host memory, which saves a copy.
template <bool FP64>
__global__ void __launch_bounds__(kBlk) k_path_resolve(PathArgs P)
{
    using T = typename std::conditional<FP64, double, float>::type;
    if (blockIdx.x == 0 && threadIdx.x < 64u * kPathStats) {
        const uint32_t k = threadIdx.x >> 6;
        unsigned long long a = 0;
        for (uint32_t b = threadIdx.x & 63u; b < P.grid; b += 64u) a += P.stats[(size_t)b * kPathStats + k];
        a = wave_sum(a);
        if (__lane_id() == 0) P.totals[k] = (P.s0 ? P.totals[k] : 0ull) + a;
    }
    const uint32_t i = blockIdx.x * kBlk + threadIdx.x;
    if (i >= P.npad) return;
    uint32_t x, y;
    pixel_of(P, i, x, y);
    if (x >= P.cam.width || y >= P.cam.height) return;
    T* sums = (T*)P.sums;
    T s[3] = {T(0), T(0), T(0)};
    if (P.s0)
        for (int k = 0; k < 3; k++) s[k] = sums[(size_t)k * P.npad + i];
    const float* q = P.rad + 3 * (size_t)i;
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

inline uint64_t align256(uint64_t v) { return (v + 255) & ~255ull; }

// Grows a buffer that nothing in flight uses.
bool grow(char** p, size_t* have, size_t need)
{
    if (*have >= need) return true;
    if (*p) (void)hipFree(*p);
    *p = nullptr;
    *have = 0;
    if (hipMalloc((void**)p, need) != hipSuccess) {
        (void)hipGetLastError();
        *p = nullptr;
        return false;
    }
    *have = need;
    return true;
}

uint32_t resident_blocks(const void* kernel, uint32_t cus)
{
    int occ = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, kernel, kPathBlk, 0) != hipSuccess || occ < 1) occ = 1;
    return std::min<uint32_t>(kMaxPathBlocks, cus * (uint32_t)occ);
}

vzStatus path_work(vzContext ctx, PathWork** out)
{
    if (!ctx->path) {
        PathWork* w = new PathWork();
        if (!w->t0.ok() || !w->t1.ok() ||
            hipMalloc((void**)&w->stats, (kMaxPathBlocks * kPathStats + 1) * sizeof(unsigned long long)) != hipSuccess ||
            hipHostMalloc((void**)&w->h_stats, kPathStats * sizeof(unsigned long long)) != hipSuccess) {
            path_free(w);
            return set_error(VZ_ERROR_OUT_OF_MEMORY, "launch workspace allocation failed");
        }
        const uint32_t cus = ctx->num_cus ? ctx->num_cus : 256;
        w->grid_lds = resident_blocks(reinterpret_cast<const void*>(k_path<false, true>), cus);
        w->grid_mem = resident_blocks(reinterpret_cast<const void*>(k_path<false, false>), cus);
        ctx->path = w;
    }
    *out = ctx->path;
    return VZ_SUCCESS;
}

}  // namespace

void path_free(PathWork* w)
{
    if (!w) return;
    if (w->paths) (void)hipFree(w->paths);
    if (w->pixels) (void)hipFree(w->pixels);
    if (w->stats) (void)hipFree(w->stats);
    if (w->h_stats) (void)hipHostFree(w->h_stats);
    delete w;
}

vzStatus path_launch(vzContext ctx, const vzScene_st* scene, const vzLaunchParams& p, hipStream_t st, RunResult* res)
{
    PathWork* w = nullptr;
    VZ_TRY(path_work(ctx, &w));
    PathArgs A;
    std::memset(&A, 0, sizeof(A));
    A.cam = make_cam(p);
    A.subframe = p.subframe_index;
    A.max_depth = p.max_depth;
    A.spp = p.samples_per_pixel;
    // 8x8 tiles; images less than 8 pixels wide or high get tiles of their
    // shape, so that padding never multiplies the pixels by more than 4
    A.lw = p.height < 8u ? 5u : (p.width < 8u ? 1u : 3u);
    const uint32_t tw = 1u << A.lw, th = kTile / tw;
    A.tiles_x = (p.width + tw - 1) / tw;
    const uint64_t ntiles = (uint64_t)A.tiles_x * ((p.height + th - 1) / th);
    if (ntiles * kTile > 0xFFFFFF00ull) return set_error(VZ_ERROR_CAPACITY, "image too large");
    A.npad = (uint32_t)(ntiles * kTile);
    const bool fp64 = (p.flags & VZ_ACCUM_FP64) != 0;
    const bool count = (p.flags & VZ_COUNT_VISITS) != 0, timed = (p.flags & VZ_TIME_STAGES) != 0;

    // the passes in as few equal chunks as the budget allows; less memory
    // than that makes more chunks
    auto split = [&](uint64_t most) { return (uint32_t)((A.spp + (A.spp + most - 1) / most - 1) / ((A.spp + most - 1) / most)); };
    uint32_t chunk = split(std::max<uint64_t>(1, std::min<uint64_t>(A.spp, kPathBudget / (16ull * A.npad))));
    for (;;) {
        const uint64_t per = align256(4ull * A.npad * chunk) + 12ull * A.npad * chunk;
        const uint64_t pix = chunk < A.spp ? align256((fp64 ? 24ull : 12ull) * A.npad) + 4ull * A.npad : 0ull;
        if (grow(&w->paths, &w->paths_bytes, per) && grow(&w->pixels, &w->pixels_bytes, pix)) break;
        if (chunk == 1u)
            return set_error(VZ_ERROR_OUT_OF_MEMORY, "launch buffers (" + std::to_string(per + pix) + " bytes) do not fit");
        chunk = split((chunk + 1) / 2);
    }
    A.seeds = (uint32_t*)w->paths;
    A.rad = (float*)(w->paths + align256(4ull * A.npad * chunk));
    A.sums = w->pixels;
    A.camseed = (uint32_t*)(w->pixels + align256((fp64 ? 24ull : 12ull) * A.npad));
    A.stats = w->stats;
    A.counter = (uint32_t*)(w->stats + kMaxPathBlocks * kPathStats);
    A.accum = p.accum;
    A.image = (uint32_t*)p.image;
    A.totals = w->h_stats;
    const bool lds = scene->n >= 2 && scene->nw <= kLdsNodes;
    const uint32_t resident = lds ? w->grid_lds : w->grid_mem;
    A.refill = lds ? kRefillLds : kRefillGlobal;
    const SceneView sc = scene->view();
    const dim3 pix_grid((A.npad + kBlk - 1) / kBlk);
    std::vector<Event> ev;
    uint32_t launches = 0;
    auto enqueue = [&]() -> vzStatus {
        VZ_HIP_TRY(hipEventRecord(w->t0.e, st));
        for (; A.s0 < A.spp; A.s0 += chunk, launches++) {
            A.ns = std::min(chunk, A.spp - A.s0);
            A.spu = kUnitPasses;
            while (A.spu > 1u && ntiles * ((A.ns + A.spu - 1) / A.spu) < (uint64_t)kUnitRounds * resident * kWaves)
                A.spu >>= 1;
            A.groups = (A.ns + A.spu - 1) / A.spu;
            A.units = (uint32_t)(ntiles * A.groups);
            A.grid = std::min(resident, A.units);
            hipLaunchKernelGGL(k_path_seeds, pix_grid, dim3(kBlk), 0, st, A);
            if (timed) {
                for (int k = 0; k < 2; k++) {
                    ev.emplace_back();
                    VZ_EVENT_TRY(ev.back());
                }
                VZ_HIP_TRY(hipEventRecord(ev[ev.size() - 2].e, st));
            }
            const dim3 grid(A.grid), blk(kPathBlk);
            if (count) {
                if (lds) hipLaunchKernelGGL((k_path<true, true>), grid, blk, 0, st, sc, A);
                else hipLaunchKernelGGL((k_path<true, false>), grid, blk, 0, st, sc, A);
            } else {
                if (lds) hipLaunchKernelGGL((k_path<false, true>), grid, blk, 0, st, sc, A);
                else hipLaunchKernelGGL((k_path<false, false>), grid, blk, 0, st, sc, A);
            }
            if (timed) VZ_HIP_TRY(hipEventRecord(ev.back().e, st));
            if (fp64) hipLaunchKernelGGL(k_path_resolve<true>, pix_grid, dim3(kBlk), 0, st, A);
            else hipLaunchKernelGGL(k_path_resolve<false>, pix_grid, dim3(kBlk), 0, st, A);
            VZ_HIP_TRY(hipGetLastError());
        }
        VZ_HIP_TRY(hipEventRecord(w->t1.e, st));
        return VZ_SUCCESS;
    };
    vzStatus rs = enqueue();
    // the workspace is free for the next launch, on any stream, once this one
    // has finished
    if (hipStreamSynchronize(st) != hipSuccess && rs == VZ_SUCCESS)
        rs = set_error(VZ_ERROR_HIP, "hipStreamSynchronize failed");
    VZ_TRY(rs);
    float ms = 0.0f;
    (void)hipEventElapsedTime(&ms, w->t0.e, w->t1.e);
    *res = RunResult();
    res->segments = w->h_stats[0];
    res->hits = w->h_stats[1];
    res->node_visits = w->h_stats[2];
    res->sphere_tests = w->h_stats[3];
    res->paths = (unsigned long long)p.width * p.height * p.samples_per_pixel;
    res->render_ms = ms;
    for (size_t k = 0; k + 1 < ev.size(); k += 2) {
        float t = 0.0f;
        VZ_HIP_TRY(hipEventElapsedTime(&t, ev[k].e, ev[k + 1].e));
        res->trace_ms += t;
        res->trace_launches++;
    }
    if (!timed) res->trace_launches = launches;
    res->iterations = launches;
    return VZ_SUCCESS;
}

}  // namespace vz
