// vz_trace.hip -- closest-hit queries over a ray array (vzTraceClosest): the
// equivalent of one optixTrace per ray (Core/RayTracer.cu:190-202) without
// shading.  Used for the bit-exact ray-set check and as a traversal
// microbenchmark.
//
// Counters (when stats are asked for).  Each workgroup writes its totals (segments, node visits, sphere
// tests) to its own slot of a partials array; a one-workgroup kernel then
// sums the slots in slot order.  No two workgroups touch one address, so
// there is no device-scope atomic (on MI355X those serialise across the 8
// XCDs) and nothing needs clearing before a call: every slot the reduction
// reads is written by the same call.  vzTraceClosest allocates the array per
// call; vzTraceClosestNoAlloc uses `scratch` below, a fixed array in the
// library's device memory.
#include <algorithm>
#include <type_traits>

#include "vz_traverse_lds.h"
#include "vz_traverse_mem.h"

namespace vz {

// Partials of up to kTraceScratchBlocks workgroups (the no-allocation entry
// point's limit on rays per call: 65536 x 256 = 16,777,216) plus the summed
// counters.  Each GPU the library runs on holds its own copy until the
// process ends; calls on one GPU share it.
static __device__ __align__(256) unsigned long long scratch[kTraceScratchBlocks * kTraceParts + 8];

namespace {

constexpr int kTraceBlk = kTraceBlockSize;

__device__ __forceinline__ uint32_t wave_sum(uint32_t v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
    return v;
}

template <int S, bool COUNT>
__global__ void __launch_bounds__(kTraceBlk) k_trace(SceneView sc, const vzRay* __restrict__ rays,
                                                     uint32_t n, vzHit* __restrict__ hits,
                                                     unsigned long long* __restrict__ parts)
{
    __shared__ uint32_t s_node[S * kTraceBlk];
    __shared__ float s_t[S * kTraceBlk];
    __shared__ unsigned long long s_red[kTraceParts][kTraceBlk / 64];
    uint32_t i = blockIdx.x * kTraceBlk + threadIdx.x;
    uint32_t nv = 0, ns = 0, seg = 0;
    if (i < n) {
        const float4* rp = reinterpret_cast<const float4*>(rays + i);
        float4 a = rp[0], b = rp[1];
        Overflow ov;
        TraceResult r = closest_hit<S, COUNT>(sc, mk(a.x, a.y, a.z), mk(b.x, b.y, b.z), a.w, b.w,
                                              s_node + threadIdx.x, s_t + threadIdx.x, kTraceBlk, ov, nv, ns);
        uint32_t prim = r.leaf == 0xFFFFFFFFu ? VZ_MISS : (sc.leaf_info[r.leaf] & 0x3FFFFFFFu);
        reinterpret_cast<uint2*>(hits)[i] = make_uint2(__float_as_uint(r.t), prim);
        seg = 1;
    }
    seg = wave_sum(seg);
    nv = COUNT ? wave_sum(nv) : 0u;
    ns = COUNT ? wave_sum(ns) : 0u;
    const uint32_t wave = threadIdx.x >> 6;
    if (__lane_id() == 0) {
        s_red[0][wave] = seg;
        s_red[1][wave] = nv;
        s_red[2][wave] = ns;
    }
    __syncthreads();
    if (threadIdx.x < kTraceParts) {
        unsigned long long t = 0;
        for (int w = 0; w < kTraceBlk / 64; w++) t += s_red[threadIdx.x][w];
        parts[(size_t)blockIdx.x * kTraceParts + threadIdx.x] = t;
    }
}

// Sums the nblk partial slots into out[0] (segments), out[2] (node visits)
// and out[3] (sphere tests), the layout of vzTraceClosest's counters.
__global__ void __launch_bounds__(kTraceBlk) k_trace_reduce(const unsigned long long* __restrict__ parts,
                                                            uint32_t nblk, unsigned long long* __restrict__ out)
{
    __shared__ unsigned long long s[kTraceParts][kTraceBlk];
    unsigned long long acc[kTraceParts] = {0, 0, 0};
    for (uint32_t b = threadIdx.x; b < nblk; b += kTraceBlk)
        for (int k = 0; k < kTraceParts; k++) acc[k] += parts[(size_t)b * kTraceParts + k];
    for (int k = 0; k < kTraceParts; k++) s[k][threadIdx.x] = acc[k];
    __syncthreads();
    for (uint32_t half = kTraceBlk / 2; half > 0; half >>= 1) {
        if (threadIdx.x < half)
            for (int k = 0; k < kTraceParts; k++) s[k][threadIdx.x] += s[k][threadIdx.x + half];
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        out[0] = s[0][0];
        out[1] = 0ull;
        out[2] = s[1][0];
        out[3] = s[2][0];
    }
}

// ---- hits alone -------------------------------------------------------------
// Without counters (no stats asked for) the rays go through persistent waves
// as paths do: wave w of W takes the packets of 64 rays w, w + W, ..., a lane
// whose ray has finished writes its hit and takes the wave's next ray once
// fewer than kTraceRefill lanes still trace (any from 16 to 48 is as good),
// sphere tests are queued and run by many lanes at a time, and a small scene
// is walked in LDS.  One thread per ray with tests at once left a wave at the
// pace of its slowest ray, each visit of it behind a node and a sphere load:
// a million rays in the book scene 100 -> 69 us, 32400 in a million spheres
// 355 -> 207 us, 131072 in 200k spheres 457 -> 317 us.  Packets of 64 keep
// neighbouring rays together: 81 us with packets of 16, 73 us with an equal
// share of consecutive rays per wave.
//
// Rays whose closest hit depends on the order of the tests (ordered) are left
// to the end of their wave and walked as before, so that hits with and without
// stats agree for every ray.  Sorting them out costs a million ordinary rays 1
// us of 81.
constexpr uint32_t kTraceLdsBlk = 768;
constexpr uint32_t kTraceMemBlk = kMemThreads;
constexpr uint32_t kTraceRefill = 32;
constexpr uint32_t kFlushNum = 2, kFlushDen = 3;  // as in vz_path.hip

struct TraceNoBound {
    VZ_DEV explicit TraceNoBound(const SceneView&) {}
};

template <bool LDSN>
__global__ void __launch_bounds__(LDSN ? kTraceLdsBlk : kTraceMemBlk) __attribute__((amdgpu_waves_per_eu(LDSN ? 6 : kMemWaves)))
k_trace_hits(SceneView view, const vzRay* __restrict__ rays, uint32_t n, vzHit* __restrict__ hits)
{
    constexpr uint32_t NT = LDSN ? kTraceLdsBlk : kTraceMemBlk;
    __shared__ typename std::conditional<LDSN, LdsScene<NT>, MemScene<NT>>::type sh;
    const uint32_t tid = threadIdx.x, wave = (uint32_t)__builtin_amdgcn_readfirstlane(tid >> 6);
    const typename std::conditional<LDSN, PlaneBound, TraceNoBound>::type pb(view);
    const SceneArrays sc = scene_arrays<false>(view);
    float bound = 0.0f;
    if (LDSN || view.nw != 0u) {
        const v3 m = plane_bounds(view);
        bound = fmaxf(fmaxf(m.x, m.y), m.z);
    }
    if constexpr (LDSN) {
        stage_scene(view, sh);
        __syncthreads();
    }
    typename std::conditional<LDSN, LdsTraversal<NT, true>, MemTraversal<NT, true>>::type tr;
    union {  // one after the other
        typename std::conditional<LDSN, LdsOverflow, MemOverflow>::type ov;
        Overflow odd_ov;
    };
    tr.npend = 0;
    uint32_t mine = 0;
    bool active = false, tdone = false;
    // the wave's next ray, the end of its packet and the packets' stride
    const uint32_t stride = gridDim.x * NT, first = (wave * gridDim.x + blockIdx.x) * 64u;
    uint32_t base = first, cur = 0;
    bool odd = false;
    for (;;) {
        for (uint64_t m; base < n && (m = __ballot(!active)) != 0ull;) {
            const uint32_t left = min(64u, n - base) - cur, take = min((uint32_t)__popcll(m), left);
            const uint32_t rk = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
            if (!active && rk < take) {
                mine = base + cur + rk;
                const float4* rp = reinterpret_cast<const float4*>(rays + mine);
                const float4 a = ldg(rp), b = ldg(rp + 1);
                if (ordered(mk(a.x, a.y, a.z), mk(b.x, b.y, b.z), b.w, bound)) {
                    if constexpr (LDSN) {
                        tr.begin(mk(a.x, a.y, a.z), mk(b.x, b.y, b.z), a.w, b.w);
                        tr.derive(pb);
                        tdone = false;
                    } else {
                        tdone = tr.begin(sc, sh, mk(a.x, a.y, a.z), mk(b.x, b.y, b.z), a.w, b.w);
                        tr.derive();
                    }
                    active = true;
                } else {
                    odd = true;
                }
            }
            cur += take;
            if (take == left) {
                cur = 0;
                base = n - base > stride ? base + stride : n;
            }
        }
        const bool more = base < n;
        if (__ballot(active) == 0ull) break;
        uint64_t busy = __ballot(active && !tdone);
        while (busy) {
            if (active && !tdone) {
                if constexpr (LDSN)
                    tdone = tr.step(sh, ov);
                else
                    tdone = tr.step(sc, sh, ov);
            }
            busy = __ballot(active && !tdone);
            const uint64_t pm = __ballot(tr.npend != 0u);
            if (pm && (__ballot(tr.npend == (LDSN ? kLdsPend : kMemPend)) != 0ull ||
                       kFlushDen * (uint32_t)__popcll(pm) >= kFlushNum * (uint32_t)__popcll(busy))) {
                tr.flush(sc, sh);
            }
            if (more && (uint32_t)__popcll(busy) < kTraceRefill) break;
        }
        tr.flush(sc, sh);
        if (active && tdone) {
            const uint32_t prim = tr.bleaf == 0xFFFFFFFFu ? VZ_MISS : (ldg(sc.info + tr.bleaf) & 0x3FFFFFFFu);
            reinterpret_cast<uint2*>(hits)[mine] = make_uint2(__float_as_uint(tr.best), prim);
            active = false;
        }
    }
    // the wave's rays whose hit depends on the order of the tests, in that
    // order, on its stacks of before
    if (__builtin_expect(__ballot(odd) == 0ull, 1)) return;
    uint32_t* stack;
    if constexpr (LDSN) stack = &sh.stack[wave][0][__lane_id()];
    else stack = &sh.node[wave][0][__lane_id()];
    for (base = first; base < n; base = n - base > stride ? base + stride : n) {
        mine = base + __lane_id();
        if (mine >= n) continue;
        const float4* rp = reinterpret_cast<const float4*>(rays + mine);
        const float4 a = ldg(rp), b = ldg(rp + 1);
        const v3 o = mk(a.x, a.y, a.z), d = mk(b.x, b.y, b.z);
        if (ordered(o, d, b.w, bound)) continue;
        uint32_t nv = 0, ns = 0;
        const TraceResult r =
            closest_hit<4, false>(view, o, d, a.w, b.w, stack, reinterpret_cast<float*>(stack + 4 * 64), 64, odd_ov, nv, ns);
        const uint32_t prim = r.leaf == 0xFFFFFFFFu ? VZ_MISS : (ldg(view.leaf_info + r.leaf) & 0x3FFFFFFFu);
        reinterpret_cast<uint2*>(hits)[mine] = make_uint2(__float_as_uint(r.t), prim);
    }
}

}  // namespace

uint32_t trace_blocks(uint32_t n) { return (n + kTraceBlk - 1) / kTraceBlk; }

vzStatus trace_rays(const SceneView& sc, const vzRay* rays, uint32_t n, vzHit* hits, hipStream_t st,
                    unsigned long long* parts, unsigned long long* counters)
{
    const uint32_t nblk = trace_blocks(n);
    if (nblk) hipLaunchKernelGGL((k_trace<8, true>), dim3(nblk), dim3(kTraceBlk), 0, st, sc, rays, n, hits, parts);
    hipLaunchKernelGGL(k_trace_reduce, dim3(1), dim3(kTraceBlk), 0, st, parts, nblk, counters);
    VZ_HIP_TRY(hipGetLastError());
    return VZ_SUCCESS;
}

vzStatus trace_hits(vzContext ctx, const SceneView& sc, const vzRay* rays, uint32_t n, vzHit* hits, hipStream_t st)
{
    if (n == 0) return VZ_SUCCESS;
    const bool lds = sc.n >= 2 && sc.nw <= kLdsNodes && sc.n <= kLdsSpheres;
    const uint32_t packets = n / 64u + (n % 64u ? 1u : 0u), cus = ctx->num_cus ? ctx->num_cus : 256;
    // as many workgroups as are resident (24 and 28 waves a CU); few rays spread
    // over the CUs, a packet to a workgroup
    if (lds)
        hipLaunchKernelGGL(k_trace_hits<true>, dim3(std::min(packets, 2u * cus)), dim3(kTraceLdsBlk), 0, st, sc, rays, n,
                           hits);
    else
        hipLaunchKernelGGL(k_trace_hits<false>, dim3(std::min(packets, kMemWaves * cus)), dim3(kTraceMemBlk), 0, st, sc, rays, n,
                           hits);
    VZ_HIP_TRY(hipGetLastError());
    return VZ_SUCCESS;
}

// The device address of this GPU's `scratch` (the current device's copy).
// The array's name in host code is only a stand-in for the symbol; kernels
// must be given this address instead.
vzStatus trace_scratch_address(unsigned long long** out)
{
    void* p = nullptr;
    hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
        return set_error(VZ_ERROR_HIP, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
    *out = static_cast<unsigned long long*>(p);
    return VZ_SUCCESS;
}

}  // namespace vz
