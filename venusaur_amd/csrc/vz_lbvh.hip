// vz_lbvh.hip -- LBVH build on the GPU, replacing optixAccelBuild over
// custom-primitive AABBs (Core/Renderer.h:160-255).
//
// Published methods: Lauterbach et al. 2009 (LBVH from Morton codes),
// Karras 2012 "Maximizing Parallelism in the Construction of BVHs, Octrees,
// and k-d Trees" (parent linking, atomic-flag bottom-up boxes).  The output
// is bit-identical to the CPU build in oracle/: same Morton quantisation,
// stable sort, Karras topology with index tie-breaks, min/max boxes and node
// quantisation.
//
// Stages (all on one stream):
//   1. centre bounds       two-pass min/max reduction
//   2. Morton codes        10 bits per axis of the centre in the bounds
//   3. radix sort          4 passes of 8-bit digits; per-tile histograms,
//                          one scan, stable scatter ranked with wave ballots
//                          (match-any over the digit bits + mbcnt) and staged
//                          through LDS so global writes are runs per digit
//   4. leaf reorder        spheres/materials into Morton (leaf) order
//   5. Karras linking      one thread per internal node
//   6. refit               one thread per leaf walks up; the second arrival at
//                          a node computes its box
//   7. packing, collapse   the 32-byte nodes; the 4-wide tree level by level,
//                          packed as 64-byte nodes and as the 48-byte ones
//                          that most traversals read; a structural check
// A scene of 2 to kSahMaxPrims spheres replaces stages 3 and 5 by a
// binned-SAH build in one workgroup (k_sah_build) that writes the same node
// layout, and goes through stages 1, 2 and 7 in one workgroup each.
#include <cstring>

#include "vz_device.h"
#include "vz_internal.h"

namespace vz {
namespace {

constexpr int kBlk = 256;
constexpr int kItems = 8;
constexpr int kTile = kBlk * kItems;  // keys per radix tile
constexpr uint32_t kLocalBit = 0x80000000u;  // parent link flag (see k_karras)
constexpr uint32_t kLargeKey = 0x40000000u;  // sort-key bit of a large sphere (see k_morton)
constexpr uint32_t kRefitLeaves = 2048;       // leaves per k_refit_local workgroup
constexpr uint32_t kOddWord = 16;             // of the counter block: materials out of the ordinary

__device__ __forceinline__ uint32_t lane_id() { return __lane_id(); }
__device__ __forceinline__ uint32_t mbcnt(uint64_t m)
{
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// ---- 1. bounds ---------------------------------------------------------------
// Centroid bounds, per workgroup.  With `grid_a` set only the spheres at or
// below its size threshold (2|r| <= grid_a[9]) count.
__global__ void __launch_bounds__(kBlk) k_bounds_partial(const float4* __restrict__ sph, uint32_t n,
                                                         const float* __restrict__ grid_a,
                                                         float* __restrict__ partial)
{
    __shared__ float s[6][kBlk];
    float lo[3] = {3.4e38f, 3.4e38f, 3.4e38f}, hi[3] = {-3.4e38f, -3.4e38f, -3.4e38f};
    const float thr = grid_a ? grid_a[9] : 0.0f;
    for (uint32_t i = blockIdx.x * kBlk + threadIdx.x; i < n; i += gridDim.x * kBlk) {
        float4 c = sph[i];
        if (grid_a && 2.0f * fabsf(c.w) > thr) continue;
        lo[0] = fminf(lo[0], c.x); lo[1] = fminf(lo[1], c.y); lo[2] = fminf(lo[2], c.z);
        hi[0] = fmaxf(hi[0], c.x); hi[1] = fmaxf(hi[1], c.y); hi[2] = fmaxf(hi[2], c.z);
    }
    for (int k = 0; k < 3; k++) { s[k][threadIdx.x] = lo[k]; s[3 + k][threadIdx.x] = hi[k]; }
    __syncthreads();
    for (int w = kBlk / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) {
            for (int k = 0; k < 3; k++) {
                s[k][threadIdx.x] = fminf(s[k][threadIdx.x], s[k][threadIdx.x + w]);
                s[3 + k][threadIdx.x] = fmaxf(s[3 + k][threadIdx.x], s[3 + k][threadIdx.x + w]);
            }
        }
        __syncthreads();
    }
    if (threadIdx.x < 6) partial[blockIdx.x * 6 + threadIdx.x] = s[threadIdx.x][0];
}

// A grid: lo[3], hi[3], scale[3] with scale = ext > 0 ? 1024/ext : 0 (iso: one
// scale 1024/max ext for every axis), and the large-sphere threshold
// out[9] = max extent / 4; an axis that no sphere reached gets lo = hi = 0.
// min and max are exact, so the reduction order does not change the result.
__device__ __forceinline__ void write_grid(const float (&lo)[3], const float (&hi)[3], uint32_t iso, float* out)
{
    float extmax = 0.0f;
    for (int k = 0; k < 3; k++) {
        float l = lo[k], h = hi[k];
        if (l > h) l = h = 0.0f;
        const float ext = h - l;
        out[k] = l;
        out[3 + k] = h;
        out[6 + k] = ext > 0.0f ? 1024.0f / ext : 0.0f;
        extmax = fmaxf(extmax, ext);
    }
    if (iso)  // one scale for every axis: cubic Morton cells
        for (int k = 0; k < 3; k++) out[6 + k] = extmax > 0.0f ? 1024.0f / extmax : 0.0f;
    out[9] = 0.25f * extmax;
}
__global__ void __launch_bounds__(kBlk) k_bounds_final(const float* __restrict__ partial, uint32_t nb,
                                                       uint32_t iso, float* __restrict__ out)
{
    __shared__ float s[6][kBlk];
    float lo[3] = {3.4e38f, 3.4e38f, 3.4e38f}, hi[3] = {-3.4e38f, -3.4e38f, -3.4e38f};
    for (uint32_t b = threadIdx.x; b < nb; b += kBlk)
        for (int k = 0; k < 3; k++) {
            lo[k] = fminf(lo[k], partial[b * 6 + k]);
            hi[k] = fmaxf(hi[k], partial[b * 6 + 3 + k]);
        }
    for (int k = 0; k < 3; k++) { s[k][threadIdx.x] = lo[k]; s[3 + k][threadIdx.x] = hi[k]; }
    __syncthreads();
    for (int w = kBlk / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w)
            for (int k = 0; k < 3; k++) {
                s[k][threadIdx.x] = fminf(s[k][threadIdx.x], s[k][threadIdx.x + w]);
                s[3 + k][threadIdx.x] = fmaxf(s[3 + k][threadIdx.x], s[3 + k][threadIdx.x + w]);
            }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        for (int k = 0; k < 3; k++) { lo[k] = s[k][0]; hi[k] = s[3 + k][0]; }
        write_grid(lo, hi, iso, out);
    }
}

// ---- 2. Morton ---------------------------------------------------------------
__device__ __forceinline__ uint32_t expand10(uint32_t v)
{
    v = (v * 0x00010001u) & 0xFF0000FFu;
    v = (v * 0x00000101u) & 0x0F00F00Fu;
    v = (v * 0x00000011u) & 0xC30C30C3u;
    v = (v * 0x00000005u) & 0x49249249u;
    return v;
}

// Sort key of sphere i.  A sphere whose diameter exceeds grid_a's threshold
// (a quarter of the largest centroid extent, e.g. the r = 1000 ground) is
// "large": its key is its Morton code on grid A (all centroids) with bit 30
// set, so the first split of the tree separates it from the rest and its box
// does not inflate a whole root-to-leaf path.  Every other sphere gets its
// Morton code on grid B: the centroids of the small spheres only, with cubic
// cells, so a thin slab of spheres is not split along its thin axis as often
// as along the others.
__device__ __forceinline__ uint32_t morton_key(const float4 c, const float* grid_a, const float* grid_b)
{
    const bool large = 2.0f * fabsf(c.w) > grid_a[9];
    const float* bnd = large ? grid_a : grid_b;
    float cc[3] = {c.x, c.y, c.z};
    uint32_t q[3];
    for (int k = 0; k < 3; k++) {
        float f = (cc[k] - bnd[k]) * bnd[6 + k];
        int qi = (int)f;
        qi = qi < 0 ? 0 : (qi > 1023 ? 1023 : qi);
        q[k] = (uint32_t)qi;
    }
    return (expand10(q[0]) << 2) | (expand10(q[1]) << 1) | expand10(q[2]) | (large ? kLargeKey : 0u);
}
__global__ void __launch_bounds__(kBlk) k_morton(const float4* __restrict__ sph, uint32_t n,
                                                 const float* __restrict__ grid_a,
                                                 const float* __restrict__ grid_b,
                                                 uint32_t* __restrict__ keys, uint32_t* __restrict__ vals,
                                                 uint32_t* __restrict__ odd)
{
    uint32_t i = blockIdx.x * kBlk + threadIdx.x;
    if (i >= n) return;
    if (i == 0u) *odd = 0u;
    keys[i] = morton_key(sph[i], grid_a, grid_b);
    vals[i] = i;
}

// ---- 3. radix sort -------------------------------------------------------------
// Exclusive scan of one value per thread over a kBlk-thread workgroup.
__device__ __forceinline__ uint32_t block_scan_excl(uint32_t v, uint32_t* s)
{
    s[threadIdx.x] = v;
    __syncthreads();
    for (uint32_t off = 1; off < (uint32_t)kBlk; off <<= 1) {
        const uint32_t t = threadIdx.x >= off ? s[threadIdx.x - off] : 0u;
        __syncthreads();
        s[threadIdx.x] += t;
        __syncthreads();
    }
    const uint32_t r = s[threadIdx.x] - v;
    __syncthreads();
    return r;
}

__global__ void __launch_bounds__(kBlk) k_radix_hist(const uint32_t* __restrict__ keys, uint32_t n,
                                                     int shift, uint32_t nblocks,
                                                     uint32_t* __restrict__ hist)
{
    __shared__ uint32_t h[256];
    h[threadIdx.x] = 0;
    __syncthreads();
    uint32_t base = blockIdx.x * kTile;
    for (int r = 0; r < kItems; r++) {
        uint32_t i = base + r * kBlk + threadIdx.x;
        if (i < n) atomicAdd(&h[(keys[i] >> shift) & 0xFFu], 1u);
    }
    __syncthreads();
    hist[threadIdx.x * nblocks + blockIdx.x] = h[threadIdx.x];
}

// Per digit (one workgroup each): exclusive scan in place of the digit's
// per-tile counts, row total to dtot[digit].  The scatter adds the digit's
// base, the exclusive scan of dtot.
__global__ void __launch_bounds__(kBlk) k_scan_rows(uint32_t* __restrict__ hist, uint32_t nblocks,
                                                    uint32_t* __restrict__ dtot)
{
    __shared__ uint32_t part[kBlk];
    uint32_t* row = hist + (size_t)blockIdx.x * nblocks;
    const uint32_t chunk = (nblocks + kBlk - 1) / kBlk;
    const uint32_t b = threadIdx.x * chunk, e = min(b + chunk, nblocks);
    uint32_t sum = 0;
    for (uint32_t i = b; i < e; i++) sum += row[i];
    const uint32_t excl = block_scan_excl(sum, part);
    uint32_t run = excl;
    for (uint32_t i = b; i < e; i++) {
        const uint32_t v = row[i];
        row[i] = run;
        run += v;
    }
    if (threadIdx.x == kBlk - 1) dtot[blockIdx.x] = excl + sum;
}

__global__ void __launch_bounds__(kBlk) k_radix_scatter(const uint32_t* __restrict__ kin,
                                                        const uint32_t* __restrict__ vin, uint32_t n,
                                                        int shift, uint32_t nblocks,
                                                        const uint32_t* __restrict__ hist,
                                                        const uint32_t* __restrict__ dtot,
                                                        uint32_t* __restrict__ kout,
                                                        uint32_t* __restrict__ vout)
{
    __shared__ uint32_t s_dbase[256];   // first output slot of each digit
    __shared__ uint32_t s_count[256];   // running per-digit count in this tile
    __shared__ uint32_t s_start[256];   // tile-local start of each digit
    __shared__ uint32_t s_wcnt[4][256];
    __shared__ uint32_t s_wpre[4][256];
    __shared__ uint32_t s_key[kTile];
    __shared__ uint32_t s_val[kTile];
    const uint32_t tid = threadIdx.x, wave = tid >> 6, lane = lane_id();
    s_dbase[tid] = block_scan_excl(dtot[tid], s_count);  // s_count as scratch
    s_count[tid] = 0;
    for (int w = 0; w < 4; w++) s_wcnt[w][tid] = 0;
    __syncthreads();
    const uint32_t base = blockIdx.x * kTile;
    uint32_t key[kItems], val[kItems], rank[kItems];
    for (int r = 0; r < kItems; r++) {
        uint32_t i = base + r * kBlk + tid;
        bool valid = i < n;
        key[r] = valid ? kin[i] : 0u;
        val[r] = valid ? vin[i] : 0u;
        uint32_t d = (key[r] >> shift) & 0xFFu;
        // lanes of this wave holding the same digit (match-any over 8 bits)
        uint64_t peers = __ballot(valid);
#pragma unroll
        for (int bit = 0; bit < 8; bit++) {
            uint64_t m = __ballot((d >> bit) & 1u);
            peers &= ((d >> bit) & 1u) ? m : ~m;
        }
        uint32_t rk = mbcnt(peers);
        if (valid && (uint32_t)(__ffsll((unsigned long long)peers) - 1) == lane)
            s_wcnt[wave][d] = (uint32_t)__popcll(peers);
        __syncthreads();
        {   // thread t owns digit t: prefix over the 4 waves, in wave order
            uint32_t run = s_count[tid];
            for (int w = 0; w < 4; w++) {
                uint32_t c = s_wcnt[w][tid];
                s_wpre[w][tid] = run;
                run += c;
                s_wcnt[w][tid] = 0;
            }
            s_count[tid] = run;
        }
        __syncthreads();
        rank[r] = valid ? s_wpre[wave][d] + rk : 0xFFFFFFFFu;
        __syncthreads();
    }
    // exclusive scan of the tile's digit counts (256 entries, one per thread)
    {
        uint32_t v = s_count[tid];
        s_start[tid] = v;
        __syncthreads();
        for (uint32_t off = 1; off < 256; off <<= 1) {
            uint32_t t = tid >= off ? s_start[tid - off] : 0u;
            __syncthreads();
            s_start[tid] += t;
            __syncthreads();
        }
        s_start[tid] -= v;
        __syncthreads();
    }
    for (int r = 0; r < kItems; r++) {
        if (rank[r] != 0xFFFFFFFFu) {
            uint32_t d = (key[r] >> shift) & 0xFFu;
            uint32_t pos = s_start[d] + rank[r];
            s_key[pos] = key[r];
            s_val[pos] = val[r];
        }
    }
    __syncthreads();
    uint32_t cnt = n - base < (uint32_t)kTile ? n - base : (uint32_t)kTile;
    for (uint32_t i = tid; i < cnt; i += kBlk) {
        uint32_t k = s_key[i];
        uint32_t d = (k >> shift) & 0xFFu;
        uint32_t g = s_dbase[d] + hist[d * nblocks + blockIdx.x] + (i - s_start[d]);
        kout[g] = k;
        vout[g] = s_val[i];
    }
}

// ---- 4. leaf reorder -----------------------------------------------------------
// *odd: some material may send rays on in directions far longer than the
// normal, or of no length (see vzScene_st::ordered).
__global__ void __launch_bounds__(kBlk) k_reorder(const float4* __restrict__ sph_in,
                                                  const vzMaterial* __restrict__ mat_in,
                                                  const uint32_t* __restrict__ perm, uint32_t n,
                                                  float4* __restrict__ sph, uint32_t* __restrict__ info,
                                                  float4* __restrict__ mat, uint32_t* __restrict__ odd)
{
    uint32_t i = blockIdx.x * kBlk + threadIdx.x;
    if (i >= n) return;
    uint32_t p = perm[i];
    sph[i] = sph_in[p];
    vzMaterial m = mat_in[p];
    uint32_t type = m.type > 2u ? 0u : m.type;
    info[i] = p | (type << 30);
    float param = type == 1u ? m.fuzz : (type == 2u ? m.ir : 0.0f);
    mat[i] = make_float4(m.albedo[0], m.albedo[1], m.albedo[2], param);
    if (!(fabsf(param) < 0x1p20f) || (type == 2u && !(fabsf(param) > 0x1p-20f))) *odd = 1u;
}

// refit reads spheres in leaf order but geometry updates arrive in prim order
__global__ void __launch_bounds__(kBlk) k_reorder_sph(const float4* __restrict__ sph_in,
                                                      const uint32_t* __restrict__ perm, uint32_t n,
                                                      float4* __restrict__ sph)
{
    uint32_t i = blockIdx.x * kBlk + threadIdx.x;
    if (i < n) sph[i] = sph_in[perm[i]];
}

// ---- 5. Karras linking -----------------------------------------------------------
__device__ __forceinline__ int kdelta(const uint32_t* __restrict__ k, int n, int i, int j)
{
    if (j < 0 || j >= n) return -1;
    uint32_t a = k[i], b = k[j];
    if (a == b) return 32 + __clz((int)((uint32_t)i ^ (uint32_t)j));
    return __clz((int)(a ^ b));
}

__global__ void __launch_bounds__(kBlk) k_karras(const uint32_t* __restrict__ K, uint32_t n_,
                                                 uint32_t* __restrict__ child,
                                                 uint32_t* __restrict__ parent_int,
                                                 uint32_t* __restrict__ parent_leaf,
                                                 uint32_t* __restrict__ visit, uint2* __restrict__ range)
{
    int n = (int)n_;
    int i = (int)(blockIdx.x * kBlk + threadIdx.x);
    if (i >= n - 1) return;
    visit[i] = 0u;
    if (i == 0) parent_int[0] = 0xFFFFFFFFu;
    int d = (kdelta(K, n, i, i + 1) - kdelta(K, n, i, i - 1)) > 0 ? 1 : -1;
    int dmin = kdelta(K, n, i, i - d);
    int lmax = 2;
    while (kdelta(K, n, i, i + lmax * d) > dmin) lmax *= 2;
    int l = 0;
    for (int t = lmax / 2; t >= 1; t /= 2)
        if (kdelta(K, n, i, i + (l + t) * d) > dmin) l += t;
    int j = i + l * d;
    int dnode = kdelta(K, n, i, j);
    int s = 0, div = 2;
    int t = (l + div - 1) / div;
    for (;;) {
        if (kdelta(K, n, i, i + (s + t) * d) > dnode) s += t;
        if (t == 1) break;
        div *= 2;
        t = (l + div - 1) / div;
    }
    int g = i + s * d + (d < 0 ? d : 0);
    int mn = min(i, j), mx = max(i, j);
    uint32_t f = 0;
    // bit 31 of a parent link: every leaf of the parent's range lies in one
    // refit workgroup, so the refit synchronises on it at workgroup scope
    const uint32_t up = (uint32_t)i | ((mn / (int)kRefitLeaves == mx / (int)kRefitLeaves) ? kLocalBit : 0u);
    if (mn == g) { f |= 1u; parent_leaf[g] = up; } else { parent_int[g] = up; }
    if (mx == g + 1) { f |= 2u; parent_leaf[g + 1] = up; } else { parent_int[g + 1] = up; }
    child[i] = (uint32_t)g | (f << 30);
    range[i] = make_uint2((uint32_t)mn, (uint32_t)mx);
}

// ---- 5'. binned-SAH build of a small scene -------------------------------------------
// For 2 .. kSahMaxPrims spheres the Morton order serves large spheres badly
// (the book scene's ground and its three big spheres), so the binary tree is
// built top down by the surface-area heuristic instead.  A range [a, b] of
// the leaf permutation at depth < kSahDepthCap: per axis whose centre extent
// ext is positive, sphere centre c falls in bin min(31, (int)(((c - lo) /
// ext) * 32)); the split after bin j costs area(L) * nL + area(R) * nR over
// the leaf-box unions and counts of bins <= j and > j (both non-empty); the
// cheapest wins, lower axis then lower bin on a tie, and the range is
// partitioned stably.  With no positive extent, or below the depth cap, the
// range splits after its first floor(m / 2) spheres.  The cap bounds the
// tree at kSahDepthCap + 10 internal levels for 1024 spheres, so the 4-wide
// tree stays within the traversal's kMaxWideDepth.
// Nodes use the Karras layout (children g and g + 1 for a split after leaf
// position g, the root is node 0), so refit, collapse and traversal are the
// LBVH's.  One workgroup; a wave splits a range by itself.  Bin boxes are
// kept as order-preserving integer keys and merged with LDS integer min/max,
// counts with adds, so the bins do not depend on the order lanes ran in; the
// sweep's unions are exact in any order and the partition is stable.  The
// result equals the oracle's sah_range bit for bit.
//
// What a split costs is the latency of its cross-lane steps, some 500 of
// them when every step of every scan was a shuffle through the LDS crossbar,
// and the barriers of a workgroup that took one range per wave and round:
// 409 us for the book scene's 486 spheres, 3.15 ms for the 1536 treelets of a
// million.  Scans and reductions now run in DPP (four-cycle VALU moves
// inside and between rows of 16 lanes), the prefix and the suffix of an axis
// side by side in the two halves of the wave, and waves take ranges from a
// queue without barriers: 173 us and 1.21 ms.
constexpr uint32_t kSahMaxPrims = 1024;
constexpr int kSahBins = 32;
constexpr uint32_t kSahDepthCap = 24;
// An LBVH of at least kTreeletMinPrims spheres has its treelets rebuilt by
// the same SAH build: every maximal subtree of at most kSahMaxPrims leaves
// whose root lies above kSahDepthCap, one workgroup each, splits counting
// depth from the whole tree's root.  On box scenes of a few thousand
// spheres SAH treelets visited more nodes than Morton order; from about 2e5
// spheres up they visit 4-6% fewer.
constexpr uint32_t kTreeletMinPrims = 131072;
constexpr uint32_t kTreeletBlocks = 2048;  // grid of k_sah_treelets (grid-stride over the treelets)
constexpr int kSahWaves = 8;       // of a treelet's workgroup
constexpr int kSahSoloWaves = 16;  // of the one workgroup that builds a small scene
constexpr int kSahBinWords = 3 * kSahBins * 7;  // per wave: [axis][bin] lo xyz, hi xyz keys, count
static_assert(kSahMaxPrims <= kRefitLeaves, "every SAH range lies in one refit workgroup");
static_assert(kSahWaves * kSahBinWords >= (int)kSahMaxPrims, "the bins hold a treelet's keys at the end");
// A wave goes on with the larger part of a split; the smaller one goes to the
// queue from kSahShare spheres up (at most kSahMaxPrims / kSahShare of them),
// and is finished first otherwise.  Ranges of up to kSahFew spheres are built
// to the end by sah_few.
constexpr uint32_t kSahFew = 21;  // times 3 axes in a wave
constexpr uint32_t kSahShare = 8;
constexpr uint32_t kSahTasks = 192;
static_assert(kSahMaxPrims / kSahShare + 1 + kSahSoloWaves <= kSahTasks, "a ticket per task and waiting wave");
static_assert(kSahShare <= kSahFew, "what a wave finishes first is built by sah_few");
constexpr uint32_t kSahNone = 0xFFFFFFFFu;
static_assert(kSahDepthCap + 10 + 1 <= kMaxWideDepth, "SAH tree depth within the traversal stack");

__device__ __forceinline__ uint32_t ord_key(float f)
{
    const uint32_t u = __float_as_uint(f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float ord_val(uint32_t k)
{
    return __uint_as_float((k & 0x80000000u) ? (k & 0x7FFFFFFFu) : ~k);
}
__device__ __forceinline__ float sah_cen(const float4 s, int k) { return k == 0 ? s.x : (k == 1 ? s.y : s.z); }
__device__ __forceinline__ int sah_bin(float c, float lo, float ext)
{
    const int j = (int)(((c - lo) / ext) * (float)kSahBins);
    return j > kSahBins - 1 ? kSahBins - 1 : j;
}
__device__ __forceinline__ float box_area6(const float* b)
{
    const float dx = b[3] - b[0], dy = b[4] - b[1], dz = b[5] - b[2];
    return dx * dy + dy * dz + dz * dx;
}
// v of another lane by DPP; lanes without a source keep their own.
template <int CTRL, int ROWS = 0xF>
__device__ __forceinline__ float dpp_f(float v)
{
    const int x = __float_as_int(v);
    return __int_as_float(__builtin_amdgcn_update_dpp(x, x, CTRL, ROWS, 0xF, false));
}
template <int CTRL, int ROWS = 0xF>
__device__ __forceinline__ uint32_t dpp_add(uint32_t v)  // v + v of another lane, + 0 where there is none
{
    return v + (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xF, false);
}
constexpr int kRowShr = 0x110, kRowBcast15 = 0x142, kRowBcast31 = 0x143;
// Inclusive prefix in each half of the wave (lanes 0-31, 32-63).
template <bool MIN>
__device__ __forceinline__ float half_scan(float v)
{
    auto op = [](float a, float b) { return MIN ? fminf(a, b) : fmaxf(a, b); };
    v = op(v, dpp_f<kRowShr + 1>(v));
    v = op(v, dpp_f<kRowShr + 2>(v));
    v = op(v, dpp_f<kRowShr + 4>(v));
    v = op(v, dpp_f<kRowShr + 8>(v));
    return op(v, dpp_f<kRowBcast15, 0xA>(v));
}
__device__ __forceinline__ uint32_t half_scan_add(uint32_t v)
{
    v = dpp_add<kRowShr + 1>(v);
    v = dpp_add<kRowShr + 2>(v);
    v = dpp_add<kRowShr + 4>(v);
    v = dpp_add<kRowShr + 8>(v);
    return dpp_add<kRowBcast15, 0xA>(v);
}
// Over the whole wave, the same value in every lane.
template <bool MIN>
__device__ __forceinline__ float wave_reduce(float v)
{
    v = half_scan<MIN>(v);
    const float o = dpp_f<kRowBcast31, 0xC>(v);
    v = MIN ? fminf(v, o) : fmaxf(v, o);
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}
// Orders LDS accesses of the wave's lanes (which the hardware runs in order)
// for the compiler, and brings its lanes together after a branch that only
// some took.
__device__ __forceinline__ void wave_order()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Stages 1 and 2 of a small scene, one workgroup, a thread per sphere: five
// launches in one.
constexpr uint32_t kSmallThreads = 1024;
static_assert(kSahMaxPrims <= kSmallThreads, "a thread per sphere");
__global__ void __launch_bounds__(kSmallThreads) k_small_keys(const float4* __restrict__ sph, uint32_t n,
                                                              uint32_t* __restrict__ keys, uint32_t* __restrict__ vals,
                                                              uint32_t* __restrict__ odd)
{
    __shared__ float part[6][kSmallThreads / 64];
    __shared__ float grid[2][10];
    const uint32_t t = threadIdx.x, w = t / 64;
    if (t == 0u) *odd = 0u;
    const float4 c = t < n ? sph[t] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    for (uint32_t g = 0; g < 2u; g++) {  // grid A: every centroid; grid B: those of the small spheres
        const bool in = t < n && (g == 0u || !(2.0f * fabsf(c.w) > grid[0][9]));
        const float cc[3] = {c.x, c.y, c.z};
        for (int k = 0; k < 3; k++) {
            const float lo = wave_reduce<true>(in ? cc[k] : 3.4e38f), hi = wave_reduce<false>(in ? cc[k] : -3.4e38f);
            if (t % 64 == 0u) {
                part[k][w] = lo;
                part[3 + k][w] = hi;
            }
        }
        __syncthreads();
        if (t == 0u) {
            float lo[3], hi[3];
            for (int k = 0; k < 3; k++) {
                lo[k] = part[k][0];
                hi[k] = part[3 + k][0];
                for (uint32_t i = 1; i < kSmallThreads / 64; i++) {
                    lo[k] = fminf(lo[k], part[k][i]);
                    hi[k] = fmaxf(hi[k], part[3 + k][i]);
                }
            }
            write_grid(lo, hi, g, grid[g]);
        }
        __syncthreads();
    }
    if (t < n) {
        keys[t] = morton_key(c, grid[0], grid[1]);
        vals[t] = t;
    }
}

// LDS of one treelet build by NW waves: the range's spheres by local index
// (gathered once), the local permutation, the queue of ranges, and the bins of
// each wave.  A range is (a | b << 10 | depth << 20
// local, node index).
template <int NW>
struct SahShared {
    float4 sph[kSahMaxPrims];
    uint32_t perm[kSahMaxPrims], tmp[kSahMaxPrims];
    uint2 task[kSahTasks];            // .x kSahNone: not written yet
    uint32_t head, tail, open;        // tickets taken, tasks written, tasks not finished
    uint32_t bin[NW][kSahBinWords];
};

// The whole subtree over the range [a, a + m), 2 <= m <= kSahFew, node `self`
// at depth d, by one wave: lane (k, i) holds the sphere at place i and weighs
// axis k, for all ranges of a level at a time.  A split of the binned sweep
// that differs from the one before it comes after some sphere's bin; the lane
// of that sphere sums both sides over its range's spheres in turn, and the
// least cost is taken, of equal ones the first axis and the lowest bin: the
// sweep's choice, without clearing, filling and scanning 96 bins.  Range by
// range a split of few spheres took 1.8 us, bound by the latency of one
// wave's instructions, and they are most of a build: k_sah_build of the book
// scene 155 -> 101 us, k_sah_treelets of a million spheres 836 -> 673 us.
__device__ __forceinline__ void sah_few(const float4* sph, uint32_t* perm, uint32_t a, uint32_t m, uint32_t d,
                                        uint32_t f, uint32_t self, uint32_t* __restrict__ child,
                                        uint32_t* __restrict__ parent_int, uint32_t* __restrict__ parent_leaf)
{
    const uint32_t lane = __lane_id(), k = lane / kSahFew, i = lane - k * kSahFew, row = k * kSahFew;
    const bool in = k < 3u && i < m;
    uint32_t s = in ? 0u : 1u, e = in ? m - 1u : 0u;  // the range of place i
    const uint64_t below = (1ull << i) - 1ull;        // places before it
    for (;;) {
        const bool on = s < e;
        if (__ballot(on) == 0ull) return;
        const uint32_t p = in ? perm[a + i] : 0u;
        const float4 sp = sph[p];
        const float c = sah_cen(sp, (int)min(k, 2u));
        float lo = 3.4e38f, hi = -3.4e38f;
        for (uint32_t j = s; __ballot(on && j <= e) != 0ull; j++) {
            const float o = __shfl(c, (int)(row + j) & 63);
            lo = fminf(lo, j <= e ? o : 3.4e38f);
            hi = fmaxf(hi, j <= e ? o : -3.4e38f);
        }
        const float ext = hi - lo;
        const bool axis_on = on && ext > 0.0f && d < kSahDepthCap;
        int bin = 0;
        if (axis_on) bin = sah_bin(c, lo, ext);
        float l[6], r[6];
        for (int q = 0; q < 3; q++) {
            l[q] = r[q] = 3.4e38f;
            l[3 + q] = r[3 + q] = -3.4e38f;
        }
        uint32_t nl = 0;
        for (uint32_t j = s; __ballot(on && j <= e) != 0ull; j++) {
            const float4 o = sph[perm[a + min(j, m - 1u)]];
            const float cc[3] = {o.x, o.y, o.z}, rr = fabsf(o.w);
            const bool left = __shfl(bin, (int)(row + j) & 63) <= bin, use = j <= e;
            nl += use && left ? 1u : 0u;
            for (int q = 0; q < 3; q++) {
                const float b0 = cc[q] - rr, b1 = cc[q] + rr;
                l[q] = fminf(l[q], use && left ? b0 : 3.4e38f);
                l[3 + q] = fmaxf(l[3 + q], use && left ? b1 : -3.4e38f);
                r[q] = fminf(r[q], use && !left ? b0 : 3.4e38f);
                r[3 + q] = fmaxf(r[3 + q], use && !left ? b1 : -3.4e38f);
            }
        }
        const uint32_t len = e - s + 1u;
        const float cost = box_area6(l) * (float)nl + box_area6(r) * (float)(len - nl);
        // costs are not negative: they compare as their bits, NaN last
        uint32_t key = 0xFFFFFFFFu;  // no split here
        if (axis_on && nl < len) key = cost == cost ? __float_as_uint(cost + 0.0f) : 0x7FFFFFFFu;
        // the axis's choice over the range
        uint32_t bkey = 0xFFFFFFFFu, bsplit = 0;  // bin | left spheres << 8
        const uint32_t mine = (uint32_t)bin | nl << 8;
        for (uint32_t j = s; __ballot(on && j <= e) != 0ull; j++) {
            const uint32_t ok = __shfl(key, (int)(row + j) & 63), os = __shfl(mine, (int)(row + j) & 63);
            if (j <= e && (ok < bkey || (ok == bkey && (os & 0xFFu) < (bsplit & 0xFFu)))) {
                bkey = ok;
                bsplit = os;
            }
        }
        // the range's choice over the axes
        uint32_t best = 0xFFFFFFFFu, split = 0, axis = 3u;
        for (uint32_t q = 0; q < 3u; q++) {
            const uint32_t ok = __shfl(bkey, (int)(q * kSahFew + i) & 63), os = __shfl(bsplit, (int)(q * kSahFew + i) & 63);
            // as floats: a cost that is not a number neither beats nor is beaten
            if (ok != 0xFFFFFFFFu && (axis == 3u || (ok < best && best != 0x7FFFFFFFu))) {
                best = ok;
                split = os;
                axis = q;
            }
        }
        const int my_bin = __shfl(bin, (int)(min(axis, 2u) * kSahFew + i) & 63);
        const uint32_t left_n = axis == 3u ? len / 2u : split >> 8;
        const bool left = axis == 3u ? i - s < left_n : my_bin <= (int)(split & 0xFFu);
        // stable partition of every range
        const uint64_t ml = __ballot(left && k == 0u);
        const uint64_t seg = (2ull << e) - (1ull << s);  // places of the range
        const uint32_t before = (uint32_t)__popcll(ml & seg & below);
        if (on && k == 0u) perm[a + (left ? s + before : s + left_n + (i - s - before))] = p;
        const uint32_t g = s + left_n - 1u;  // last place of the left part
        if (on && k == 0u && i == s) {
            const uint32_t G = f + a + g, mr = len - left_n;  // children G and G + 1
            const uint32_t up = self | (((f + a + s) / kRefitLeaves == (f + a + e) / kRefitLeaves) ? kLocalBit : 0u);
            if (left_n == 1u) parent_leaf[G] = up; else parent_int[G] = up;
            if (mr == 1u) parent_leaf[G + 1u] = up; else parent_int[G + 1u] = up;
            child[self] = G | (left_n == 1u ? 1u << 30 : 0u) | (mr == 1u ? 2u << 30 : 0u);
        }
        wave_order();
        if (on) {
            self = f + a + g + (i <= g ? 0u : 1u);
            d++;
            if (i <= g) e = g;
            else s = g + 1u;
        }
    }
}

// Splits the range [a, b] (more than kSahFew spheres) at depth d, by one wave: its
// permutation is partitioned; returns the last index of the left part.
__device__ __forceinline__ uint32_t sah_split(const float4* sph, uint32_t* perm, uint32_t* tmp, uint32_t* bins, uint32_t a,
                                              uint32_t b, uint32_t d)
{
    const uint32_t lane = __lane_id(), m = b - a + 1u;
    // centre bounds; a range of at most a wave stays in registers
    float lo[3] = {3.4e38f, 3.4e38f, 3.4e38f}, hi[3] = {-3.4e38f, -3.4e38f, -3.4e38f};
    uint32_t p = 0;
    float4 sp = make_float4(0.f, 0.f, 0.f, 0.f);
    for (uint32_t i = a + lane; i <= b; i += 64u) {
        p = perm[i];
        sp = sph[p];
        for (int k = 0; k < 3; k++) {
            lo[k] = fminf(lo[k], sah_cen(sp, k));
            hi[k] = fmaxf(hi[k], sah_cen(sp, k));
        }
    }
    float ext[3];
    bool any = false;
    for (int k = 0; k < 3; k++) {
        lo[k] = wave_reduce<true>(lo[k]);
        hi[k] = wave_reduce<false>(hi[k]);
        ext[k] = hi[k] - lo[k];
        any = any || ext[k] > 0.0f;
    }
    if (!any || d >= kSahDepthCap) return a + m / 2u - 1u;
    // stable partition of a range in registers: spheres of bins up to bj to the left
    auto part_wave = [&](int bin, int bj, uint32_t nl) {
        const bool valid = lane < m, left = valid && bin <= bj;
        const uint64_t ml = __ballot(left), mr = __ballot(valid && !left);
        if (valid) perm[left ? a + mbcnt(ml) : a + nl + mbcnt(mr)] = p;
        wave_order();
        return a + nl - 1u;
    };
    for (int x = (int)lane; x < kSahBinWords; x += 64) bins[x] = x % 7 < 3 ? 0xFFFFFFFFu : 0u;
    wave_order();
    int mine[3] = {0, 0, 0};
    for (uint32_t i = a + lane; i <= b; i += 64u) {
        if (m > 64u) sp = sph[perm[i]];
        const float rr = fabsf(sp.w);
        const uint32_t klo[3] = {ord_key(sp.x - rr), ord_key(sp.y - rr), ord_key(sp.z - rr)};
        const uint32_t khi[3] = {ord_key(sp.x + rr), ord_key(sp.y + rr), ord_key(sp.z + rr)};
        for (int k = 0; k < 3; k++) {
            if (!(ext[k] > 0.0f)) continue;
            mine[k] = sah_bin(sah_cen(sp, k), lo[k], ext[k]);
            uint32_t* bn = &bins[(k * kSahBins + mine[k]) * 7];
            for (int q = 0; q < 3; q++) {
                atomicMin(&bn[q], klo[q]);
                atomicMax(&bn[3 + q], khi[q]);
            }
            atomicAdd(&bn[6], 1u);
        }
    }
    wave_order();
    // The cheapest split of each axis: lane j < 32 holds the union of bins
    // 0..j (min and max, exact in any order), lane 32 + j that of bins 31-j..31;
    // the split after bin j adds lane j's and lane 62 - j's products.
    int bk = -1, bj = 0;
    uint32_t nl = 0;
    float bc = 0.0f;
    for (int k = 0; k < 3; k++) {
        if (!(ext[k] > 0.0f)) continue;
        const int j = (int)(lane < 32u ? lane : 63u - lane);
        const uint32_t* bn = &bins[(k * kSahBins + j) * 7];
        uint32_t cnt = bn[6];
        float box[6];
        for (int q = 0; q < 3; q++) {
            box[q] = half_scan<true>(cnt ? ord_val(bn[q]) : 3.4e38f);
            box[3 + q] = half_scan<false>(cnt ? ord_val(bn[3 + q]) : -3.4e38f);
        }
        cnt = half_scan_add(cnt);
        const float part = box_area6(box) * (float)cnt;
        const uint32_t rn = __shfl(cnt, (int)(62u - lane) & 63);
        const float right = __shfl(part, (int)(62u - lane) & 63);
        const bool ok = lane < (uint32_t)kSahBins - 1u && cnt > 0u && rn > 0u;
        const float cost = part + right;
        const uint64_t okm = __ballot(ok);
        if (okm == 0ull) continue;
        // the first minimum (the first split at all if no cost is a number)
        const float best = wave_reduce<true>(ok ? cost : __builtin_huge_valf());
        const uint64_t bm = __ballot(ok && cost == best);
        const int cj = __ffsll((unsigned long long)(bm ? bm : okm)) - 1;
        const float c = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(cost), cj));
        if (bk < 0 || c < bc) {
            bk = k;
            bj = cj;
            bc = c;
            nl = (uint32_t)__builtin_amdgcn_readlane((int)cnt, cj);
        }
    }
    if (bk < 0) return a + m / 2u - 1u;
    if (m <= 64u) return part_wave(bk == 0 ? mine[0] : (bk == 1 ? mine[1] : mine[2]), bj, nl);
    uint32_t offl = a, offr = a + nl;
    const float blo = bk == 0 ? lo[0] : (bk == 1 ? lo[1] : lo[2]), bext = bk == 0 ? ext[0] : (bk == 1 ? ext[1] : ext[2]);
    for (uint32_t i0 = a; i0 <= b; i0 += 64u) {
        const uint32_t i = i0 + lane;
        const bool valid = i <= b;
        const uint32_t pi = valid ? perm[i] : 0u;
        const bool left = valid && sah_bin(sah_cen(sph[pi], bk), blo, bext) <= bj;
        const uint64_t ml = __ballot(left), mr = __ballot(valid && !left);
        if (valid) tmp[left ? offl + mbcnt(ml) : offr + mbcnt(mr)] = pi;
        offl += (uint32_t)__popcll(ml);
        offr += (uint32_t)__popcll(mr);
    }
    wave_order();
    for (uint32_t i = a + lane; i <= b; i += 64u) perm[i] = tmp[i];
    wave_order();
    return a + nl - 1u;
}

// Rebuilds the subtree over leaves [f, f + m) (2 <= m <= kSahMaxPrims), root
// node r at depth d0, in place: leaf_prim and keys are permuted within the
// range, and the child words and parent links of the subtree's nodes are
// rewritten.  In the Karras layout a subtree's node indices are fixed by its
// leaf range and root index, so the nodes above it are untouched.  Called
// by a whole workgroup of NW waves.
template <int NW>
__device__ __forceinline__ void sah_treelet(const float4* __restrict__ sph, uint32_t f, uint32_t m, uint32_t r,
                                            uint32_t d0, uint32_t* __restrict__ leaf_prim,
                                            uint32_t* __restrict__ keys, uint32_t* __restrict__ child,
                                            uint32_t* __restrict__ parent_int, uint32_t* __restrict__ parent_leaf,
                                            SahShared<NW>& sh)
{
    constexpr uint32_t NT = 64 * NW;
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t w = (uint32_t)__builtin_amdgcn_readfirstlane(tid >> 6);
    for (uint32_t i = tid; i < m; i += NT) {
        sh.sph[i] = sph[leaf_prim[f + i]];
        sh.perm[i] = i;
    }
    if (tid < kSahTasks) sh.task[tid] = tid == 0u ? make_uint2((m - 1u) << 10 | d0 << 20, r) : make_uint2(kSahNone, 0u);
    if (tid == 0) {
        sh.head = 0u;
        sh.tail = 1u;
        sh.open = 1u;
    }
    __syncthreads();
    for (;;) {
        // A ticket names a task, perhaps one that has not been written yet.
        // Every open task is being worked on by some wave (or is this wave's
        // to take), which writes no task after it has closed its own; so the
        // wait ends with this ticket's task or with none open.
        uint32_t ticket = 0, tx = kSahNone;
        if (lane == 0) ticket = atomicAdd(&sh.head, 1u);
        wave_order();
        ticket = (uint32_t)__builtin_amdgcn_readfirstlane(ticket);
        for (;;) {
            const uint32_t open = __hip_atomic_load(&sh.open, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP);
            tx = __hip_atomic_load(&sh.task[ticket].x, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP);
            if (tx != kSahNone || open == 0u) break;
            __builtin_amdgcn_s_sleep(1);
        }
        tx = (uint32_t)__builtin_amdgcn_readfirstlane(tx);
        if (tx == kSahNone) break;
        uint32_t self = (uint32_t)__builtin_amdgcn_readfirstlane(sh.task[ticket].y);
        for (;;) {
            const uint32_t a = tx & 0x3FFu, b = (tx >> 10) & 0x3FFu, d = tx >> 20;
            if (b - a < kSahFew) {
                sah_few(sh.sph, sh.perm, a, b - a + 1u, d, f, self, child, parent_int, parent_leaf);
                break;
            }
            const uint32_t g = sah_split(sh.sph, sh.perm, sh.tmp, sh.bin[w], a, b, d);
            const uint32_t G = f + g;  // split after leaf G: children G and G + 1
            const uint32_t ml = g - a + 1u, mr = b - g;
            if (lane == 0) {
                const uint32_t up = self | (((f + a) / kRefitLeaves == (f + b) / kRefitLeaves) ? kLocalBit : 0u);
                if (ml == 1u) parent_leaf[G] = up; else parent_int[G] = up;
                if (mr == 1u) parent_leaf[G + 1u] = up; else parent_int[G + 1u] = up;
                child[self] = G | (ml == 1u ? 1u << 30 : 0u) | (mr == 1u ? 2u << 30 : 0u);
            }
            wave_order();
            const uint2 tl = make_uint2(a | g << 10 | (d + 1u) << 20, G);
            const uint2 tr = make_uint2((g + 1u) | b << 10 | (d + 1u) << 20, G + 1u);
            const uint2 big = ml >= mr ? tl : tr, small = ml >= mr ? tr : tl;
            const uint32_t ms = min(ml, mr);
            if (ms >= kSahShare) {
                if (lane == 0) {
                    atomicAdd(&sh.open, 1u);
                    const uint32_t at = atomicAdd(&sh.tail, 1u);
                    sh.task[at].y = small.y;
                    __hip_atomic_store(&sh.task[at].x, small.x, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
                }
                wave_order();
            } else if (ms >= 2u) {
                sah_few(sh.sph, sh.perm, small.x & 0x3FFu, ms, d + 1u, f, small.y, child, parent_int, parent_leaf);
            }
            tx = big.x;
            self = big.y;
        }
        if (lane == 0) __hip_atomic_fetch_sub(&sh.open, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
        // keeps the wave's lanes together: without it the compiler sent all
        // lanes but the first straight past the next `if (lane == 0)`, and
        // they took ticket 0 again, by themselves, for ever
        wave_order();
    }
    __syncthreads();
    // permute the range's primitive ids and keys in place, staged through
    // LDS (the bins are free now) so every global read has landed before the
    // barrier that precedes the writes
    uint32_t* kbuf = &sh.bin[0][0];
    for (uint32_t i = tid; i < m; i += NT) {
        const uint32_t p = sh.perm[i];
        sh.tmp[i] = leaf_prim[f + p];
        kbuf[i] = keys[f + p];
    }
    __syncthreads();
    for (uint32_t i = tid; i < m; i += NT) {
        leaf_prim[f + i] = sh.tmp[i];
        keys[f + i] = kbuf[i];
    }
    __syncthreads();  // the LDS is reused by the next treelet
}

// A small scene: the whole tree is one SAH build (keys and identity
// permutation in sphere order in, leaf order out).
__global__ void __launch_bounds__(64 * kSahSoloWaves) k_sah_build(const float4* __restrict__ sph, uint32_t n,
                                                           uint32_t* __restrict__ leaf_prim,
                                                           uint32_t* __restrict__ keys,
                                                           uint32_t* __restrict__ child,
                                                           uint32_t* __restrict__ parent_int,
                                                           uint32_t* __restrict__ parent_leaf)
{
    __shared__ SahShared<kSahSoloWaves> sh;
    if (threadIdx.x == 0) parent_int[0] = 0xFFFFFFFFu;
    sah_treelet<kSahSoloWaves>(sph, 0u, n, 0u, 0u, leaf_prim, keys, child, parent_int, parent_leaf, sh);
}

// A large LBVH: the roots of its treelets, the maximal subtrees of at most
// kSahMaxPrims leaves whose root lies above kSahDepthCap.  Internal node i
// (leaves range[i]) is one when it is small enough and its parent is not;
// its depth is the length of its parent chain.  Appended as (first leaf,
// leaves, node, depth) in any order: the treelets are disjoint.
__global__ void __launch_bounds__(kBlk) k_treelet_roots(const uint2* __restrict__ range,
                                                        const uint32_t* __restrict__ parent_int, uint32_t ni,
                                                        uint4* __restrict__ list, uint32_t* __restrict__ count)
{
    const uint32_t i = blockIdx.x * kBlk + threadIdx.x;
    if (i == 0u || i >= ni) return;
    const uint2 ri = range[i];
    const uint32_t m = ri.y - ri.x + 1u;
    const uint32_t p = parent_int[i] & ~kLocalBit;
    const uint2 rp = range[p];
    if (m > kSahMaxPrims || rp.y - rp.x + 1u <= kSahMaxPrims) return;
    uint32_t d = 1, q = p;
    while (q != 0u && d <= kMaxDepth) {
        q = parent_int[q] & ~kLocalBit;
        d++;
    }
    if (d >= kSahDepthCap) return;
    list[atomicAdd(count, 1u)] = make_uint4(ri.x, m, i, d);
}

__global__ void __launch_bounds__(64 * kSahWaves) k_sah_treelets(const float4* __restrict__ sph,
                                                              const uint4* __restrict__ list,
                                                              const uint32_t* __restrict__ count,
                                                              uint32_t* __restrict__ leaf_prim,
                                                              uint32_t* __restrict__ keys,
                                                              uint32_t* __restrict__ child,
                                                              uint32_t* __restrict__ parent_int,
                                                              uint32_t* __restrict__ parent_leaf)
{
    __shared__ SahShared<kSahWaves> sh;
    const uint32_t cnt = *count;
    for (uint32_t t = blockIdx.x; t < cnt; t += gridDim.x) {
        const uint4 e = list[t];
        sah_treelet<kSahWaves>(sph, e.x, e.y, e.z, e.w, leaf_prim, keys, child, parent_int, parent_leaf, sh);
    }
}

// ---- 6. refit + pack ---------------------------------------------------------------
__device__ __forceinline__ uint32_t pick_exp(float lo, float hi)
{
    float ext = hi - lo;
    uint32_t e = 1;
    if (ext > 0.0f) {
        float m = ext / 255.0f;
        uint32_t b = __float_as_uint(m);
        uint32_t ex = b >> 23, mant = b & 0x7FFFFFu;
        e = (ex == 0u) ? 1u : ex + (mant != 0u ? 1u : 0u);
        if (e < 1u) e = 1u;
    }
    while (e < 254u && __builtin_fmaf(__uint_as_float(e << 23), 255.0f, lo) < hi) e++;
    return e;
}

__device__ __forceinline__ uint32_t quant_lo(float v, float lo, float s)
{
    int q = (int)floorf((v - lo) / s);
    q = q < 0 ? 0 : (q > 255 ? 255 : q);
    while (q > 0 && __builtin_fmaf(s, (float)q, lo) > v) q--;
    return (uint32_t)q;
}

__device__ __forceinline__ uint32_t quant_hi(float v, float lo, float s)
{
    int q = (int)ceilf((v - lo) / s);
    q = q < 0 ? 0 : (q > 255 ? 255 : q);
    while (q < 255 && __builtin_fmaf(s, (float)q, lo) < v) q++;
    return (uint32_t)q;
}


__device__ __forceinline__ void leaf_box(const float4 sp, float* b)
{
    const float r = fabsf(sp.w);
    b[0] = sp.x - r; b[1] = sp.y - r; b[2] = sp.z - r;
    b[3] = sp.x + r; b[4] = sp.y + r; b[5] = sp.z + r;
}

// A node's box (lo, hi), six floats: in 64 bits, since node * 6 outgrows 32
// below the 2^30 spheres a scene may have.
template <class F>
__device__ __forceinline__ F* node_box(F* boxes, uint32_t node)
{
    return boxes + (size_t)node * 6;
}

// Union of the two child boxes.
__device__ __forceinline__ void join_boxes(const float (&cb)[2][6], float (&nb)[6])
{
    for (int k = 0; k < 3; k++) {
        nb[k] = fminf(cb[0][k], cb[1][k]);
        nb[3 + k] = fmaxf(cb[0][3 + k], cb[1][3 + k]);
    }
}

// The 32-byte packed node p, once every box is known: one thread per node.
// The refit's climbs used to pack each node on their way, which put some 20
// divisions on every level of their serial chains (local part of a million
// spheres 315 us, of the book scene 65 us).
__device__ __forceinline__ void pack_node(uint32_t p, const float4* __restrict__ sph, const uint32_t* __restrict__ child,
                                          const float* __restrict__ boxes, uint4* __restrict__ nodes)
{
    const uint32_t cw = child[p], g = cw & 0x3FFFFFFFu, flags = cw >> 30;
    float cb[2][6], nb[6];
    for (uint32_t c = 0; c < 2; c++) {
        if ((flags >> c) & 1u) leaf_box(sph[g + c], cb[c]);
        else
            for (int k = 0; k < 6; k++) cb[c][k] = node_box(boxes, g + c)[k];
    }
    join_boxes(cb, nb);
    uint32_t meta = 0, q[3];
    for (int k = 0; k < 3; k++) {
        const float lo = nb[k], hi = nb[3 + k];
        const uint32_t e = pick_exp(lo, hi);
        const float sc = __uint_as_float(e << 23);
        meta |= e << (8 * k);
        const uint32_t l0 = quant_lo(cb[0][k], lo, sc), h0 = quant_hi(cb[0][3 + k], lo, sc);
        const uint32_t l1 = quant_lo(cb[1][k], lo, sc), h1 = quant_hi(cb[1][3 + k], lo, sc);
        q[k] = l0 | (h0 << 8) | (l1 << 16) | (h1 << 24);
    }
    meta |= flags << 24;
    nodes[2 * (size_t)p] = make_uint4(__float_as_uint(nb[0]), __float_as_uint(nb[1]), __float_as_uint(nb[2]), meta);
    nodes[2 * (size_t)p + 1] = make_uint4(q[0], q[1], q[2], g);
}
__global__ void __launch_bounds__(kBlk) k_pack_nodes(const float4* __restrict__ sph, const uint32_t* __restrict__ child,
                                                     const float* __restrict__ boxes, uint32_t ni,
                                                     uint4* __restrict__ nodes)
{
    const uint32_t p = blockIdx.x * kBlk + threadIdx.x;
    if (p < ni) pack_node(p, sph, child, boxes, nodes);
}

// Bottom-up refit (Karras 2012, section 4): one thread per leaf climbs, and
// the second thread to reach a node refits it.  Split in two kernels so that
// the bulk of the nodes needs no cross-XCD coherence:
//   k_refit_local  one workgroup per kRefitLeaves leaves.  Every node whose
//                  leaf range lies inside the workgroup's range also has its
//                  index there, so its child word, parent link, arrival
//                  counter, box and height all live in LDS.  A climb stops
//                  below the first node whose range crosses workgroups and
//                  publishes the finished child (a leaf or a local node) on
//                  the frontier list.
//   k_refit_top    climbs from every frontier entry through the crossing
//                  nodes (about n / kRefitLeaves * log2 kRefitLeaves of them)
//                  in global memory: up to kTopOneLeaves leaves by one
//                  workgroup at workgroup scope, above by kTopBlocks of them
//                  at agent scope, where each step writes back what its L2
//                  holds dirty (little: the kernel boundary wrote the local
//                  results back) and so takes some 4 us, but many run at a
//                  time.  Whole refits by one workgroup and by many, us: 200k
//                  spheres 255 and 298, 393k 344 and 381, 550k 422 and 435,
//                  700k 489 and 498 (504 and 501), a million 673 and 607.  With
//                  every node at agent scope in one kernel the build of a
//                  million spheres took 10 ms.
constexpr uint32_t kLeafItem = 0x80000000u;  // frontier entry is a leaf index
constexpr uint32_t kRefitThreads = 1024;
constexpr uint32_t kLeavesPerThread = kRefitLeaves / kRefitThreads;

__global__ void __launch_bounds__(kRefitThreads) k_refit_local(const float4* __restrict__ sph, uint32_t n,
                                                               const uint32_t* __restrict__ child,
                                                               const uint32_t* __restrict__ parent_int,
                                                               const uint32_t* __restrict__ parent_leaf,
                                                               float* __restrict__ boxes,
                                                               uint32_t* __restrict__ height,
                                                               uint32_t* __restrict__ frontier,
                                                               uint32_t* __restrict__ fcount)
{
    __shared__ uint32_t s_visit[kRefitLeaves];
    __shared__ uint32_t s_child[kRefitLeaves];
    __shared__ uint32_t s_up[kRefitLeaves];
    __shared__ uint32_t s_h[kRefitLeaves];
    __shared__ float s_box[6][kRefitLeaves];
    const uint32_t tid = threadIdx.x, base = blockIdx.x * kRefitLeaves;
    for (uint32_t i = tid; i < kRefitLeaves; i += kRefitThreads) {
        s_visit[i] = 0u;
        const uint32_t g = base + i;
        if (g + 1u < n) {  // internal nodes are 0 .. n-2
            s_child[i] = child[g];
            s_up[i] = parent_int[g];
        }
    }
    __syncthreads();
    for (uint32_t r = 0; r < kLeavesPerThread; r++) {
        const uint32_t leaf = base + r * kRefitThreads + tid;
        if (leaf >= n) break;
        uint32_t up = parent_leaf[leaf];
        uint32_t done = leaf | kLeafItem;  // the highest node this climb has finished
        float nb[6];
        uint32_t nh = 0;
        while (up & kLocalBit) {
            const uint32_t p = up & ~kLocalBit, slot = p - base;
            if (__hip_atomic_fetch_add(&s_visit[slot], 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_WORKGROUP) == 0u)
                break;
            const uint32_t cw = s_child[slot];
            const uint32_t g = cw & 0x3FFFFFFFu, flags = cw >> 30;
            float cb[2][6];
            uint32_t h = 0;
            for (int c = 0; c < 2; c++) {
                const uint32_t ch = g + (uint32_t)c;
                if ((flags >> c) & 1u) {
                    leaf_box(sph[ch], cb[c]);
                } else {
                    const uint32_t cs = ch - base;
                    for (int k = 0; k < 6; k++)
                        cb[c][k] = __hip_atomic_load(&s_box[k][cs], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                    h = max(h, __hip_atomic_load(&s_h[cs], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
                }
            }
            join_boxes(cb, nb);
            nh = h + 1u;
            for (int k = 0; k < 6; k++) {
                __hip_atomic_store(&s_box[k][slot], nb[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                node_box(boxes, p)[k] = nb[k];  // every node's exact box: packing and the 4-wide collapse read them
            }
            __hip_atomic_store(&s_h[slot], nh, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            done = p;
            if (p == 0u) break;  // the whole tree was local
            up = s_up[slot];
        }
        if (up & kLocalBit) {
            // stopped inside the workgroup: first arrival, or the local root
            if (done != 0u) continue;
        }
        if (!(done & kLeafItem)) {  // a finished local node: publish its box and height
            for (int k = 0; k < 6; k++) node_box(boxes, done)[k] = nb[k];
            height[done] = nh;
        }
        if (done != 0u) frontier[atomicAdd(fcount, 1u)] = done;
    }
}

constexpr uint32_t kTopBlocks = 64;
constexpr uint32_t kTopOneLeaves = 320 * kRefitLeaves;

template <int SCOPE>  // of the climbs' counters, boxes and heights
__global__ void __launch_bounds__(kRefitThreads) k_refit_top(const float4* __restrict__ sph,
                                                    const uint32_t* __restrict__ child,
                                                    const uint32_t* __restrict__ parent_int,
                                                    const uint32_t* __restrict__ parent_leaf,
                                                    const uint32_t* __restrict__ frontier,
                                                    const uint32_t* __restrict__ fcount, uint32_t* visit,
                                                    float* boxes, uint32_t* height)
{
    const uint32_t count = *fcount;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < count; i += gridDim.x * blockDim.x) {
        const uint32_t item = frontier[i];
        uint32_t p = ((item & kLeafItem) ? parent_leaf[item & ~kLeafItem] : parent_int[item]) & ~kLocalBit;
        for (;;) {
            if (__hip_atomic_fetch_add(&visit[p], 1u, __ATOMIC_ACQ_REL, SCOPE) == 0u) break;
            const uint32_t cw = child[p];
            const uint32_t g = cw & 0x3FFFFFFFu, flags = cw >> 30;
            float cb[2][6];
            uint32_t h = 0;
            for (int c = 0; c < 2; c++) {
                const uint32_t ch = g + (uint32_t)c;
                if ((flags >> c) & 1u) {
                    leaf_box(sph[ch], cb[c]);
                } else {
                    for (int k = 0; k < 6; k++)
                        cb[c][k] = __hip_atomic_load(node_box(boxes, ch) + k, __ATOMIC_RELAXED, SCOPE);
                    h = max(h, __hip_atomic_load(&height[ch], __ATOMIC_RELAXED, SCOPE));
                }
            }
            float nb[6];
            join_boxes(cb, nb);
            for (int k = 0; k < 6; k++) __hip_atomic_store(node_box(boxes, p) + k, nb[k], __ATOMIC_RELAXED, SCOPE);
            __hip_atomic_store(&height[p], h + 1u, __ATOMIC_RELAXED, SCOPE);
            if (p == 0u) break;
            p = parent_int[p] & ~kLocalBit;
        }
    }
}

// ---- 7. the 4-wide tree ---------------------------------------------------------
// Collapsed top down from the binary tree, level by level: a wide root's
// children start as its binary node's two children; while there are fewer
// than 4, the internal child of largest box area (the first on a tie) is
// opened into its two children in place, so slots keep left-to-right leaf
// order.  Every internal child becomes a wide root of the next level.  Wide
// indices number the roots in binary index order (an exclusive scan of the
// root flags), so the tree does not depend on the order threads ran in.
// Each wide node (64 bytes) is quantised relative to its own box like the
// binary nodes: lo corner, per-axis power-of-two scale, planes rounded
// outward; meta holds the scale exponents, the slots' leaf flags (bits
// 24-27) and valid flags (28-31).
constexpr uint32_t kWideRoot = 0x80000000u;  // wide-root flag of a binary node
constexpr uint32_t kLeafRef = 0x80000000u;   // a wide child that is a leaf
// Words behind the roots per level [0, kMaxDepth].
constexpr uint32_t kWideCount = kMaxDepth + 1;   // wide nodes
constexpr uint32_t kLeafCount = kMaxDepth + 2;   // leaves given a place so far
constexpr uint32_t kWideError = kMaxDepth + 3;   // the structural check's result
constexpr uint32_t kTreeHeight = kMaxDepth + 4;  // of the binary tree
constexpr uint32_t kFirstLevel = kMaxDepth + 5;  // first level that k_wide_few left
constexpr uint32_t kOddMaterials = kMaxDepth + 6;  // as k_reorder found them
constexpr uint32_t kBound = kMaxDepth + 7;       // largest |coordinate| of the root box (float)
constexpr uint32_t kWideWords = kMaxDepth + 8;
constexpr uint32_t kScanItems = 4;            // root flags per thread in the index scan
constexpr uint32_t kScanTile = kBlk * kScanItems;

__device__ __forceinline__ float box_area(const float* b)
{
    const float dx = b[3] - b[0], dy = b[4] - b[1], dz = b[5] - b[2];
    return dx * dy + dy * dz + dz * dx;
}

__device__ __forceinline__ uint32_t child_ref(uint32_t cw, int c)
{
    const uint32_t g = (cw & 0x3FFFFFFFu) + (uint32_t)c;
    return ((cw >> (30 + c)) & 1u) ? (g | kLeafRef) : g;
}

// The children of wide root r: starts as its binary node's two, and opens the
// internal one of largest box area while there are fewer than 4.  Areas are
// kept, so every box is read once.
__device__ __forceinline__ uint32_t wide_children(uint32_t r, const uint32_t* __restrict__ child,
                                                  const float* __restrict__ boxes, uint32_t (&ks)[4])
{
    const uint32_t cw = child[r];
    float area[4] = {-1.0f, -1.0f, -1.0f, -1.0f};  // of leaves and absent slots: never opened
    ks[0] = child_ref(cw, 0);
    ks[1] = child_ref(cw, 1);
    ks[2] = ks[3] = 0u;
    bool internal[4] = {!(ks[0] & kLeafRef), !(ks[1] & kLeafRef), false, false};
    for (int k = 0; k < 2; k++)
        if (internal[k]) area[k] = box_area(node_box(boxes, ks[k]));
    uint32_t n_k = 2;
#pragma unroll
    for (int round = 0; round < 2; round++) {
        int best = -1;
        float ba = 0.0f;
#pragma unroll
        for (int k = 0; k < 4; k++)
            if (internal[k] && (best < 0 || area[k] > ba)) {
                best = k;
                ba = area[k];
            }
        if (best < 0) break;
        const uint32_t opened = best == 0 ? ks[0] : (best == 1 ? ks[1] : (best == 2 ? ks[2] : ks[3]));
        const uint32_t ow = child[opened];
        const uint32_t c0 = child_ref(ow, 0), c1 = child_ref(ow, 1);
        const bool i0 = !(c0 & kLeafRef), i1 = !(c1 & kLeafRef);
        const float a0 = i0 ? box_area(node_box(boxes, c0)) : -1.0f;
        const float a1 = i1 ? box_area(node_box(boxes, c1)) : -1.0f;
        // c0 takes the opened slot, c1 the next; the slots after move up
#pragma unroll
        for (int k = 3; k >= 0; k--) {
            if (k > best + 1) {
                ks[k] = ks[k > 0 ? k - 1 : 0];
                area[k] = area[k > 0 ? k - 1 : 0];
                internal[k] = internal[k > 0 ? k - 1 : 0];
            } else if (k == best + 1) {
                ks[k] = c1;
                area[k] = a1;
                internal[k] = i1;
            } else if (k == best) {
                ks[k] = c0;
                area[k] = a0;
                internal[k] = i0;
            }
        }
        n_k++;
    }
    return n_k;
}

struct LevelArrays {
    const uint32_t* child;
    const float* boxes;
    uint32_t* front[2];   // roots of the even levels, of the odd ones
    uint32_t *wkids, *wflag;
    uint32_t *tidx, *tchild, *tleaf;  // of a root: its place in level order, its first child's, its first leaf's
};

// One level: every wide root of the frontier picks its children; internal
// children are the next level's frontier.  alloc(in, leaves, at, leaf_at),
// called by the last lane of a wave, gives the wave's children and leaves
// their places (once per child, and a maximum per root for the depth, kept one
// address busy: 414 us for the levels of a million spheres).
template <class Alloc>
__device__ __forceinline__ void wide_roots(const LevelArrays& A, uint32_t level, uint32_t count, uint32_t before,
                                           uint32_t first, uint32_t stride, Alloc alloc)
{
    const uint32_t lane = lane_id();
    const uint32_t* front_in = A.front[level & 1u];
    uint32_t* front_out = A.front[(level & 1u) ^ 1u];
    for (uint32_t i0 = first & ~63u; i0 < count; i0 += stride) {
        const uint32_t i = i0 + lane;
        uint32_t ks[4] = {0u, 0u, 0u, 0u}, n_k = 0, n_in = 0, r = 0;
        if (i < count) {
            r = front_in[i];
            n_k = wide_children(r, A.child, A.boxes, ks);
            reinterpret_cast<uint4*>(A.wkids)[r] = make_uint4(ks[0], ks[1], ks[2], ks[3]);
            A.wflag[r] = kWideRoot | n_k;
            for (uint32_t k = 0; k < 4u; k++) n_in += k < n_k && !(ks[k] & kLeafRef) ? 1u : 0u;
        }
        const uint32_t n_leaf = n_k - n_in;
        uint32_t incl = n_in, lincl = n_leaf;
        for (uint32_t off = 1; off < 64u; off <<= 1) {
            const uint32_t x = __shfl_up(incl, off), y = __shfl_up(lincl, off);
            if (lane >= off) {
                incl += x;
                lincl += y;
            }
        }
        uint32_t base = 0, lbase = 0;
        if (lane == 63u) alloc(incl, lincl, base, lbase);
        uint32_t at = __shfl(base, 63) + incl - n_in;
        const uint32_t lat = __shfl(lbase, 63) + lincl - n_leaf;
        if (i < count) {
            A.tidx[r] = before + i;
            A.tchild[r] = before + count + at;
            A.tleaf[r] = lat;
        }
        for (uint32_t k = 0; k < 4u; k++) {
            if (k >= n_k || (ks[k] & kLeafRef)) continue;
            A.wflag[ks[k]] = kWideRoot;
            front_out[at++] = ks[k];
        }
    }
}

// Levels by one workgroup, while they have at most `limit` roots.
constexpr uint32_t kFewThreads = 1024;
struct FewShared {
    uint32_t next[3];  // roots of the next level; three by turns, so that one barrier a level is enough
    uint32_t leaves;
};
__device__ __forceinline__ void few_levels(const LevelArrays& A, uint32_t* cnt, uint32_t& level, uint32_t& count,
                                           uint32_t before, uint32_t limit, FewShared& sh)
{
    uint32_t turn = 0;
    while (count != 0u && count <= limit && level < kMaxDepth) {
        uint32_t* next = &sh.next[turn];
        turn = turn == 2u ? 0u : turn + 1u;
        if (threadIdx.x == 0u) sh.next[turn] = 0u;
        wide_roots(A, level, count, before, threadIdx.x, kFewThreads,
                   [&](uint32_t in, uint32_t leaves, uint32_t& at, uint32_t& leaf_at) {
                       if (in) at = atomicAdd(next, in);
                       if (leaves) leaf_at = atomicAdd(&sh.leaves, leaves);
                   });
        __syncthreads();
        before += count;
        count = *next;
        level++;
        if (threadIdx.x == 0u) cnt[level] = count;
    }
}

// Clears the level words and sets up level 0: the root, unless the tree is
// deeper than the host will take.
__device__ __forceinline__ uint32_t first_level(const LevelArrays& A, uint32_t* cnt, const uint32_t* height,
                                                const uint32_t* odd, FewShared& sh)
{
    const uint32_t t = threadIdx.x, h = height[0], count = h + 1u <= kMaxDepth ? 1u : 0u;
    if (t < kWideWords) cnt[t] = t == 0u ? count : (t == kTreeHeight ? h : (t == kOddMaterials ? *odd : 0u));
    if (t == 0u) {
        A.wflag[0] = kWideRoot;
        A.front[0][0] = 0u;
        sh.next[0] = 0u;
        sh.leaves = 0u;
    }
    __syncthreads();
    return count;
}

// The levels of a larger scene.  One workgroup takes those at the top, which
// have few roots; the next `mids` levels have a launch each; whatever is left
// below, one workgroup again.  A launch for every level that the binary depth
// allows for, most of them empty, cost 4 us each: 22 of them at 200k spheres,
// 25 at a million.  With kFewRoots at a workgroup's size the top levels
// take some 4 us each, no longer than a launch.
constexpr uint32_t kFewRoots = 2048;
__global__ void __launch_bounds__(kFewThreads) k_wide_few(LevelArrays A, uint32_t* cnt, const uint32_t* height,
                                                          const uint32_t* odd, uint32_t resume, uint32_t mids)
{
    __shared__ FewShared sh;
    uint32_t level = 0, count, before = 0;
    if (!resume) {
        count = first_level(A, cnt, height, odd, sh);
        few_levels(A, cnt, level, count, 0u, kFewRoots, sh);
        if (threadIdx.x == 0u) {
            cnt[kFirstLevel] = level;
            cnt[kLeafCount] = sh.leaves;
        }
        return;
    }
    level = cnt[kFirstLevel] + mids;
    if (level >= kMaxDepth) return;
    count = cnt[level];
    for (uint32_t l = 0; l < level; l++) before += cnt[l];
    if (threadIdx.x == 0u) {
        sh.next[0] = 0u;
        sh.leaves = cnt[kLeafCount];
    }
    __syncthreads();
    few_levels(A, cnt, level, count, before, 0xFFFFFFFFu, sh);
}
__global__ void __launch_bounds__(kBlk) k_wide_level(LevelArrays A, uint32_t* __restrict__ cnt, uint32_t mid)
{
    const uint32_t level = cnt[kFirstLevel] + mid, lane = lane_id();
    if (level >= kMaxDepth) return;
    const uint32_t count = cnt[level];
    // roots of the levels above: the first of this level in level order
    uint32_t before = lane < level ? cnt[lane] : 0u;
    for (int o = 32; o >= 1; o >>= 1) before += __shfl_xor(before, o);
    wide_roots(A, level, count, before, blockIdx.x * kBlk + threadIdx.x, gridDim.x * kBlk,
               [&](uint32_t in, uint32_t leaves, uint32_t& at, uint32_t& leaf_at) {
                   if (in) at = atomicAdd(&cnt[level + 1], in);
                   if (leaves) leaf_at = atomicAdd(&cnt[kLeafCount], leaves);
               });
}

// Wide indices: an exclusive scan of the root flags over the binary nodes,
// in tiles of kScanTile (tile totals, their scan, then each tile's own).
__global__ void __launch_bounds__(kBlk) k_wscan_tiles(const uint32_t* __restrict__ wflag, uint32_t ni,
                                                      uint32_t* __restrict__ tsum)
{
    __shared__ uint32_t s[kBlk];
    uint32_t c = 0;
    const uint32_t base = blockIdx.x * kScanTile;
    for (uint32_t r = 0; r < kScanItems; r++) {
        const uint32_t i = base + r * kBlk + threadIdx.x;
        if (i < ni && (wflag[i] & kWideRoot)) c++;
    }
    const uint32_t e = block_scan_excl(c, s);
    if (threadIdx.x == kBlk - 1) tsum[blockIdx.x] = e + c;
}

__global__ void __launch_bounds__(kBlk) k_wscan_top(uint32_t* __restrict__ tsum, uint32_t nt,
                                                    uint32_t* __restrict__ total)
{
    __shared__ uint32_t part[kBlk];
    const uint32_t chunk = (nt + kBlk - 1) / kBlk;
    const uint32_t b = threadIdx.x * chunk, e = min(b + chunk, nt);
    uint32_t sum = 0;
    for (uint32_t i = b; i < e; i++) sum += tsum[i];
    const uint32_t excl = block_scan_excl(sum, part);
    uint32_t run = excl;
    for (uint32_t i = b; i < e; i++) {
        const uint32_t v = tsum[i];
        tsum[i] = run;
        run += v;
    }
    if (threadIdx.x == kBlk - 1) *total = excl + sum;
}

__global__ void __launch_bounds__(kBlk) k_wscan_apply(const uint32_t* __restrict__ wflag, uint32_t ni,
                                                      const uint32_t* __restrict__ tsum,
                                                      uint32_t* __restrict__ widx)
{
    __shared__ uint32_t s[kBlk];
    const uint32_t base = blockIdx.x * kScanTile + threadIdx.x * kScanItems;  // items contiguous per thread
    uint32_t f[kScanItems], c = 0;
    for (uint32_t r = 0; r < kScanItems; r++) {
        const uint32_t i = base + r;
        f[r] = (i < ni && (wflag[i] & kWideRoot)) ? 1u : 0u;
        c += f[r];
    }
    uint32_t run = tsum[blockIdx.x] + block_scan_excl(c, s);
    for (uint32_t r = 0; r < kScanItems; r++) {
        const uint32_t i = base + r;
        if (f[r]) widx[i] = run;
        run += f[r];
    }
}

// What k_wide_pack writes for the traversals that do not count: the same tree
// as 48-byte nodes, three 16-byte loads a visit instead of four, and the
// leaves in the order of the nodes that name them.  A node's internal
// children come first in its slots and lie next to each other in level
// order, its leaves after them likewise, so one index each stands for all of
// them (a traversal of many rays is bound by the L1's accesses as much as by
// the VALU).  Words: the node box's lo corner (3 floats); scale exponents
// (bytes 0-2) and the number of internal children (byte 3); the quantised lo
// planes of the 4 slots for x, y, z, then the hi planes (byte c = slot c; an
// empty slot's lie the wrong way round); the first internal child (in units
// of 16 bytes), the first leaf.  An empty slot that an extreme ray passes all
// the same names a leaf of some other node, or one of the spare ones at the
// end: testing it is harmless.
struct TravOut {
    const uint32_t *tidx, *tchild, *tleaf;
    const uint32_t* info;   // leaf order
    const float4* mat;
    uint32_t n;             // leaves
    uint4* nodes;           // 3 per node
    float4* sph;            // traversal order, 3 spare at the end
    uint32_t* tinfo;
    float4* tmat;
    uint32_t* bound;        // see kBound
};

__device__ __forceinline__ void wide_pack(uint32_t r, const float4* sph, const uint32_t* wkids, const uint32_t* wflag,
                                          const uint32_t* widx, const float* boxes, uint4* wnodes, const TravOut& T)
{
    const uint32_t fl = wflag[r];
    if (!(fl & kWideRoot)) return;
    const uint32_t cnt = fl & 7u;
    const float* nb = node_box(boxes, r);
    uint32_t meta = 0, qlo[3] = {0u, 0u, 0u}, qhi[3] = {0u, 0u, 0u}, ch[4] = {0u, 0u, 0u, 0u};
    uint32_t tlo[3] = {0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFFFFFFu}, thi[3] = {0u, 0u, 0u};
    float sc[3];
    for (int k = 0; k < 3; k++) {
        const uint32_t e = pick_exp(nb[k], nb[3 + k]);
        sc[k] = __uint_as_float(e << 23);
        meta |= e << (8 * k);
    }
    const uint4 refs = reinterpret_cast<const uint4*>(wkids)[r];
    const uint32_t ref[4] = {refs.x, refs.y, refs.z, refs.w};
    uint32_t n_in = 0;
    for (uint32_t c = 0; c < cnt; c++) n_in += (ref[c] & kLeafRef) ? 0u : 1u;
    const uint32_t scales = meta, leaf0 = T.tleaf[r];
    uint32_t slot_in = 0, slot_leaf = n_in;
    for (uint32_t c = 0; c < cnt; c++) {
        float cb[6];
        uint32_t t;  // the child's slot in the 48-byte node
        if (ref[c] & kLeafRef) {
            const uint32_t leaf = ref[c] & ~kLeafRef;
            const float4 s = sph[leaf];
            leaf_box(s, cb);
            ch[c] = leaf;
            meta |= 1u << (24 + c);
            t = slot_leaf++;
            const uint32_t at = leaf0 + t - n_in;
            T.sph[at] = s;
            T.tinfo[at] = T.info[leaf];
            T.tmat[at] = T.mat[leaf];
        } else {
            for (int k = 0; k < 6; k++) cb[k] = node_box(boxes, ref[c])[k];
            ch[c] = widx[ref[c]];
            t = slot_in++;
        }
        meta |= 1u << (28 + c);
        for (int k = 0; k < 3; k++) {
            const uint32_t lo = quant_lo(cb[k], nb[k], sc[k]), hi = quant_hi(cb[3 + k], nb[k], sc[k]);
            qlo[k] |= lo << (8 * c);
            qhi[k] |= hi << (8 * c);
            tlo[k] = (tlo[k] & ~(0xFFu << (8 * t))) | lo << (8 * t);
            thi[k] |= hi << (8 * t);
        }
    }
    uint4* w = wnodes + (size_t)widx[r] * 4;
    w[0] = make_uint4(__float_as_uint(nb[0]), __float_as_uint(nb[1]), __float_as_uint(nb[2]), meta);
    w[1] = make_uint4(qlo[0], qlo[1], qlo[2], qhi[0]);
    w[2] = make_uint4(qhi[1], qhi[2], ch[0], ch[1]);
    w[3] = make_uint4(ch[2], ch[3], 0u, 0u);
    uint4* v = T.nodes + (size_t)T.tidx[r] * 3;
    v[0] = make_uint4(__float_as_uint(nb[0]), __float_as_uint(nb[1]), __float_as_uint(nb[2]), scales | n_in << 24);
    v[1] = make_uint4(tlo[0], tlo[1], tlo[2], thi[0]);
    v[2] = make_uint4(thi[1], thi[2], 3u * T.tchild[r], leaf0);
    if (r == 0u) {
        float m = 0.0f;
        for (int k = 0; k < 6; k++) m = fmaxf(m, fabsf(nb[k]));
        *T.bound = __float_as_uint(m);
        // the spare leaves are one of the scene's once more
        for (uint32_t k = 0; k < 3; k++) {
            T.sph[T.n + k] = sph[0];
            T.tinfo[T.n + k] = T.info[0];
            T.tmat[T.n + k] = T.mat[0];
        }
    }
}
__global__ void __launch_bounds__(kBlk) k_wide_pack(const float4* __restrict__ sph, const uint32_t* __restrict__ wkids,
                                                    const uint32_t* __restrict__ wflag,
                                                    const uint32_t* __restrict__ widx,
                                                    const float* __restrict__ boxes, uint32_t ni,
                                                    uint4* __restrict__ wnodes, TravOut T)
{
    const uint32_t r = blockIdx.x * kBlk + threadIdx.x;
    if (r < ni) wide_pack(r, sph, wkids, wflag, widx, boxes, wnodes, T);
}

__global__ void k_zero(uint32_t* a, uint32_t n)
{
    uint32_t i = blockIdx.x * kBlk + threadIdx.x;
    if (i < n) a[i] = 0u;
}
__global__ void k_zero3(uint32_t* a, uint32_t na, uint32_t* b, uint32_t nb, uint32_t* c, uint32_t nc)
{
    uint32_t i = blockIdx.x * kBlk + threadIdx.x;
    if (i < na) a[i] = 0u;
    if (i < nb) b[i] = 0u;
    if (i < nc) c[i] = 0u;
}

__global__ void k_fill(uint32_t* a, uint32_t n, uint32_t v)
{
    uint32_t i = blockIdx.x * kBlk + threadIdx.x;
    if (i < n) a[i] = v;
}

// Validation of device-resident input: first[0] = lowest index of a sphere
// with a non-finite centre or a zero/non-finite radius, first[1] = lowest
// index of a material with an unknown type (0xFFFFFFFF: none).
__global__ void __launch_bounds__(kBlk) k_check_input(const float4* __restrict__ sph,
                                                      const vzMaterial* __restrict__ mat, uint32_t n,
                                                      uint32_t* __restrict__ first)
{
    for (uint32_t i = blockIdx.x * kBlk + threadIdx.x; i < n; i += gridDim.x * kBlk) {
        const float4 c = sph[i];
        if (!(isfinite(c.x) && isfinite(c.y) && isfinite(c.z) && isfinite(c.w) && c.w != 0.0f))
            atomicMin(&first[0], i);
        if (mat && mat[i].type > VZ_DIELECTRIC) atomicMin(&first[1], i);
    }
}

inline uint32_t blocks_for(uint32_t n, uint32_t per) { return (n + per - 1) / per; }

}  // namespace

void* SceneBlocks::take(size_t bytes, size_t* got)
{
    {
        std::lock_guard<std::mutex> lk(mu_);
        size_t best = kept_.size();
        for (size_t i = 0; i < kept_.size(); i++)  // the smallest that fits, not above twice the size
            if (kept_[i].bytes >= bytes && kept_[i].bytes <= 2 * bytes &&
                (best == kept_.size() || kept_[i].bytes < kept_[best].bytes))
                best = i;
        if (best < kept_.size()) {
            void* p = kept_[best].p;
            *got = kept_[best].bytes;
            kept_bytes_ -= *got;
            kept_.erase(kept_.begin() + best);
            return p;
        }
    }
    *got = bytes;
    return nullptr;
}

void SceneBlocks::give(void* p, size_t bytes)
{
    {
        std::lock_guard<std::mutex> lk(mu_);
        if (kept_.size() < 256 && kept_bytes_ + bytes <= kKeepBytes) {
            kept_.push_back({p, bytes});
            kept_bytes_ += bytes;
            return;
        }
    }
    (void)hipFree(p);
}

void SceneBlocks::trim()
{
    std::lock_guard<std::mutex> lk(mu_);
    for (const Block& b : kept_) (void)hipFree(b.p);
    kept_.clear();
    kept_bytes_ = 0;
}

bool device_alloc(vzContext ctx, void** p, size_t bytes)
{
    if (hipMalloc(p, bytes) == hipSuccess) return true;
    (void)hipGetLastError();
    ctx->scene_blocks.trim();
    if (hipMalloc(p, bytes) == hipSuccess) return true;
    (void)hipGetLastError();
    *p = nullptr;
    return false;
}

vzStatus lbvh_alloc(vzScene s)
{
    const uint32_t n = s->n, ni = n > 1 ? n - 1 : 1;
    s->hist_blocks = blocks_for(n, kTile);
    uint64_t bytes = 0;   // the arrays' own sizes (vzAccelInfo.device_bytes)
    size_t at = 0;        // their places in the block, 256-byte aligned
    struct Part {
        void** p;
        size_t at;
    };
    std::vector<Part> parts;
    auto part = [&](auto** p, size_t b) {
        parts.push_back({(void**)p, at});
        at += (b + 255) & ~(size_t)255;
        bytes += b;
    };
    part(&s->d_sph_in, sizeof(float4) * n);
    part(&s->d_mat_in, sizeof(vzMaterial) * n);
    for (int i = 0; i < 2; i++) {
        part(&s->d_keys[i], sizeof(uint32_t) * n);
        part(&s->d_vals[i], sizeof(uint32_t) * n);
    }
    part(&s->d_hist, sizeof(uint32_t) * 256 * (s->hist_blocks + 1));
    part(&s->d_bounds, sizeof(float) * (6 * 1024 + 32));  // partials, grid A, grid B
    part(&s->d_sph, sizeof(float4) * n);
    part(&s->d_leaf_info, sizeof(uint32_t) * n);
    part(&s->d_mat, sizeof(float4) * n);
    part(&s->d_nodes, sizeof(uint4) * 2 * ni);
    part(&s->d_boxes, sizeof(float) * 6 * ni);
    part(&s->d_child, sizeof(uint32_t) * ni);
    part(&s->d_parent_int, sizeof(uint32_t) * ni);
    part(&s->d_parent_leaf, sizeof(uint32_t) * n);
    part(&s->d_visit, sizeof(uint32_t) * ni);
    part(&s->d_height, sizeof(uint32_t) * ni);
    part(&s->d_frontier, sizeof(uint32_t) * n);
    part(&s->d_fcount, 256);
    part(&s->d_wnodes, sizeof(uint4) * 4 * ni);
    part(&s->d_tnodes, sizeof(uint4) * 3 * ni);
    part(&s->d_tsph, sizeof(float4) * (n + 3));
    part(&s->d_tinfo, sizeof(uint32_t) * (n + 3));
    part(&s->d_tmat, sizeof(float4) * (n + 3));
    part(&s->d_wkids, sizeof(uint32_t) * 4 * ni);
    part(&s->d_wflag, sizeof(uint32_t) * ni);
    part(&s->d_widx, sizeof(uint32_t) * (ni + blocks_for(ni, kScanTile) + 1));  // + tile sums
    part(&s->d_wfront[0], sizeof(uint32_t) * ni);
    part(&s->d_wfront[1], sizeof(uint32_t) * ni);
    part(&s->d_wcnt, sizeof(uint32_t) * kWideWords);
    s->arena = s->ctx->scene_blocks.take(at, &s->arena_bytes);
    if (!s->arena && !device_alloc(s->ctx, &s->arena, at))
        return set_error(VZ_ERROR_OUT_OF_MEMORY, "hipMalloc of scene buffers failed");
    for (const Part& q : parts) *q.p = (char*)s->arena + q.at;
    s->device_bytes = bytes;
    return VZ_SUCCESS;
}

void lbvh_free(vzScene s)
{
    if (s->arena) s->ctx->scene_blocks.give(s->arena, s->arena_bytes);
    s->arena = nullptr;
}

// Structural check of both packed forms of the 4-wide tree, so that traversal
// needs no per-visit guards: every child index in range, every leaf
// referenced by exactly one slot, every wide node but the root by exactly one
// slot and the root by none.  Then a walk from the root reaches each node at
// most once and ends.  References count 1 from a 64-byte node and kTravRef
// from a 48-byte one.  Any violation sets *err.
constexpr uint32_t kTravRef = 0x10000u;
__device__ __forceinline__ void wide_refs(uint32_t i, const uint4* wnodes, uint32_t nw, uint32_t n, uint32_t* wref,
                                          uint32_t* lref, uint32_t* err)
{
    const uint4 a = wnodes[4 * (size_t)i], c = wnodes[4 * (size_t)i + 2], d = wnodes[4 * (size_t)i + 3];
    const uint32_t valid = a.w >> 28, leafm = (a.w >> 24) & 0xFu;
    const uint32_t ch[4] = {c.z, c.w, d.x, d.y};
    for (int k = 0; k < 4; k++) {
        if (!((valid >> k) & 1u)) continue;
        if ((leafm >> k) & 1u) {
            if (ch[k] < n) atomicAdd(&lref[ch[k]], 1u);
            else *err = 1u;
        } else {
            if (ch[k] != 0u && ch[k] < nw) atomicAdd(&wref[ch[k]], 1u);
            else *err = 1u;
        }
    }
}
// r: a binary node, fl its wide-root flag word.
__device__ __forceinline__ void trav_refs(uint32_t r, uint32_t fl, const uint4* tnodes, const uint32_t* tidx,
                                          uint32_t nw, uint32_t n, uint32_t* tref, uint32_t* lref, uint32_t* err)
{
    if (!(fl & kWideRoot)) return;
    const uint32_t t = tidx[r];
    if (t >= nw) {
        *err = 1u;
        return;
    }
    const uint32_t meta = tnodes[3 * (size_t)t].w, first3 = tnodes[3 * (size_t)t + 2].z, first = first3 / 3u;
    const uint32_t leaf = tnodes[3 * (size_t)t + 2].w, n_in = meta >> 24, n_leaf = (fl & 7u) - n_in;
    if (n_in > 4u || n_leaf > 4u || leaf > n || n_leaf > n - leaf || (n_in && first == 0u) ||
        (n_in && first3 != 3u * first) || (n_in && first > nw) || (n_in && n_in > nw - first)) {
        *err = 1u;
        return;
    }
    for (uint32_t k = 0; k < n_in; k++) atomicAdd(&tref[first + k], 1u);
    for (uint32_t k = 0; k < n_leaf; k++) atomicAdd(&lref[leaf + k], kTravRef);
}
__device__ __forceinline__ bool refs_wrong(uint32_t i, uint32_t nw, const uint32_t* wref, const uint32_t* tref,
                                           const uint32_t* lref)
{
    return lref[i] != 1u + kTravRef || (i < nw && (wref[i] != (i == 0u ? 0u : 1u) || tref[i] != wref[i]));
}
__global__ void __launch_bounds__(kBlk) k_wide_refs(const uint4* __restrict__ wnodes, const uint4* __restrict__ tnodes,
                                                    const uint32_t* __restrict__ wflag,
                                                    const uint32_t* __restrict__ tidx, uint32_t ni,
                                                    const uint32_t* __restrict__ nwp, uint32_t n,
                                                    uint32_t* __restrict__ wref, uint32_t* __restrict__ tref,
                                                    uint32_t* __restrict__ lref, uint32_t* __restrict__ err)
{
    const uint32_t nw = *nwp;
    for (uint32_t i = blockIdx.x * kBlk + threadIdx.x; i < ni; i += gridDim.x * kBlk) {
        if (i < nw) wide_refs(i, wnodes, nw, n, wref, lref, err);
        trav_refs(i, wflag[i], tnodes, tidx, nw, n, tref, lref, err);
    }
}
__global__ void __launch_bounds__(kBlk) k_wide_verify(const uint32_t* __restrict__ nwp, uint32_t n,
                                                      const uint32_t* __restrict__ wref,
                                                      const uint32_t* __restrict__ tref,
                                                      const uint32_t* __restrict__ lref, uint32_t* __restrict__ err)
{
    const uint32_t nw = *nwp;
    for (uint32_t i = blockIdx.x * kBlk + threadIdx.x; i < n; i += gridDim.x * kBlk)
        if (refs_wrong(i, nw, wref, tref, lref)) *err = 1u;
}

// Everything that follows the refit of a small scene (at most kSahMaxPrims
// spheres, a thread each), one workgroup: the binary nodes, the levels, the
// wide indices, both packed forms and their check.  As launches of their own
// these were 22, each shorter than the gap to the next, and the host waited
// once between them: loading and tracing the book scene 440 -> 324 us with
// k_small_keys.
__global__ void __launch_bounds__(kSmallThreads) k_wide_small(LevelArrays A, const float4* sph, uint32_t n,
                                                              uint4* nodes, const uint32_t* height,
                                                              const uint32_t* odd, uint32_t* cnt,
                                                              uint32_t* widx, uint4* wnodes, TravOut T)
{
    __shared__ FewShared sh;
    __shared__ uint32_t wref[kSmallThreads], tref[kSmallThreads], lref[kSmallThreads], wsum[kSmallThreads / 64];
    const uint32_t t = threadIdx.x, ni = n - 1u;
    wref[t] = tref[t] = lref[t] = 0u;
    if (t > 0u && t < ni) A.wflag[t] = 0u;
    if (t < ni) pack_node(t, sph, A.child, A.boxes, nodes);
    uint32_t level = 0, count = first_level(A, cnt, height, odd, sh);
    if (count == 0u) return;
    few_levels(A, cnt, level, count, 0u, 0xFFFFFFFFu, sh);
    const uint32_t fl = t < ni ? A.wflag[t] : 0u;
    const uint64_t m = __ballot((fl & kWideRoot) != 0u);
    if (t % 64 == 0u) wsum[t / 64] = (uint32_t)__popcll(m);
    __syncthreads();
    uint32_t nw = 0, idx = mbcnt(m);
    for (uint32_t w = 0; w < kSmallThreads / 64; w++) {
        if (w < t / 64) idx += wsum[w];
        nw += wsum[w];
    }
    if (fl & kWideRoot) widx[t] = idx;
    if (t == 0u) cnt[kWideCount] = nw;
    __syncthreads();
    if (t < ni) wide_pack(t, sph, A.wkids, A.wflag, widx, A.boxes, wnodes, T);
    __syncthreads();
    if (t < nw) wide_refs(t, wnodes, nw, n, wref, lref, cnt + kWideError);
    trav_refs(t, fl, T.nodes, A.tidx, nw, n, tref, lref, cnt + kWideError);
    __syncthreads();
    if (t < n && refs_wrong(t, nw, wref, tref, lref)) cnt[kWideError] = 1u;
}

// The packed nodes and the 4-wide tree of the current binary tree (after
// every build and refit).
static vzStatus collapse_wide(vzScene s, hipStream_t st)
{
    const uint32_t n = s->n, ni = n - 1;
    uint32_t* cnt = s->d_wcnt;
    // places in level order, in buffers free at this point: the refit's
    // counters and the sort's second buffers
    const LevelArrays A{s->d_child, s->d_boxes, {s->d_wfront[0], s->d_wfront[1]}, s->d_wkids, s->d_wflag,
                        s->d_visit, s->d_keys[1], s->d_vals[1]};
    const TravOut T{A.tidx, A.tchild, A.tleaf, s->d_leaf_info, s->d_mat, n, s->d_tnodes, s->d_tsph, s->d_tinfo,
                    s->d_tmat, cnt + kBound};
    const uint32_t* odd = s->d_fcount + kOddWord;
    if (n <= kSahMaxPrims) {
        hipLaunchKernelGGL(k_wide_small, dim3(1), dim3(kSmallThreads), 0, st, A, s->d_sph, n, s->d_nodes, s->d_height,
                           odd, cnt, s->d_widx, s->d_wnodes, T);
    } else {
        const dim3 all(blocks_for(n, kBlk));
        hipLaunchKernelGGL(k_pack_nodes, all, dim3(kBlk), 0, st, s->d_sph, s->d_child, s->d_boxes, ni, s->d_nodes);
        // the levels of more than kFewRoots roots: some log4(n) - 6 of them
        // below the top, more where the tree is uneven (empty ones cost a
        // launch, ones left over one workgroup's time)
        uint32_t mids = 0;
        if (ni > kFewRoots)
            for (uint32_t v = ni; v > 4u; v /= 4u) mids++;
        const uint32_t grid = std::min<uint32_t>(1024u, blocks_for(ni, kBlk));
        hipLaunchKernelGGL(k_wide_few, dim3(1), dim3(kFewThreads), 0, st, A, cnt, s->d_height, odd, 0u, 0u);
        for (uint32_t m = 0; m < mids; m++)
            hipLaunchKernelGGL(k_wide_level, dim3(grid), dim3(kBlk), 0, st, A, cnt, m);
        if (mids) hipLaunchKernelGGL(k_wide_few, dim3(1), dim3(kFewThreads), 0, st, A, cnt, s->d_height, odd, 1u, mids);
        uint32_t* tsum = s->d_widx + ni;
        const uint32_t ntile = blocks_for(ni, kScanTile);
        hipLaunchKernelGGL(k_wscan_tiles, dim3(ntile), dim3(kBlk), 0, st, s->d_wflag, ni, tsum);
        hipLaunchKernelGGL(k_wscan_top, dim3(1), dim3(kBlk), 0, st, tsum, ntile, cnt + kWideCount);
        hipLaunchKernelGGL(k_wscan_apply, dim3(ntile), dim3(kBlk), 0, st, s->d_wflag, ni, tsum, s->d_widx);
        hipLaunchKernelGGL(k_wide_pack, all, dim3(kBlk), 0, st, s->d_sph, s->d_wkids, s->d_wflag, s->d_widx,
                           s->d_boxes, ni, s->d_wnodes, T);
        // reference counts in buffers free at this point: the level fronts and
        // the refit frontier (both rebuilt by every refit)
        uint32_t *wref = s->d_wfront[0], *tref = s->d_wfront[1], *lref = s->d_frontier;
        hipLaunchKernelGGL(k_zero3, all, dim3(kBlk), 0, st, wref, ni, tref, ni, lref, n);
        hipLaunchKernelGGL(k_wide_refs, dim3(grid), dim3(kBlk), 0, st, s->d_wnodes, s->d_tnodes, s->d_wflag, A.tidx,
                           ni, cnt + kWideCount, n, wref, tref, lref, cnt + kWideError);
        hipLaunchKernelGGL(k_wide_verify, dim3(grid), dim3(kBlk), 0, st, cnt + kWideCount, n, wref, tref, lref,
                           cnt + kWideError);
    }
    VZ_HIP_TRY(hipGetLastError());
    uint32_t h[kWideWords] = {};
    VZ_HIP_TRY(hipMemcpyAsync(h, cnt, sizeof(h), hipMemcpyDeviceToHost, st));
    VZ_HIP_TRY(hipStreamSynchronize(st));
    s->depth = h[kTreeHeight] + 1;
    if (s->depth > kMaxDepth)
        return set_error(VZ_ERROR_CAPACITY, "BVH depth " + std::to_string(s->depth) +
                                                " exceeds the traversal stack (" +
                                                std::to_string(kMaxDepth) + ")");
    s->nw = h[kWideCount];
    float bound;
    std::memcpy(&bound, &h[kBound], sizeof(bound));
    s->ordered = h[kOddMaterials] == 0u && bound < kOrderedBound;
    s->wdepth = 1;  // the leaf level below the deepest roots'
    for (uint32_t L = 0; L <= kMaxDepth; L++)
        if (h[L]) s->wdepth = L + 2;
    if (h[kWideError] != 0u) return set_error(VZ_ERROR_INTERNAL, "4-wide BVH failed its structural check");
    if (s->wdepth > kMaxWideDepth)
        return set_error(VZ_ERROR_CAPACITY, "4-wide BVH depth " + std::to_string(s->wdepth) +
                                                " exceeds the traversal stack (" + std::to_string(kMaxWideDepth) + ")");
    return VZ_SUCCESS;
}

static vzStatus refit_core(vzScene s, hipStream_t st)
{
    uint32_t n = s->n;
    if (n < 2) return VZ_SUCCESS;
    if (n > kSahMaxPrims)
        hipLaunchKernelGGL(k_zero3, dim3(blocks_for(n - 1, kBlk)), dim3(kBlk), 0, st, s->d_visit, n - 1, s->d_fcount, 1u,
                           s->d_wflag, n - 1);
    hipLaunchKernelGGL(k_refit_local, dim3(blocks_for(n, kRefitLeaves)), dim3(kRefitThreads), 0, st, s->d_sph,
                       n, s->d_child, s->d_parent_int, s->d_parent_leaf, s->d_boxes, s->d_height,
                       s->d_frontier, s->d_fcount);
    if (n > kRefitLeaves) {  // nodes that cross the workgroups' ranges
        const bool one = n <= kTopOneLeaves;
        hipLaunchKernelGGL(one ? k_refit_top<__HIP_MEMORY_SCOPE_WORKGROUP> : k_refit_top<__HIP_MEMORY_SCOPE_AGENT>,
                           dim3(one ? 1 : kTopBlocks), dim3(kRefitThreads), 0, st, s->d_sph, s->d_child,
                           s->d_parent_int, s->d_parent_leaf, s->d_frontier, s->d_fcount, s->d_visit, s->d_boxes,
                           s->d_height);
    }
    return collapse_wide(s, st);
}

vzStatus lbvh_build(vzScene s, hipStream_t st)
{
    uint32_t n = s->n;
    uint32_t nb = std::min<uint32_t>(1024, blocks_for(n, kBlk));
    Event e0, e1;
    VZ_EVENT_TRY(e0);
    VZ_EVENT_TRY(e1);
    VZ_HIP_TRY(hipEventRecord(e0.e, st));
    float* partial = s->d_bounds;
    float* fin = s->d_bounds + 6 * 1024;
    float* grid_b = fin + 16;
    if (n <= kSahMaxPrims) {
        hipLaunchKernelGGL(k_small_keys, dim3(1), dim3(kSmallThreads), 0, st, s->d_sph_in, n, s->d_keys[0],
                           s->d_vals[0], s->d_fcount + kOddWord);
    } else {
        hipLaunchKernelGGL(k_bounds_partial, dim3(nb), dim3(kBlk), 0, st, s->d_sph_in, n, nullptr, partial);
        hipLaunchKernelGGL(k_bounds_final, dim3(1), dim3(kBlk), 0, st, partial, nb, 0u, fin);
        hipLaunchKernelGGL(k_bounds_partial, dim3(nb), dim3(kBlk), 0, st, s->d_sph_in, n, fin, partial);
        hipLaunchKernelGGL(k_bounds_final, dim3(1), dim3(kBlk), 0, st, partial, nb, 1u, grid_b);
        hipLaunchKernelGGL(k_morton, dim3(blocks_for(n, kBlk)), dim3(kBlk), 0, st, s->d_sph_in, n, fin, grid_b,
                           s->d_keys[0], s->d_vals[0], s->d_fcount + kOddWord);
    }
    s->builder = (n >= 2 && n <= kSahMaxPrims) ? VZ_BUILD_SAH : VZ_BUILD_LBVH;
    // keys and leaf order end in buffers 0 either way
    s->d_morton = s->d_keys[0];
    s->d_leaf_prim = s->d_vals[0];
    if (s->builder == VZ_BUILD_SAH) {
        hipLaunchKernelGGL(k_sah_build, dim3(1), dim3(64 * kSahSoloWaves), 0, st, s->d_sph_in, n, s->d_leaf_prim,
                           s->d_morton, s->d_child, s->d_parent_int, s->d_parent_leaf);
    } else {
        uint32_t tiles = s->hist_blocks;
        uint32_t* dtot = s->d_hist + 256 * tiles;
        for (int pass = 0; pass < 4; pass++) {  // four passes: the result is back in buffers 0
            int src = pass & 1, dst = src ^ 1;
            hipLaunchKernelGGL(k_radix_hist, dim3(tiles), dim3(kBlk), 0, st, s->d_keys[src], n, pass * 8,
                               tiles, s->d_hist);
            hipLaunchKernelGGL(k_scan_rows, dim3(256), dim3(kBlk), 0, st, s->d_hist, tiles, dtot);
            hipLaunchKernelGGL(k_radix_scatter, dim3(tiles), dim3(kBlk), 0, st, s->d_keys[src],
                               s->d_vals[src], n, pass * 8, tiles, s->d_hist, dtot, s->d_keys[dst], s->d_vals[dst]);
        }
        if (n >= 2) {
            // node leaf ranges go to the wide-children buffer, which the collapse rewrites later
            uint2* range = reinterpret_cast<uint2*>(s->d_wkids);
            hipLaunchKernelGGL(k_karras, dim3(blocks_for(n - 1, kBlk)), dim3(kBlk), 0, st, s->d_morton, n,
                               s->d_child, s->d_parent_int, s->d_parent_leaf, s->d_visit, range);
            if (n >= kTreeletMinPrims) {
                // the treelet list uses the node-box buffer, which the refit fills afterwards
                uint4* list = reinterpret_cast<uint4*>(s->d_boxes);
                uint32_t* count = s->d_fcount + 8;
                hipLaunchKernelGGL(k_zero, dim3(1), dim3(kBlk), 0, st, count, 1u);
                hipLaunchKernelGGL(k_treelet_roots, dim3(blocks_for(n - 1, kBlk)), dim3(kBlk), 0, st, range,
                                   s->d_parent_int, n - 1, list, count);
                hipLaunchKernelGGL(k_sah_treelets, dim3(kTreeletBlocks), dim3(64 * kSahWaves), 0, st, s->d_sph_in,
                                   list, count, s->d_leaf_prim, s->d_morton, s->d_child, s->d_parent_int,
                                   s->d_parent_leaf);
            }
        }
    }
    hipLaunchKernelGGL(k_reorder, dim3(blocks_for(n, kBlk)), dim3(kBlk), 0, st, s->d_sph_in,
                       s->d_mat_in, s->d_leaf_prim, n, s->d_sph, s->d_leaf_info, s->d_mat, s->d_fcount + kOddWord);
    VZ_HIP_TRY(hipGetLastError());
    vzStatus rs = refit_core(s, st);
    VZ_HIP_TRY(hipEventRecord(e1.e, st));
    VZ_HIP_TRY(hipEventSynchronize(e1.e));
    float ms = 0.0f;
    VZ_HIP_TRY(hipEventElapsedTime(&ms, e0.e, e1.e));
    s->build_ms = ms;
    if (n < 2) {
        s->depth = 1;
        s->nw = 0;
        s->wdepth = 1;
    }
    return rs;
}

vzStatus lbvh_check_input(vzScene s, const vzMaterial* mat, hipStream_t st, uint32_t* bad_sphere,
                          uint32_t* bad_material)
{
    uint32_t* first = s->d_fcount + 2;  // words 2-3 of the refit counter block
    uint32_t h[2] = {0u, 0u};
    hipLaunchKernelGGL(k_fill, dim3(1), dim3(kBlk), 0, st, first, 2u, 0xFFFFFFFFu);
    const uint32_t nb = std::min<uint32_t>(1024u, blocks_for(s->n, kBlk));
    hipLaunchKernelGGL(k_check_input, dim3(nb), dim3(kBlk), 0, st, s->d_sph_in, mat, s->n, first);
    VZ_HIP_TRY(hipGetLastError());
    VZ_HIP_TRY(hipMemcpyAsync(h, first, sizeof(h), hipMemcpyDeviceToHost, st));
    VZ_HIP_TRY(hipStreamSynchronize(st));
    *bad_sphere = h[0];
    *bad_material = h[1];
    return VZ_SUCCESS;
}

vzStatus lbvh_refit(vzScene s, hipStream_t st)
{
    uint32_t n = s->n;
    Event e0, e1;
    VZ_EVENT_TRY(e0);
    VZ_EVENT_TRY(e1);
    VZ_HIP_TRY(hipEventRecord(e0.e, st));
    hipLaunchKernelGGL(k_reorder_sph, dim3(blocks_for(n, kBlk)), dim3(kBlk), 0, st, s->d_sph_in,
                       s->d_leaf_prim, n, s->d_sph);
    VZ_HIP_TRY(hipGetLastError());
    vzStatus rs = refit_core(s, st);
    VZ_HIP_TRY(hipEventRecord(e1.e, st));
    VZ_HIP_TRY(hipEventSynchronize(e1.e));
    float ms = 0.0f;
    VZ_HIP_TRY(hipEventElapsedTime(&ms, e0.e, e1.e));
    s->build_ms = ms;
    return rs;
}

}  // namespace vz
