// vz_traverse_mem.h -- closest-hit traversal of a scene too large for LDS by
// the kernels that do not count node visits (vz_traverse.h holds the one that
// does; hits are the same).
//
// It reads the scene's 48-byte nodes (k_wide_pack, vz_lbvh.hip): three
// 16-byte loads a visit, one index for all internal children and one for all
// leaves of a node.  A wave's 64 rays read mostly different nodes, nearly
// every visit misses the 32 KB L1, and the L1 takes about one line per cycle:
// with the 64-byte nodes it was busy 77% of the cycles in a frame of a million
// spheres, the VALU (two thirds of a visit are conversions, min, max and
// selects, 4 cycles each) most of the rest.  Children hit are put in order by
// five min/max pairs on their entry distances, whose four lowest bits hold the
// child's place (cut, so never beyond the distance), with leaf and missed
// slots above any distance.  Million spheres at 1080p and 64 samples 181 ->
// 162 ms.
//
// LDS decides the waves that hide the loads' latency: a stack entry is a node
// and the upper 16 bits of its distance, a queued visit's leaves are one index
// and a mask of four.  12 entries and 3 visits are 87 bytes a lane, 28 waves
// on a CU, and hardly an entry goes to private memory: the same frame 162 ms
// with 8 entries of 8 bytes and 24 waves, 193 with 4, 148 with 14 of 6 bytes
// and 24 waves, 143 with 12 and 28, 146 with 10 and 32 waves (64 registers).
#pragma once
#include "vz_traverse.h"

namespace vz {

constexpr uint32_t kMemWaves = 7;       // waves per SIMD
constexpr uint32_t kMemThreads = 256;   // a wave per SIMD and workgroup, so that any number of them fits evenly
constexpr uint32_t kMemStack = 12;      // stack entries per lane in LDS, later ones in private memory
constexpr uint32_t kMemPend = 3;        // queued visits per lane

// LDS of a workgroup of NT threads, [wave][slot][lane].
template <uint32_t NT>
struct MemScene {
    uint32_t node[NT / 64][kMemStack][64];
    uint32_t leaf[NT / 64][kMemPend][64];
    uint16_t dist[NT / 64][kMemStack][64];
    uint8_t mask[NT / 64][kMemPend][64];
};

// Stack entries beyond those in LDS.  Nodes are numbered in units of 16
// bytes: 3 times their index.
struct MemOverflow {
    uint2 e[kWideOverflow];
};

// ANYT: tmin may be negative or NaN.  Entries then hold distances from zero
// up and none is dropped for its distance while the best hit lies behind the
// origin.  Scene: node_array() (null for a single sphere), sphere_array(),
// info_array().
template <uint32_t NT, bool ANYT = false>
struct MemTraversal {
    static constexpr uint32_t kMiss = 0xFFFFFFFFu;
    v3 o, d;
    float inv[3];
    float tmin, best;
    uint32_t bleaf, node, sp, npend;

    // Returns true when there is nothing to walk: a single sphere, queued.
    template <class Scene>
    VZ_DEV bool begin(const Scene& sc, MemScene<NT>& sh, v3 o_, v3 d_, float tmin_, float tmax_)
    {
        o = o_;
        d = d_;
        tmin = tmin_;
        best = tmax_;
        bleaf = kMiss;
        node = sp = npend = 0u;
        if (sc.node_array() != nullptr) return false;
        queue(sh, 0u, 1u);
        return true;
    }

    // What follows from the ray: after begin(), and wherever it is cheaper than
    // keeping it (k_path).
    VZ_DEV void derive() { ray_inverse(d, inv); }

    // Tests the queued leaves; keeps the lexicographic minimum of (t, prim).
    template <class Scene>
    VZ_DEV void flush(const Scene& sc, const MemScene<NT>& sh)
    {
        const uint32_t w = threadIdx.x / 64, l = threadIdx.x % 64;
        uint32_t m = 0u, leaf0 = 0u;
        while (m | npend) {
            if (m == 0u) {
                npend--;
                m = sh.mask[w][npend][l];
                leaf0 = sh.leaf[w][npend][l];
            }
            const uint32_t leaf = leaf0 + (uint32_t)__builtin_ctz(m);
            m &= m - 1u;
            float t;
            if (hit_gated(o, d, inv, tmin, best, ldg(sc.sphere_array() + leaf), t))
                keep_nearer(t, leaf, sc.info_array(), best, bleaf);
        }
    }

    // One node visit; returns true when the traversal has finished.  Leaf
    // slots that are hit are queued, an entry a visit (the caller flushes
    // before the queue could overflow, and before it reads the hit).
    template <class Scene>
    VZ_DEV bool step(const Scene& sc, MemScene<NT>& sh, MemOverflow& ov)
    {
        const uint4* q = sc.node_array() + node;
        const uint4 A = ldg(q), B = ldg(q + 1), C = ldg(q + 2);
        const float no[3] = {__uint_as_float(A.x), __uint_as_float(A.y), __uint_as_float(A.z)};
        const float org[3] = {o.x, o.y, o.z};
        const uint32_t lo_w[3] = {B.x, B.y, B.z}, hi_w[3] = {B.w, C.x, C.y};
        const uint32_t n_in = A.w >> 24;
        // Slab distances of the planes s*q + no (q a plane byte) as one fma
        // per plane, fma(q, s*inv, (no - o)*inv), moved outwards by e = (255 s
        // + |no| + |no - o|) |inv| 2^-19 + 2^-126.  The exact-form distance
        // fl(fl(fl(s*q + no) - o) * inv) differs from the unmoved fma value by
        // less than 10 u (255 s + |no| + |no - o|) |inv| (u = 2^-24, e = 32 u
        // of it) and kRobust adds at most 16 u of it: every near distance here
        // is <= the exact form's and every far distance >= the exact form's
        // times kRobust, so the test passes whenever the sphere gate's does.
        float a[3], bn[3], bf[3];
        uint32_t qn[3], qf[3];
#pragma unroll
        for (int k = 0; k < 3; k++) {
            const float s = scale_of(A.w, k);
            const float dd = no[k] - org[k];
            const float w = __builtin_fmaf(255.0f, s, fabsf(no[k])) + fabsf(dd);
            const float e = __builtin_fmaf(w, fabsf(inv[k]), 0x1p-107f), b = dd * inv[k];
            a[k] = s * inv[k];
            bn[k] = __builtin_fmaf(e, -0x1p-19f, b);
            bf[k] = __builtin_fmaf(e, 0x1p-19f, b);
            // the near planes are the lo planes for a positive direction
            const bool ng = inv[k] < 0.0f;
            qn[k] = ng ? hi_w[k] : lo_w[k];
            qf[k] = ng ? lo_w[k] : hi_w[k];
        }
        const float lim = best * kRobust;
        uint32_t key[4];
        bool hit[4];
#pragma unroll
        for (uint32_t c = 0; c < 4; c++) {
            float n3[3], f3[3];
#pragma unroll
            for (int k = 0; k < 3; k++) {
                n3[k] = __builtin_fmaf((float)((qn[k] >> (8 * c)) & 0xFFu), a[k], bn[k]);
                f3[k] = __builtin_fmaf((float)((qf[k] >> (8 * c)) & 0xFFu), a[k], bf[k]);
            }
            const float lo_t = fmaxf(fmaxf(fmaxf(tmin, n3[0]), n3[1]), n3[2]);
            const float hi_t = fminf(fminf(fminf(lim, f3[0]), f3[1]), f3[2]);
            hit[c] = lo_t <= hi_t;
            const uint32_t e = (__float_as_uint(ANYT ? fmaxf(lo_t, 0.0f) : lo_t) & ~15u) | 3u * c;
            key[c] = hit[c] && c < n_in ? e : kMiss;
        }
        uint32_t leaves = hit[3] ? 1u : 0u;
        leaves = leaves + leaves + (hit[2] ? 1u : 0u);  // an add with carry each
        leaves = leaves + leaves + (hit[1] ? 1u : 0u);
        leaves = leaves + leaves + (hit[0] ? 1u : 0u);
        leaves >>= n_in;  // internal children come first
        if (leaves) queue(sh, C.w, leaves);
        // ascending by five compare-exchanges
        auto order = [](uint32_t& x, uint32_t& y) {
            const uint32_t lo = min(x, y), hi = max(x, y);
            x = lo;
            y = hi;
        };
        order(key[0], key[1]);
        order(key[2], key[3]);
        order(key[0], key[2]);
        order(key[1], key[3]);
        order(key[1], key[2]);
        if (key[0] != kMiss) {
            if (key[1] != kMiss) {
                if (sp <= (kMemStack - 3u) * kRow) {  // room in LDS for three
                    if (key[2] != kMiss) {
                        if (key[3] != kMiss) push(sh, C.z, key[3]);
                        push(sh, C.z, key[2]);
                    }
                    push(sh, C.z, key[1]);
                } else {
                    for (int c = 3; c >= 1; c--)
                        if (key[c] != kMiss) {
                            if (sp < kMemStack * kRow) {
                                push(sh, C.z, key[c]);
                            } else {
                                // never more than it holds (kMaxWideDepth)
                                const uint32_t i = sp / kRow - kMemStack;
                                if (i < kWideOverflow) ov.e[i] = make_uint2(C.z + (key[c] & 15u), key[c] & ~15u);
                                sp += kRow;
                            }
                        }
                }
            }
            node = C.z + (key[0] & 15u);
            return false;
        }
        // the nearest stacked child that can still hold a closer hit
        for (;;) {
            if (sp == 0u) return true;
            sp -= kRow;
            float t;
            if (sp < kMemStack * kRow) {
                node = *node_at(sh, sp);
                t = __uint_as_float((uint32_t)*dist_at(sh, sp) << 16);
            } else {
                const uint32_t i = min(sp / kRow - kMemStack, kWideOverflow - 1u);
                node = ov.e[i].x;
                t = __uint_as_float(ov.e[i].y);
            }
            if (t <= (ANYT ? fmaxf(lim, 0.0f) : lim)) return false;
        }
    }

private:
    // sp counts bytes of a row of distances (a wave's, 2 bytes a lane)
    static constexpr uint32_t kRow = 128;
    static VZ_DEV uint32_t* node_at(MemScene<NT>& sh, uint32_t at)
    {
        return reinterpret_cast<uint32_t*>(reinterpret_cast<char*>(&sh.node[threadIdx.x / 64][0][threadIdx.x % 64]) +
                                           2u * at);
    }
    static VZ_DEV uint16_t* dist_at(MemScene<NT>& sh, uint32_t at)
    {
        return reinterpret_cast<uint16_t*>(reinterpret_cast<char*>(&sh.dist[threadIdx.x / 64][0][threadIdx.x % 64]) +
                                           at);
    }
    VZ_DEV void push(MemScene<NT>& sh, uint32_t base, uint32_t key)
    {
        *node_at(sh, sp) = base + (key & 15u);
        *dist_at(sh, sp) = (uint16_t)(key >> 16);
        sp += kRow;
    }
    VZ_DEV void queue(MemScene<NT>& sh, uint32_t leaf0, uint32_t m)
    {
        sh.leaf[threadIdx.x / 64][npend][threadIdx.x % 64] = leaf0;
        sh.mask[threadIdx.x / 64][npend][threadIdx.x % 64] = (uint8_t)m;
        npend++;
    }
};

}  // namespace vz
