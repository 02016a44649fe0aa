// vz_traverse_mem.h -- closest-hit traversal of a scene too large for LDS by
// the kernels that do not count node visits (vz_traverse.h holds the one that
// does; hits are the same).
//
// It reads the scene's 48-byte nodes (k_wide_pack, vz_lbvh.hip): three
// 16-byte loads a visit, one index for all internal children and one for all
// leaves of a node.  A wave's 64 rays read mostly different nodes, and the L1
// takes about one line per cycle, so the loads bound a visit as much as the
// VALU does: with the 64-byte nodes the L1 was busy 77% of the cycles in a
// frame of a million spheres.  Children hit are put in order by five min/max
// pairs on their entry distances, whose four lowest bits hold the child's
// place (cut, so never beyond the distance), with leaf and missed slots above
// any distance.  A stack entry is (node, distance) in LDS, [slot][lane], the
// oldest beyond kWideStackS of them in private memory.  Sphere tests are
// queued and run when many lanes of the wave hold some.
#pragma once
#include "vz_traverse.h"

namespace vz {

// LDS of a workgroup of NT threads.
template <uint32_t NT>
struct MemScene {
    uint2 stack[kWideStackS * NT];
    uint32_t pend[kPend * NT];
};

// Nodes are numbered in units of 16 bytes: 3 times their index.
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
    uint32_t bleaf, node, sp, bottom, npend;

    // Returns true when there is nothing to walk: a single sphere, queued.
    template <class Scene>
    VZ_DEV bool init(const Scene& sc, MemScene<NT>& sh, v3 o_, v3 d_, float tmin_, float tmax_)
    {
        o = o_;
        d = d_;
        tmin = tmin_;
        best = tmax_;
        bleaf = kMiss;
        node = sp = bottom = npend = 0u;
        ray_inverse(d, inv);
        if (sc.node_array() != nullptr) return false;
        sh.pend[threadIdx.x] = 0u;
        npend = 1u;
        return true;
    }

    // Tests the queued leaves; keeps the lexicographic minimum of (t, prim).
    template <class Scene>
    VZ_DEV void flush(const Scene& sc, const MemScene<NT>& sh)
    {
        while (npend) {
            npend--;
            const uint32_t leaf = sh.pend[npend * NT + threadIdx.x];
            float t;
            if (hit_gated(o, d, inv, tmin, best, ldg(sc.sphere_array() + leaf), t))
                keep_nearer(t, leaf, sc.info_array(), best, bleaf);
        }
    }

    // One node visit; returns true when the traversal has finished.  Leaf
    // slots that are hit are queued (at most 4; the caller flushes before
    // the queue could overflow, and before it reads the hit).
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
        bool leaf[4];
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
            const bool hit = lo_t <= hi_t, in = c < n_in;
            leaf[c] = hit && !in;
            key[c] = hit && in ? (__float_as_uint(ANYT ? fmaxf(lo_t, 0.0f) : lo_t) & ~15u) | 3u * c : kMiss;
        }
        const uint32_t leaf0 = C.w - n_in;
#pragma unroll
        for (uint32_t c = 0; c < 4; c++)
            if (leaf[c]) {
                sh.pend[npend * NT + threadIdx.x] = leaf0 + c;
                npend++;
            }
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
                // room in LDS for three: the oldest go to the overflow (never
                // more than it holds: kMaxWideDepth)
                while (sp + 3u - bottom > kWideStackS) {
                    if (bottom < kWideOverflow) ov.e[bottom] = sh.stack[(bottom % kWideStackS) * NT + threadIdx.x];
                    bottom++;
                }
                if (key[2] != kMiss) {
                    if (key[3] != kMiss) push(sh, C.z, key[3]);
                    push(sh, C.z, key[2]);
                }
                push(sh, C.z, key[1]);
            }
            node = C.z + (key[0] & 15u);
            return false;
        }
        // the nearest stacked child that can still hold a closer hit
        for (;;) {
            if (sp == 0u) return true;
            sp--;
            uint2 e;
            if (sp < bottom) {
                e = ov.e[sp < kWideOverflow ? sp : kWideOverflow - 1u];
                bottom = sp;
            } else {
                e = sh.stack[(sp % kWideStackS) * NT + threadIdx.x];
            }
            node = e.x;
            if (__uint_as_float(e.y) <= (ANYT ? fmaxf(lim, 0.0f) : lim)) return false;
        }
    }

private:
    VZ_DEV void push(MemScene<NT>& sh, uint32_t base, uint32_t key)
    {
        sh.stack[(sp % kWideStackS) * NT + threadIdx.x] = make_uint2(base + (key & 15u), key & ~15u);
        sp++;
    }
};

}  // namespace vz
