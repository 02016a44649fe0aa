// vz_traverse_lds.h -- closest-hit traversal of a small scene whose 4-wide
// nodes a workgroup has staged in LDS (vz_traverse.h holds the traversal of
// nodes in memory; hits are the same, node visits are not counted here).
//
// The nodes are staged decoded: the slots' planes as floats, so that a slot
// costs one fma and one min or max per plane, without the conversions and the
// per-node scales of the packed form.  The rounding bound that makes the box
// test accept whatever the sphere gate accepts is per ray: planes are at most
// Pmax away from the origin, which the root box gives.
//
// Measured against the packed nodes in LDS (64 bytes, decoded at every
// visit, sphere tests at once, children ranked pair by pair): the 1080p book
// frame at 256 samples 78.1 -> 61.1 ms, VALU instructions 3.37e10 -> 2.49e10 a
// launch of 128 passes.  The spheres are staged too (60.7 -> 59.1 ms with one
// set-up for camera and scattered rays): a queued test otherwise waits for the
// L1.  78 KB of LDS per 768 threads keep two workgroups, 24 waves, on a CU.
//
// They come from the 48-byte nodes (k_wide_pack, vz_lbvh.hip), whose internal
// children come first in the slots and whose leaves follow one another, with
// the leaves in that order.  Node, 112 bytes at a byte offset that is also its
// number:
//   0   float lo[4], hi[4] of the slots on x;  32 on y;  64 on z
//       (an empty slot: lo = +inf, hi = -inf)
//   96  uint32 per slot: the child node's offset, or 0xFFFF << 16 for a leaf
//       or an empty slot.  Slot 3's low 4 bits are the number of internal
//       children, and if that is below 4 the next 12 the first leaf.
// An empty slot stands for a leaf further on, which a ray whose terms overflow,
// and which passes every slot, tests without harm.
//
// A stack entry, and the key by which the children hit are put in order (five
// min/max pairs), is one word: the entry distance's upper 16 bits (cut, so
// never beyond the distance) and the child's offset; leaf and missed slots lie
// above any distance.  A visit's leaves are queued as one word, the first leaf
// and a mask of four.  With the child's offset behind another LDS load, a
// queue entry per leaf and a ring of 8 entries whose room each push checked:
// 1080p book frame at 256 samples 62.3 ms instead of 59.3.
#pragma once
#include "vz_traverse.h"

namespace vz {

constexpr uint32_t kLdsNodes = 256;        // a scene of at most this many 4-wide nodes is staged
constexpr uint32_t kLdsSpheres = 3 * kLdsNodes + 1;  // leaves of so many 4-wide nodes, at most
constexpr uint32_t kLdsNodeBytes = 112;
constexpr uint32_t kLdsKeyMask = 0xFFFF0000u;
constexpr uint32_t kLdsStack = 10;  // stack words per lane in LDS, later ones in private memory
constexpr uint32_t kLdsPend = 4;    // queued visits per lane

// LDS of a workgroup of NT threads, [wave][slot][lane].
template <uint32_t NT>
struct LdsScene {
    uint4 nodes[kLdsNodes * kLdsNodeBytes / 16];
    float4 spheres[kLdsSpheres + 3];
    uint32_t stack[NT / 64][kLdsStack][64];
    uint16_t pend[NT / 64][kLdsPend][64];
};

// Copies the spheres into LDS and decodes the 48-byte nodes, whole workgroup.
template <uint32_t NT>
VZ_DEV void stage_scene(const SceneView& sc, LdsScene<NT>& sh)
{
    for (uint32_t i = threadIdx.x; i < sc.n + 3u; i += NT) sh.spheres[i] = ldg(sc.tspheres + i);
    for (uint32_t i = threadIdx.x; i < sc.nw; i += NT) {
        const uint4 A = ldg(sc.tnodes + 3 * i), B = ldg(sc.tnodes + 3 * i + 1), C = ldg(sc.tnodes + 3 * i + 2);
        const float no[3] = {__uint_as_float(A.x), __uint_as_float(A.y), __uint_as_float(A.z)};
        const uint32_t lo_w[3] = {B.x, B.y, B.z}, hi_w[3] = {B.w, C.x, C.y}, n_in = A.w >> 24;
        uint4* out = sh.nodes + i * (kLdsNodeBytes / 16);
#pragma unroll
        for (int k = 0; k < 3; k++) {
            const float s = scale_of(A.w, k);
            uint32_t lo[4], hi[4];
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const uint32_t ql = (lo_w[k] >> (8 * c)) & 0xFFu, qh = (hi_w[k] >> (8 * c)) & 0xFFu;
                const bool v = ql <= qh;
                lo[c] = __float_as_uint(v ? __builtin_fmaf((float)ql, s, no[k]) : __builtin_huge_valf());
                hi[c] = __float_as_uint(v ? __builtin_fmaf((float)qh, s, no[k]) : -__builtin_huge_valf());
            }
            out[2 * k] = make_uint4(lo[0], lo[1], lo[2], lo[3]);
            out[2 * k + 1] = make_uint4(hi[0], hi[1], hi[2], hi[3]);
        }
        uint32_t w[4];
#pragma unroll
        for (uint32_t c = 0; c < 4; c++)
            w[c] = c < n_in ? (C.z / 3u + c) * kLdsNodeBytes : kLdsKeyMask;
        w[3] |= n_in < 4u ? n_in | C.w << 4 : 4u;
        out[6] = make_uint4(w[0], w[1], w[2], w[3]);
    }
}

// 2^-20 of the largest |plane| of a scene on each axis, at least 2^-70 (|1/d|
// of an ordinary ray is above 2^-41, so that its bound stays a normal number).
struct PlaneBound {
    float p[3];
    VZ_DEV explicit PlaneBound(const SceneView& sc)
    {
        const v3 m = plane_bounds(sc);
        p[0] = fmaxf(0x1p-20f * m.x, 0x1p-70f);
        p[1] = fmaxf(0x1p-20f * m.y, 0x1p-70f);
        p[2] = fmaxf(0x1p-20f * m.z, 0x1p-70f);
    }
};

// Stack words beyond the LDS ones, oldest first.
struct LdsOverflow {
    uint32_t w[kWideOverflow];
};

// ANYT: tmin may be negative or NaN.  Entries then hold distances from zero
// up and none is dropped for its distance while the best hit lies behind the
// origin.
template <uint32_t NT, bool ANYT = false>
struct LdsTraversal {
    v3 o, d;
    float inv[3], bn[3], bf[3];
    uint32_t off[3];   // 16 where the ray runs towards -k: its near planes are the hi planes
    float tmin, best;
    uint32_t bleaf, node, sp, npend;

    VZ_DEV void begin(v3 o_, v3 d_, float tmin_, float tmax_)
    {
        o = o_;
        d = d_;
        tmin = tmin_;
        best = tmax_;
        bleaf = 0xFFFFFFFFu;
        node = sp = npend = 0u;
    }

    // What follows from the ray: after begin(), and wherever it is cheaper than
    // keeping it (k_path).
    // Plane distances are fma(p, inv, -o inv), near ones moved down by e and
    // far ones up by 2 e, e = (Pmax + |o|) |inv| 2^-20.  The exact form
    // fl(fl(p - o) inv) and the unmoved fma differ by less than 5.2 u (Pmax +
    // |o|) |inv| (u = 2^-24, e = 16 u of it), so near distances are at most
    // the exact form's and far ones at least the exact form's times kRobust
    // (16 u more): the test passes whenever the sphere gate's does.  An
    // overflow of a term leaves an infinity or a NaN that min and max drop:
    // the slot passes.
    VZ_DEV void derive(const PlaneBound& pb)
    {
        const bool ordinary = ray_inverse(d, inv);
        const float oo[3] = {o.x, o.y, o.z};
#pragma unroll
        for (int k = 0; k < 3; k++) {
            off[k] = inv[k] < 0.0f ? 16u : 0u;
            const float m = oo[k] * inv[k];
            const float e = __builtin_fmaf(fabsf(oo[k]), 0x1p-20f, pb.p[k]) * fabsf(inv[k]);
            bn[k] = -m - e;
            bf[k] = __builtin_fmaf(2.0f, e, -m);
        }
        if (!ordinary)  // a bound that may underflow
            for (int k = 0; k < 3; k++) {
                bn[k] -= 0x1p-126f;
                bf[k] += 0x1p-125f;
            }
    }

    // Tests the queued leaves; keeps the lexicographic minimum of (t, prim).
    VZ_DEV void flush(const SceneArrays& sc, const LdsScene<NT>& sh)
    {
        uint32_t m = 0u, leaf0 = 0u;
        while (m | npend) {
            if (m == 0u) {
                npend--;
                m = sh.pend[threadIdx.x / 64][npend][threadIdx.x % 64];
                leaf0 = m >> 4;
                m &= 15u;
            }
            const uint32_t leaf = leaf0 + (uint32_t)__builtin_ctz(m);
            m &= m - 1u;
            float t;
            if (hit_gated(o, d, inv, tmin, best, sh.spheres[leaf], t)) keep_nearer(t, leaf, sc.info, best, bleaf);
        }
    }

    // One node visit; returns true when the traversal has finished.  Leaf
    // slots that are hit are queued, an entry a visit (the caller flushes
    // before the queue could overflow, and before it reads the hit).
    VZ_DEV bool step(LdsScene<NT>& sh, LdsOverflow& ov)
    {
        const char* base = reinterpret_cast<const char*>(sh.nodes);
        float4 nr[3], fr[3];
#pragma unroll
        for (int k = 0; k < 3; k++) {
            nr[k] = *reinterpret_cast<const float4*>(base + (node + off[k]) + 32 * k);
            fr[k] = *reinterpret_cast<const float4*>(base + ((node + 16u) - off[k]) + 32 * k);
        }
        const uint4 w4 = *reinterpret_cast<const uint4*>(base + node + 96);
        const float lim = best * kRobust;
        const uint32_t w[4] = {w4.x, w4.y, w4.z, w4.w};
        uint32_t key[4];
        bool hit[4];
#pragma unroll
        for (int c = 0; c < 4; c++) {
            float n3[3], f3[3];
#pragma unroll
            for (int k = 0; k < 3; k++) {
                const float pn = c == 0 ? nr[k].x : (c == 1 ? nr[k].y : (c == 2 ? nr[k].z : nr[k].w));
                const float pf = c == 0 ? fr[k].x : (c == 1 ? fr[k].y : (c == 2 ? fr[k].z : fr[k].w));
                n3[k] = __builtin_fmaf(pn, inv[k], bn[k]);
                f3[k] = __builtin_fmaf(pf, inv[k], bf[k]);
            }
            const float lo_t = fmaxf(fmaxf(fmaxf(tmin, n3[0]), n3[1]), n3[2]);
            const float hi_t = fminf(fminf(fminf(lim, f3[0]), f3[1]), f3[2]);
            hit[c] = lo_t <= hi_t;
            const uint32_t e = (__float_as_uint(ANYT ? fmaxf(lo_t, 0.0f) : lo_t) & kLdsKeyMask) | w[c];
            key[c] = hit[c] ? e : 0xFFFFFFFFu;
        }
        uint32_t leaves = hit[0] ? 1u : 0u;
        leaves |= hit[1] ? 2u : 0u;
        leaves |= hit[2] ? 4u : 0u;
        leaves |= hit[3] ? 8u : 0u;
        leaves >>= w[3] & 7u;  // internal children come first
        if (leaves) {
            sh.pend[threadIdx.x / 64][npend][threadIdx.x % 64] = (uint16_t)((w[3] & 0xFFF0u) | leaves);
            npend++;
        }
        // ascending by five compare-exchanges
        auto order = [](uint32_t& a, uint32_t& b) {
            const uint32_t x = min(a, b), y = max(a, b);
            a = x;
            b = y;
        };
        order(key[0], key[1]);
        order(key[2], key[3]);
        order(key[0], key[2]);
        order(key[1], key[3]);
        order(key[1], key[2]);
        if (key[0] < kLdsKeyMask) {
            if (key[1] < kLdsKeyMask) {
                if (sp <= (kLdsStack - 3u) * kRow) {  // room in LDS for three
                    if (key[2] < kLdsKeyMask) {
                        if (key[3] < kLdsKeyMask) push(sh, key[3]);
                        push(sh, key[2]);
                    }
                    push(sh, key[1]);
                } else {
                    for (int c = 3; c >= 1; c--)
                        if (key[c] < kLdsKeyMask) {
                            if (sp < kLdsStack * kRow) {
                                push(sh, key[c]);
                            } else {
                                // never more than it holds (kMaxWideDepth)
                                const uint32_t i = sp / kRow - kLdsStack;
                                if (i < kWideOverflow) ov.w[i] = key[c];
                                sp += kRow;
                            }
                        }
                }
            }
            node = key[0] & 0xFFF0u;
            return false;
        }
        // the nearest stacked child that can still hold a closer hit
        for (;;) {
            if (sp == 0u) return true;
            sp -= kRow;
            uint32_t e;
            if (sp < kLdsStack * kRow) {
                e = *slot(sh, sp);
                // kept apart from the other load: the two become one flat load
                // otherwise, and every pop waits for the memory pipe (1080p
                // book frame 55.6 ms against 56.2)
                asm volatile("" : "+v"(e));
            } else {
                e = ov.w[min(sp / kRow - kLdsStack, kWideOverflow - 1u)];
            }
            node = e & 0xFFF0u;
            if (__uint_as_float(e & kLdsKeyMask) <= (ANYT ? fmaxf(lim, 0.0f) : lim)) return false;
        }
    }

private:
    static constexpr uint32_t kRow = 256;  // sp counts bytes of a row of the stack, a word a lane
    static VZ_DEV uint32_t* slot(LdsScene<NT>& sh, uint32_t at)
    {
        return reinterpret_cast<uint32_t*>(reinterpret_cast<char*>(&sh.stack[threadIdx.x / 64][0][threadIdx.x % 64]) +
                                           at);
    }
    VZ_DEV void push(LdsScene<NT>& sh, uint32_t e)
    {
        *slot(sh, sp) = e;
        sp += kRow;
    }
};

}  // namespace vz
