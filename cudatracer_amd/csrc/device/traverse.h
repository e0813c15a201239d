// Ray traversal on gfx950.
//
// Exact mode keeps the reference's arithmetic, node order and culling so the
// closest-hit primitive ids are bit-exact, ties included:
//   quad tree   MBVHNode::intersect / traverseMBVH[Shadow], src/BVH/MBVHNode.cuh:69-205
//   binary tree BVHNode::Intersect / traverseBVH[Shadow],   src/BVH/BVHNode.cuh:50-204
//   triangle    triangle::intersect,                        src/Core/Triangle.cuh:13-44
// Empty quad slots (count 0, always "hit" in the reference) are not pushed:
// popping them is a no-op, so the visit order of real nodes is unchanged.
//
// Execution shape (what changes is only how a wave64 interleaves its lanes;
// every lane performs the reference's sequence of pops, node tests, pushes
// and triangle tests for its own ray):
//   - persistent waves claim rays for their idle lanes with one atomic once
//     kRefillIdle of them are idle, from queue ranges of their XCD (see
//     Fetcher); neither the claim nor the new rays' loads are waited for on
//     their own;
//   - one step per loop iteration and lane, a node test or one triangle of
//     the current leaf, with one memory round trip for both kinds (trav_step);
//   - once a wave has at most 16 rays and no more come, each ray gets the four
//     lanes of a quad (trace_quads);
//   - the per-lane stack lives in LDS, laid out [depth][thread]; pushes are
//     branch-free stores at the stack top (a store for a culled child is
//     overwritten by the next one); entries beyond the LDS depth spill to
//     the block's global region, laid out the same way.  The builder's depth
//     limit (64) bounds the stack at 97 entries; the stack bound
//     (Queues::max_stack, 128 by default) guards user-supplied trees.
// 1,048,576 rays against 524,287 triangles: 0.641 ms per call with two round
// trips per step, waited-for claims and one lane a ray throughout, 0.497 ms
// as it is; the 1080p atrium frame 3.87 and 3.50 ms.
#pragma once

#include "dev_common.h"

extern __shared__ uint32_t ct_lds_stack[];

namespace ctd {

CT_DEV uint32_t fbits(float f) { return __float_as_uint(f); }
CT_DEV uint32_t lane_id() { return __lane_id(); }

// Optional per-lane work counters: node and triangle tests of closest-hit
// rays, and of any-hit rays.
struct TravCount {
    uint32_t nodes, tris, snodes, stris;
};

// Moller-Trumbore with precomputed edges (edge1 = p1 - p0 and edge2 = p2 - p0
// are computed on the host with the same float subtraction).
CT_DEV bool tri_test(f3 o, f3 d, float& t, f3 p0, f3 edge1, f3 edge2, float eps) {
    const f3 h = cross(d, edge2);
    const float a = dot(edge1, h);
    if (a > -eps && a < eps) return false;
    const float f = 1.0f / a;
    const f3 s = o - p0;
    const float u = f * dot(s, h);
    if (u < 0.0f || u > 1.0f) return false;
    const f3 q = cross(s, edge1);
    const float v = f * dot(d, q);
    if (v < 0.0f || u + v > 1.0f) return false;
    const float tt = f * dot(edge2, q);
    if (tt > eps && t > tt) {
        t = tt;
        return true;
    }
    return false;
}

CT_DEV float tag(float v, uint32_t slot) { return __uint_as_float((fbits(v) & 0xFFFFFFFCu) | slot); }

// Per-lane stack: LDS positions [0, depth), global spill [depth, max_stack).
// Both are laid out [position][thread]: position p of thread i is at byte
// 4 * (p * blockDim + i) of the LDS stack or, spilled, at byte
// 4 * ((p - depth) * blockDim + i) of the block's spill region.  The stack is
// held as `top`, the LDS byte offset of the next free position, so a push or
// a pop is an add and the depth checks compare with uniform limits.  The
// spill region is addressed through a raw buffer resource (vector buffer
// loads/stores, bounds-checked by the hardware), which also keeps the
// compiler from folding LDS and spill reads into one flat access.
struct LaneStack {
    uint32_t top;      // p * stride4 + 4 * threadIdx.x for the next free position p
    uint32_t stride4;  // 4 * blockDim.x
    uint32_t lds_end;  // depth * stride4: positions from here on are spilled
    uint32_t max_end;  // max_stack * stride4
    __amdgpu_buffer_rsrc_t spill;  // this block's spill region
    bool overflow;

    CT_DEV static uint32_t& lds(uint32_t byte) {
        return *reinterpret_cast<uint32_t*>(reinterpret_cast<char*>(ct_lds_stack) + byte);
    }
    CT_DEV void reset() {
        top = 4u * threadIdx.x;
        overflow = false;
    }
    CT_DEV bool empty() const { return top < stride4; }
    // Store at byte a: LDS, spill region, or dropped beyond max_stack (push4
    // flags the overflow).
    CT_DEV void put(uint32_t a, uint32_t v) {
        if (a < lds_end) lds(a) = v;
        else if (a < max_end) __builtin_amdgcn_raw_buffer_store_b32(v, spill, a - lds_end, 0, 0);
    }
    CT_DEV uint32_t top_pop() {
        top -= stride4;
        // LDS read at a clamped offset (always in bounds), buffer read only
        // for spilled entries
        uint32_t v = lds(top < lds_end ? top : lds_end - 4u);
        if (top >= lds_end) {
            v = __builtin_amdgcn_raw_buffer_load_b32(spill, top - lds_end, 0, 0);
            // waited for here, not at the join: every pop would wait for
            // whatever memory operations are in flight
            __asm__ volatile("" : "+v"(v));
        }
        return v;
    }
    // Push v0..v3 where k0..k3 (in that order), all but the last of them: that
    // one would be popped next, so it stays in `next`.  Every value but v3 is
    // stored at the next free position; a culled one is overwritten by the
    // next store or left above the new top.  Branch-free when all positions
    // are in LDS.  False if there is nothing to push.  The bound counts the
    // kept entry as if it were stored.
    CT_DEV bool push4(uint32_t v0, bool k0, uint32_t v1, bool k1, uint32_t v2, bool k2, uint32_t v3, bool k3,
                      uint32_t& next) {
        if (!(k0 || k1 || k2 || k3)) return false;
        const uint32_t a0 = top, a1 = a0 + (k0 ? stride4 : 0u), a2 = a1 + (k1 ? stride4 : 0u),
                       a3 = a2 + (k2 ? stride4 : 0u);
        const uint32_t end = a3 + (k3 ? stride4 : 0u);
        next = k3 ? v3 : (k2 ? v2 : (k1 ? v1 : v0));
        top = end - stride4;
        if (a2 < lds_end) {
            lds(a0) = v0;
            lds(a1) = v1;
            lds(a2) = v2;
        } else {
            put(a0, v0);
            put(a1, v1);
            put(a2, v2);
        }
        // a position at or beyond max_stack was needed
        if (end >= max_end + stride4) overflow = true;
        return true;
    }
    // Push v, if at all, under an entry that is kept in a register and counts
    // as if it were stored on top.
    CT_DEV void push_under(uint32_t v, bool keep) {
        const uint32_t end = top + (keep ? stride4 : 0u);
        if (top < lds_end) lds(top) = v;  // left above the new top if not kept
        else if (keep) put(top, v);
        top = end;
        if (end >= max_end) overflow = true;
    }
    // Push v0..v3 where k0..k3, all of them.
    CT_DEV void push4_all(uint32_t v0, bool k0, uint32_t v1, bool k1, uint32_t v2, bool k2, uint32_t v3, bool k3) {
        const uint32_t a0 = top, a1 = a0 + (k0 ? stride4 : 0u), a2 = a1 + (k1 ? stride4 : 0u),
                       a3 = a2 + (k2 ? stride4 : 0u);
        top = a3 + (k3 ? stride4 : 0u);
        put(a0, v0);
        put(a1, v1);
        put(a2, v2);
        put(a3, v3);
        if (top >= max_end + stride4) {
            overflow = true;
            top = max_end + 4u * threadIdx.x;
        }
    }
};

// Push the hit children of a quad node, sorted by the tagged tmin (nearest
// popped first) with the reference's 5-comparator network.
CT_DEV bool push_children(uint32_t hm, float m0, float m1, float m2, float m3, uint32_t e0, uint32_t e1,
                          uint32_t e2, uint32_t e3, LaneStack& st, uint32_t& next) {
    if (hm == 0u) return false;
    float s0 = m0, s1 = m1, s2 = m2, s3 = m3, tmp;
    if (s0 > s1) { tmp = s0; s0 = s1; s1 = tmp; }
    if (s2 > s3) { tmp = s2; s2 = s3; s3 = tmp; }
    if (s0 > s2) { tmp = s0; s0 = s2; s2 = tmp; }
    if (s1 > s3) { tmp = s1; s1 = s3; s3 = tmp; }
    if (s2 > s3) { tmp = s2; s2 = s3; s3 = tmp; }
    auto entry = [&](uint32_t slot) { return slot == 0 ? e0 : (slot == 1 ? e1 : (slot == 2 ? e2 : e3)); };
    const uint32_t q3 = fbits(s3) & 3u, q2 = fbits(s2) & 3u, q1 = fbits(s1) & 3u, q0 = fbits(s0) & 3u;
    return st.push4(entry(q3), (hm >> q3) & 1u, entry(q2), (hm >> q2) & 1u, entry(q1), (hm >> q1) & 1u, entry(q0),
                    (hm >> q0) & 1u, next);
}

// The entry of an empty slot, and of a culled child in the sort.
constexpr uint32_t kNoEntry = 0xFFFFFFFFu;

// Quad node test (MBVHNode::intersect) on a node's rows in nodes4f: four slabs in the reference's float
// order, tmin tagged with the slot, the 5-comparator network, then pushes in
// the order of traverseMBVH and traverseMBVHShadow (sorted position 3 first).
CT_DEV bool node4_step(const float4 (&n)[7], f3 o, f3 inv, float t, LaneStack& st, uint32_t& next) {
    const float4 bminx = n[0], bmaxx = n[1], bminy = n[2], bmaxy = n[3], bminz = n[4], bmaxz = n[5];
    const float4 ent = n[6];
    float m0, m1, m2, m3, x0, x1, x2, x3;
#define CT_SLAB(MN, MX, lo, hi)                                                 \
    {                                                                           \
        float t1 = (bminx.lo - o.x) * inv.x, t2 = (bmaxx.lo - o.x) * inv.x;     \
        float mn = gmin(t1, t2), mx = gmax(t1, t2);                             \
        t1 = (bminy.lo - o.y) * inv.y;                                          \
        t2 = (bmaxy.lo - o.y) * inv.y;                                          \
        mn = gmax(mn, gmin(t1, t2));                                            \
        mx = gmin(mx, gmax(t1, t2));                                            \
        t1 = (bminz.lo - o.z) * inv.z;                                          \
        t2 = (bmaxz.lo - o.z) * inv.z;                                          \
        mn = gmax(mn, gmin(t1, t2));                                            \
        mx = gmin(mx, gmax(t1, t2));                                            \
        MN = tag(mn, hi);                                                       \
        MX = mx;                                                                \
    }
    CT_SLAB(m0, x0, x, 0u)
    CT_SLAB(m1, x1, y, 1u)
    CT_SLAB(m2, x2, z, 2u)
    CT_SLAB(m3, x3, w, 3u)
#undef CT_SLAB
    const uint32_t e0 = fbits(ent.x), e1 = fbits(ent.y), e2 = fbits(ent.z), e3 = fbits(ent.w);
    // hit mask on the tagged values; empty slots never pushed
    const uint32_t hm = ((x0 > 0.0f && m0 <= x0 && m0 < t && e0 != kNoEntry) ? 1u : 0u) |
                        ((x1 > 0.0f && m1 <= x1 && m1 < t && e1 != kNoEntry) ? 2u : 0u) |
                        ((x2 > 0.0f && m2 <= x2 && m2 < t && e2 != kNoEntry) ? 4u : 0u) |
                        ((x3 > 0.0f && m3 <= x3 && m3 < t && e3 != kNoEntry) ? 8u : 0u);
    return push_children(hm, m0, m1, m2, m3, e0, e1, e2, e3, st, next);
}

// Fast quad node test: the same tagged entry distances, hit flags and push
// order as node4_step, from the hardware min/max instructions (one v_min or
// v_max per slab pair, v_min3/v_max3 across axes) instead of the
// compare-and-select that (y < x) ? y : x costs.  That is exact under
// conditions that fast_ray() checks once per ray and this function once per
// node:
//  - inv is finite with |inv| > 0.5 and o is finite, so no slab value
//    (plane - o) * inv is NaN (planes are finite, see plane_flags), and a
//    slab value is zero only when plane - o is: a non-zero difference times
//    |inv| > 0.5 stays above half the smallest denormal;
//  - plane - o is never -0 (o has no +0 component, or no plane is -0), so
//    every zero slab value is +0 * inv, of the sign of inv on its axis;
//  - inside a slab pair (one axis) equal values therefore have equal bits,
//    and v_min / v_max return what (y < x) ? y : x and (x < y) ? y : x
//    return;
//  - across axes only zeros of opposite sign can tie.  For the exit distance
//    that does not matter (a zero fails x > 0 in either sign); where an
//    entry distance is zero (the origin on a face of the box) the four entry
//    distances are recomputed with the reference's fold, which keeps the
//    zero of the first axis (exact slab pairs, then (x < y) ? y : x);
//  - no key is NaN, so the reference network's last comparator (2,3) never
//    swaps: after (0,2) and (1,3), s2 = max(s0, s2) <= max(s1, s3) = s3.  The
//    entries ride through the first four comparators instead of being looked
//    up from the sorted keys' slot tags.
CT_DEV bool fast_ray(f3 o, f3 inv, uint32_t plane_flags) {
    constexpr float kMax = 3.40282347e38f;
    const bool inv_ok = fabsf(inv.x) > 0.5f && fabsf(inv.x) <= kMax && fabsf(inv.y) > 0.5f &&
                        fabsf(inv.y) <= kMax && fabsf(inv.z) > 0.5f && fabsf(inv.z) <= kMax;
    const bool o_ok = fabsf(o.x) <= kMax && fabsf(o.y) <= kMax && fabsf(o.z) <= kMax;
    const bool z_ok = !(plane_flags & kPlaneNegZero) || (fbits(o.x) != 0u && fbits(o.y) != 0u && fbits(o.z) != 0u);
    return !(plane_flags & kPlaneNaN) && inv_ok && o_ok && z_ok;
}

// nodes4f: the tree in the fast layout (k_prepare_quad): six plane rows and
// the four stack entries, seven loads per node.
CT_DEV bool node4_fast(const float4* __restrict__ nodes4f, uint32_t e, const float4 (&n)[7], f3 o, f3 inv, float t,
                       LaneStack& st, uint32_t& next) {
    const float4 bminx = n[0], bmaxx = n[1], bminy = n[2], bmaxy = n[3], bminz = n[4], bmaxz = n[5];
    const float4 ent = n[6];
    float m0, m1, m2, m3, x0, x1, x2, x3;
#define CT_SLABF(MN, MX, lo)                                                      \
    {                                                                             \
        const float ax = (bminx.lo - o.x) * inv.x, bx = (bmaxx.lo - o.x) * inv.x; \
        const float ay = (bminy.lo - o.y) * inv.y, by = (bmaxy.lo - o.y) * inv.y; \
        const float az = (bminz.lo - o.z) * inv.z, bz = (bmaxz.lo - o.z) * inv.z; \
        MN = fmaxf(fmaxf(fminf(ax, bx), fminf(ay, by)), fminf(az, bz));           \
        MX = fminf(fminf(fmaxf(ax, bx), fmaxf(ay, by)), fmaxf(az, bz));           \
    }
    CT_SLABF(m0, x0, x)
    CT_SLABF(m1, x1, y)
    CT_SLABF(m2, x2, z)
    CT_SLABF(m3, x3, w)
#undef CT_SLABF
    // keep the exit distances in this block: sunk past the branch below they
    // would hold all 24 slab values live (and be re-canonicalised there)
    __asm__ volatile("" ::"v"(x0), "v"(x1), "v"(x2), "v"(x3));
    if (fminf(fminf(fabsf(m0), fabsf(m1)), fminf(fabsf(m2), fabsf(m3))) == 0.0f) {
        // rare: the planes are reloaded (an opaque index) one child at a time
        // rather than held live beside everything else
        uint32_t r = e;
        __asm__ volatile("" : "+v"(r));
        const float* p = reinterpret_cast<const float*>(nodes4f + 8 * (size_t)r);
#pragma unroll 1
        for (uint32_t i = 0; i < 4; ++i) {
            const float v = gmax(gmax(fminf((p[i] - o.x) * inv.x, (p[4 + i] - o.x) * inv.x),
                                      fminf((p[8 + i] - o.y) * inv.y, (p[12 + i] - o.y) * inv.y)),
                                 fminf((p[16 + i] - o.z) * inv.z, (p[20 + i] - o.z) * inv.z));
            m0 = i == 0 ? v : m0;
            m1 = i == 1 ? v : m1;
            m2 = i == 2 ? v : m2;
            m3 = i == 3 ? v : m3;
        }
    }
    m0 = tag(m0, 0u);
    m1 = tag(m1, 1u);
    m2 = tag(m2, 2u);
    m3 = tag(m3, 3u);
    // An empty slot's entry is kNoEntry, so the count test is the entry test:
    // the sorted path carries kNoEntry through the network and never pushes
    // it.
    const uint32_t e0 = fbits(ent.x), e1 = fbits(ent.y), e2 = fbits(ent.z), e3 = fbits(ent.w);
    const bool h0 = x0 > 0.0f && m0 <= x0 && m0 < t;
    const bool h1 = x1 > 0.0f && m1 <= x1 && m1 < t;
    const bool h2 = x2 > 0.0f && m2 <= x2 && m2 < t;
    const bool h3 = x3 > 0.0f && m3 <= x3 && m3 < t;
    if (!(h0 || h1 || h2 || h3)) return false;
    // comparators (0,1) and (2,3) on keys and entries, then (0,2) and (1,3)
    // on entries (their keys are not compared again)
    uint32_t q0 = h0 ? e0 : kNoEntry, q1 = h1 ? e1 : kNoEntry, q2 = h2 ? e2 : kNoEntry, q3 = h3 ? e3 : kNoEntry;
    const bool s01 = m0 > m1, s23 = m2 > m3;
    const float a = s01 ? m1 : m0, b = s01 ? m0 : m1, c = s23 ? m3 : m2, d = s23 ? m2 : m3;
    const uint32_t ea = s01 ? q1 : q0, eb = s01 ? q0 : q1, ec = s23 ? q3 : q2, ed = s23 ? q2 : q3;
    const bool s02 = a > c, s13 = b > d;
    q0 = s02 ? ec : ea;
    q2 = s02 ? ea : ec;
    q1 = s13 ? ed : eb;
    q3 = s13 ? eb : ed;
    return st.push4(q3, q3 != kNoEntry, q2, q2 != kNoEntry, q1, q1 != kNoEntry, q0, q0 != kNoEntry, next);
}

// The compact quad tree (ACCEL kTreeCompact): node i of the quad tree in 16
// words (64 bytes, half a cache line, against the 112 bytes node4_fast
// reads), written by k_prepare_quad:
//   0..2    p.x, p.y, p.z: the node's grid corner (float bits)
//   3       biased exponents of the x, y, z grid steps 2^k (bytes 0..2)
//   4, 5    low and high x offsets of slots 0..3 (byte i = slot i)
//   6, 7    low and high y offsets;  8, 9  low and high z offsets
//   10, 11  zero
//   12..15  the four stack entries (kNoEntry for an empty slot)
// A child's box is [p + lo 2^k, p + hi 2^k] per axis, quantised outwards, so
// it contains the quad node's box (why no further margin is needed:
// compact_axis in device/kernels.hip).  The ray moves into the node's grid once per node,
// t = q (2^k / d) + (p - o) / d: one conversion and one fma per plane, with
// the hardware min/max (no slab value is NaN for a compact_ray).  Entry
// distances carry the slot tag and go through node4_fast's network, so the
// children are visited nearest first, in the exact traversal's order except
// where the quantised distances order two children differently.
constexpr int kTreeCompact = 5;

// Rays the compact node test takes: finite origin, |1/d| <= 2^64 (so
// 2^k / d stays finite for the steps k <= kCompactMaxExp the encoder allows).
// The others use node4_step on the same tree.
constexpr int kCompactMaxExp = 60;
CT_DEV bool compact_ray(f3 o, f3 inv) {
    constexpr float kMax = 3.40282347e38f, kInvMax = 18446744073709551616.0f;  // 2^64
    return fabsf(inv.x) <= kInvMax && fabsf(inv.y) <= kInvMax && fabsf(inv.z) <= kInvMax && fabsf(o.x) <= kMax &&
           fabsf(o.y) <= kMax && fabsf(o.z) <= kMax;
}

CT_DEV uint4 ubits4(float4 v) { return make_uint4(fbits(v.x), fbits(v.y), fbits(v.z), fbits(v.w)); }

CT_DEV bool cnode4_step(const float4 (&n)[7], f3 o, f3 inv, float t, LaneStack& st, uint32_t& next) {
    const uint4 h = ubits4(n[0]), qa = ubits4(n[1]), qb = ubits4(n[2]), ent = ubits4(n[3]);
    const float ax = __uint_as_float((h.w & 0xFFu) << 23) * inv.x;
    const float ay = __uint_as_float(((h.w >> 8) & 0xFFu) << 23) * inv.y;
    const float az = __uint_as_float(((h.w >> 16) & 0xFFu) << 23) * inv.z;
    const float bx = (__uint_as_float(h.x) - o.x) * inv.x, by = (__uint_as_float(h.y) - o.y) * inv.y,
                bz = (__uint_as_float(h.z) - o.z) * inv.z;
    float m0, m1, m2, m3, x0, x1, x2, x3;
#define CT_CSLAB(MN, MX, SH)                                                                              \
    {                                                                                                     \
        const float lx = fmaf((float)((qa.x >> SH) & 0xFFu), ax, bx), hx = fmaf((float)((qa.y >> SH) & 0xFFu), ax, bx); \
        const float ly = fmaf((float)((qa.z >> SH) & 0xFFu), ay, by), hy = fmaf((float)((qa.w >> SH) & 0xFFu), ay, by); \
        const float lz = fmaf((float)((qb.x >> SH) & 0xFFu), az, bz), hz = fmaf((float)((qb.y >> SH) & 0xFFu), az, bz); \
        MN = fmaxf(fmaxf(fminf(lx, hx), fminf(ly, hy)), fminf(lz, hz));                                  \
        MX = fminf(fminf(fmaxf(lx, hx), fmaxf(ly, hy)), fmaxf(lz, hz));                                  \
    }
    CT_CSLAB(m0, x0, 0u)
    CT_CSLAB(m1, x1, 8u)
    CT_CSLAB(m2, x2, 16u)
    CT_CSLAB(m3, x3, 24u)
#undef CT_CSLAB
    m0 = tag(m0, 0u);
    m1 = tag(m1, 1u);
    m2 = tag(m2, 2u);
    m3 = tag(m3, 3u);
    const bool h0 = x0 > 0.0f && m0 <= x0 && m0 < t;
    const bool h1 = x1 > 0.0f && m1 <= x1 && m1 < t;
    const bool h2 = x2 > 0.0f && m2 <= x2 && m2 < t;
    const bool h3 = x3 > 0.0f && m3 <= x3 && m3 < t;
    if (!(h0 || h1 || h2 || h3)) return false;
    uint32_t q0 = h0 ? ent.x : kNoEntry, q1 = h1 ? ent.y : kNoEntry, q2 = h2 ? ent.z : kNoEntry,
             q3 = h3 ? ent.w : kNoEntry;
    const bool s01 = m0 > m1, s23 = m2 > m3;
    const float a = s01 ? m1 : m0, b = s01 ? m0 : m1, c = s23 ? m3 : m2, d = s23 ? m2 : m3;
    const uint32_t ea = s01 ? q1 : q0, eb = s01 ? q0 : q1, ec = s23 ? q3 : q2, ed = s23 ? q2 : q3;
    const bool s02 = a > c, s13 = b > d;
    q0 = s02 ? ec : ea;
    q2 = s02 ? ea : ec;
    q1 = s13 ? ed : eb;
    q3 = s13 ? eb : ed;
    return st.push4(q3, q3 != kNoEntry, q2, q2 != kNoEntry, q1, q1 != kNoEntry, q0, q0 != kNoEntry, next);
}

// Wide compressed node (128 B, up to 8 children, layout in host/cnode.h).
// The ray is moved into the node's grid once per node, t = q * (s / d) +
// (p - o) / d, so each child plane costs one conversion and one fma (the
// decoded boxes contain the exact ones by a grid step, which covers the
// rounding of this form).  The nearest hit child is visited first, the others
// in slot order: a full sort of 8 measured slower.  sort = false (any-hit)
// goes in slot order.
//
// Bound by its instructions and, at eight waves a SIMD, by registers: with
// finite slab terms (then no slab value is NaN) the tests use the hardware
// minimum and maximum, 8 instructions a child where compare-and-select takes
// 20, with the same comparisons' results (they do not see a zero's sign).  The
// general test, for terms that are not finite, is a loop, since a second unrolled
// copy would cost the registers again; the seven entries below the nearest are
// stored in sequence, without 19 registers spilled for values and flags.
// Atrium 1080p 6.57 to 4.82 ms, 7.24M triangles at 4K 13.1 to 9.0 ms, 1,048,576
// rays 1.01 to 0.71 ms.
//
// A ray parallel to an axis has no 1 / d there (its terms would be infinity minus
// infinity, and a NaN in x culls every child): ray_inv.
CT_DEV bool fnode8_step(bool sort, const float4 (&n)[7], f3 o, f3 inv, float t, LaneStack& st, uint32_t& next) {
    const uint4 h = ubits4(n[0]), qx = ubits4(n[1]), qy = ubits4(n[2]), qz = ubits4(n[3]), ca = ubits4(n[4]),
                cb = ubits4(n[5]);
    const float sx = __uint_as_float((h.w & 0xFFu) << 23), sy = __uint_as_float(((h.w >> 8) & 0xFFu) << 23),
                sz = __uint_as_float(((h.w >> 16) & 0xFFu) << 23);
    // the ray in the node's grid: t = q * (s / d) + (p - o) / d
    const float ax = sx * inv.x, ay = sy * inv.y, az = sz * inv.z;
    const float bx = (__uint_as_float(h.x) - o.x) * inv.x, by = (__uint_as_float(h.y) - o.y) * inv.y,
                bz = (__uint_as_float(h.z) - o.z) * inv.z;
    const uint32_t valid = h.w >> 24;
    uint32_t hm = 0, bslot = 0;
    float best = 3.0e38f;
    if (fabsf(ax) + fabsf(ay) + fabsf(az) + fabsf(bx) + fabsf(by) + fabsf(bz) <= 3.40282347e38f) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const uint32_t sh = 8u * (uint32_t)(i & 3);
            const uint32_t lxw = i < 4 ? qx.x : qx.y, hxw = i < 4 ? qx.z : qx.w;
            const uint32_t lyw = i < 4 ? qy.x : qy.y, hyw = i < 4 ? qy.z : qy.w;
            const uint32_t lzw = i < 4 ? qz.x : qz.y, hzw = i < 4 ? qz.z : qz.w;
            const float lx = fmaf((float)((lxw >> sh) & 0xFFu), ax, bx), hx = fmaf((float)((hxw >> sh) & 0xFFu), ax, bx);
            const float ly = fmaf((float)((lyw >> sh) & 0xFFu), ay, by), hy = fmaf((float)((hyw >> sh) & 0xFFu), ay, by);
            const float lz = fmaf((float)((lzw >> sh) & 0xFFu), az, bz), hz = fmaf((float)((hzw >> sh) & 0xFFu), az, bz);
            const float mn = fmaxf(fmaxf(fminf(lx, hx), fminf(ly, hy)), fminf(lz, hz));
            const float mx = fminf(fminf(fmaxf(lx, hx), fmaxf(ly, hy)), fmaxf(lz, hz));
            const bool hit = ((valid >> i) & 1u) && mx > 0.0f && mn <= mx && mn < t;
            hm |= hit ? (1u << i) : 0u;
            if (hit && mn < best) { best = mn; bslot = (uint32_t)i; }
        }
    } else {
#pragma unroll 1
        for (uint32_t i = 0; i < 8; ++i) {
            const uint32_t sh = 8u * (i & 3u);
            const uint32_t lxw = i < 4 ? qx.x : qx.y, hxw = i < 4 ? qx.z : qx.w;
            const uint32_t lyw = i < 4 ? qy.x : qy.y, hyw = i < 4 ? qy.z : qy.w;
            const uint32_t lzw = i < 4 ? qz.x : qz.y, hzw = i < 4 ? qz.z : qz.w;
            float t1 = fmaf((float)((lxw >> sh) & 0xFFu), ax, bx), t2 = fmaf((float)((hxw >> sh) & 0xFFu), ax, bx);
            float mn = gmin(t1, t2), mx = gmax(t1, t2);
            t1 = fmaf((float)((lyw >> sh) & 0xFFu), ay, by);
            t2 = fmaf((float)((hyw >> sh) & 0xFFu), ay, by);
            mn = gmax(mn, gmin(t1, t2));
            mx = gmin(mx, gmax(t1, t2));
            t1 = fmaf((float)((lzw >> sh) & 0xFFu), az, bz);
            t2 = fmaf((float)((hzw >> sh) & 0xFFu), az, bz);
            mn = gmax(mn, gmin(t1, t2));
            mx = gmin(mx, gmax(t1, t2));
            const bool hit = ((valid >> i) & 1u) && mx > 0.0f && mn <= mx && mn < t;
            hm |= hit ? (1u << i) : 0u;
            if (hit && mn < best) { best = mn; bslot = i; }
        }
    }
    if (hm == 0u) return false;
    const uint32_t ent[8] = {ca.x, ca.y, ca.z, ca.w, cb.x, cb.y, cb.z, cb.w};
    if (sort) {
        // nearest hit child on top; slot 7 takes the nearest child's place
        const uint32_t a0 = (bslot & 1u) ? ent[1] : ent[0], a1 = (bslot & 1u) ? ent[3] : ent[2];
        const uint32_t a2 = (bslot & 1u) ? ent[5] : ent[4], a3 = (bslot & 1u) ? ent[7] : ent[6];
        const uint32_t b0 = (bslot & 2u) ? a1 : a0, b1 = (bslot & 2u) ? a3 : a2;
        const uint32_t near = (bslot & 4u) ? b1 : b0;
        next = near;
        uint32_t a[8];
        a[0] = st.top;
#pragma unroll
        for (int i = 0; i < 7; ++i) {
            const uint32_t k = (uint32_t)i == bslot ? hm >> 7 : (hm >> i) & 1u;
            a[i + 1] = a[i] + (k ? st.stride4 : 0u);
        }
        if (a[6] < st.lds_end) {
#pragma unroll
            for (int i = 0; i < 7; ++i) st.lds(a[i]) = (uint32_t)i == bslot ? ent[7] : ent[i];
        } else {
#pragma unroll
            for (int i = 0; i < 7; ++i) st.put(a[i], (uint32_t)i == bslot ? ent[7] : ent[i]);
        }
        st.top = a[7];
        // the nearest child counts as if it were stored too
        if (a[7] >= st.max_end) st.overflow = true;
        return true;
    }
    st.push4_all(ent[0], hm & 1u, ent[1], (hm >> 1) & 1u, ent[2], (hm >> 2) & 1u, ent[3], (hm >> 3) & 1u);
    if (st.push4(ent[4], (hm >> 4) & 1u, ent[5], (hm >> 5) & 1u, ent[6], (hm >> 6) & 1u, ent[7], (hm >> 7) & 1u, next))
        return true;
    next = st.top_pop();
    return true;
}

// BVHNode::Intersect (BVHNode.cuh:50-62): no culling against the current t.
CT_DEV bool box2(float4 lo, float4 hi, f3 o, f3 inv, float& tmin) {
    const f3 t1 = (xyz(lo) - o) * inv;
    const f3 t2 = (xyz(hi) - o) * inv;
    const f3 mn = mk3(gmin(t1.x, t2.x), gmin(t1.y, t2.y), gmin(t1.z, t2.z));
    const f3 mx = mk3(gmax(t1.x, t2.x), gmax(t1.y, t2.y), gmax(t1.z, t2.z));
    tmin = gmax(mn.x, gmax(mn.y, mn.z));
    const float tmax = gmin(mx.x, gmin(mx.y, mx.z));
    return tmax >= 0.0f && tmin < tmax;
}

// The same test with the hardware minimum and maximum.  Without NaN they give
// box2's values up to the sign of a zero, which no comparison here sees, so a
// ray that finite_ray() accepts visits the same nodes in the same order.  Two
// boxes take 46 instructions instead of 70: the box's frame of 65,536 paths
// spends its time in chains of these steps.
CT_DEV bool box2_fast(float4 lo, float4 hi, f3 o, f3 inv, float& tmin) {
    const f3 t1 = (xyz(lo) - o) * inv;
    const f3 t2 = (xyz(hi) - o) * inv;
    tmin = fmaxf(fmaxf(fminf(t1.x, t2.x), fminf(t1.y, t2.y)), fminf(t1.z, t2.z));
    const float tmax = fminf(fminf(fmaxf(t1.x, t2.x), fmaxf(t1.y, t2.y)), fmaxf(t1.z, t2.z));
    return tmax >= 0.0f && tmin < tmax;
}
// No slab value (plane - o) * inv of the binary tree is NaN: planes (checked
// at upload) and origin are finite, and inv is neither infinite (0 * inf) nor
// zero (an overflown difference times 0).
CT_DEV bool finite_ray(f3 o, f3 inv, uint32_t plane_flags) {
    constexpr float kMax = 3.40282347e38f;
    auto ok = [](float v) { return fabsf(v) > 0.0f && fabsf(v) <= kMax; };
    return !(plane_flags & kPlaneInf2) && ok(inv.x) && ok(inv.y) && ok(inv.z) && fabsf(o.x) <= kMax &&
           fabsf(o.y) <= kMax && fabsf(o.z) <= kMax;
}

// The stack item of a binary node with rows {min, left_first}, {max, count}:
// the pair of an interior node's children, kLeafBit | first triangle record
// of a leaf, or kEmptyLeaf (count 0, only in user-supplied trees: pushed like
// any other, skipped when popped).
constexpr uint32_t kEmptyLeaf = 0xFFFFFFFEu;
CT_DEV uint32_t item2(float4 lo, float4 hi) {
    const uint32_t count = fbits(hi.w);
    return count == 0u ? kEmptyLeaf : fbits(lo.w) | (~count & kLeafBit);
}

// Binary interior step (traverseBVH, BVHNode.cuh:107-139): both children
// tested; if both hit, the strictly nearer is pushed first.  n: the rows of
// the two children, which are adjacent; reading what a child is from its own
// rows here makes a step one dependent load (fetching the popped node first
// and then its children was two).  Bound by instructions where rays are many:
// with a push of its own and no slab values canonicalised, 9% fewer vector
// instructions in a launch; 16 uneven views of the small box 66.6 to 64.7 ms,
// a frame of 65,536 paths 550 to 527 us.
CT_DEV bool node2_step(const float4 (&n)[7], f3 o, f3 inv, bool fast, LaneStack& st, uint32_t& next) {
    float n1, n2;
    bool hl, hr;
    if (fast) {
        hl = box2_fast(n[0], n[1], o, inv, n1);
        hr = box2_fast(n[2], n[3], o, inv, n2);
    } else {
        // an opaque copy of the origin: the slab values that both tests
        // compute would otherwise be hoisted above the branch, where the fast
        // test has to canonicalise them again
        f3 oo = o;
        __asm__ volatile("" : "+v"(oo.x), "+v"(oo.y), "+v"(oo.z));
        hl = box2(n[0], n[1], oo, inv, n1);
        hr = box2(n[2], n[3], oo, inv, n2);
    }
    if (!(hl || hr)) return false;
    const uint32_t l = item2(n[0], n[1]), r = item2(n[2], n[3]);
    const bool both = hl && hr, right = hr && (!hl || n1 < n2);
    next = right ? r : l;
    st.push_under(right ? l : r, both);
    return true;
}

// ----------------------------------------------------------------------
// Persistent traversal driver.  Source: how ray i is loaded; Sink: what is
// done with the result.  ACCEL 4 = quad tree, kTreeCompact = the quad tree
// in the compact layout, 8 = wide compressed tree, 2 = binary tree.
// A lane without a ray.
constexpr uint32_t kDead = 0xFFFFFFFFu;

// Raises the error flag, a word in pinned host memory: a plain store (every
// writer stores the same), which the host sees once the stream has finished.
CT_DEV void raise(uint32_t* err) { *reinterpret_cast<volatile uint32_t*>(err) = 1u; }

// What a launch traces: every ray closest-hit (extend, ray-level closest
// hit), every ray any-hit (ray-level shadow rays), or two queues at once, a
// closest-hit queue and an any-hit queue, each lane in the mode of the ray
// it holds (the frame loop's bounce b: the extension rays of bounce b and
// the shadow rays of bounce b - 1 in one launch, so neither launch's tail
// idles the machine).
enum TraceMode { kClosest = 0, kAny = 1, kDual = 2 };

// The queues [0, n) and [0, n2) are cut into kFetchRanges contiguous ranges
// each, four per XCD: workgroups are dispatched to the XCDs round-robin by
// block id, so the blocks b = x (mod 8) share XCD x's L2 and trace
// neighbouring rays of the ranges x, x + 8, x + 16 and x + 24 (range = block
// id mod 32).  Range r's claim counter counts through its rays of the first
// queue, then its rays of the second; each counter is on its own cache line:
// with all counters in one line the atomics of all XCDs serialised and
// throughput halved.  A range is drained only by its own blocks (moving
// waves to other ranges at the end measured slower); every range has blocks
// as long as the grid has at least kFetchRanges of them, smaller grids move
// on to the next ranges.
//
struct Fetcher {
    uint32_t* base;  // counter of range 0 (range r at base + r * kFetchSlot)
    uint32_t n, n2;  // rays of the first and the second queue
    int range, left;                    // the range, and how many more may be tried
    uint32_t lo, nfirst, lo2, total;    // its claim space

    // Index v < nfirst of a range's claim space [0, total) is ray lo + v of
    // the first queue, otherwise ray lo2 + v - nfirst of the second.
    CT_DEV void open() {
        lo = (uint32_t)(((uint64_t)n * (uint32_t)range) / kFetchRanges);
        const uint32_t hi = (uint32_t)(((uint64_t)n * (uint32_t)(range + 1)) / kFetchRanges);
        lo2 = (uint32_t)(((uint64_t)n2 * (uint32_t)range) / kFetchRanges);
        const uint32_t hi2 = (uint32_t)(((uint64_t)n2 * (uint32_t)(range + 1)) / kFetchRanges);
        nfirst = hi - lo;
        total = nfirst + (hi2 - lo2);
    }
    // Claim `want` indices; lane 0's result is the first.
    CT_DEV uint32_t claim(uint32_t want) const {
        // Only lane 0's is read (readfirstlane).  The others' is any value,
        // not an uninitialised one, and not a constant, which would wait for
        // the previous claim still in flight to this register.
        uint32_t got;
        __asm__ volatile("" : "=v"(got));
        if (lane_id() == 0) got = atomicAdd(base + range * kFetchSlot, want);
        return got;
    }
    // The range is drained: open the next one, false if there is none.
    CT_DEV bool next() {
        if (--left < 0) return false;
        range = (range + 1) % kFetchRanges;
        open();
        return true;
    }
};

// A 16-byte row through a pointer the compiler must know to be global memory
// (selected from two arrays, it would otherwise take the flat path).
using gptr = const __attribute__((address_space(1))) char*;
typedef float row4 __attribute__((ext_vector_type(4)));
CT_DEV float4 load_row(gptr p) {
    const row4 v = *(const __attribute__((address_space(1))) row4*)p;
    return make_float4(v.x, v.y, v.z, v.w);
}

// Node records of each tree: bytes apart, 16-byte rows read.
template <int ACCEL>
struct NodeFmt;
template <>
struct NodeFmt<4> {
    static constexpr int kStride = 128, kRows = 7;
    CT_DEV static const void* base(const DevScene& sc) { return sc.nodes4f; }
};
template <>
struct NodeFmt<2> {
    static constexpr int kStride = 32, kRows = 4;  // an item is a pair of nodes
    CT_DEV static const void* base(const DevScene& sc) { return sc.nodes2; }
};
template <>
struct NodeFmt<kTreeCompact> {
    static constexpr int kStride = 64, kRows = 4;
    CT_DEV static const void* base(const DevScene& sc) { return sc.cnodes; }
};
template <>
struct NodeFmt<8> {
    static constexpr int kStride = 128, kRows = 6;
    CT_DEV static const void* base(const DevScene& sc) { return sc.fnodes; }
};

// The triangle of leaf item cur with rows a, b, c.  Returns true when an
// any-hit ray is done; cur becomes the leaf's next triangle, or pop is set.
CT_DEV bool leaf_step(float4 a, float4 b, float4 c, float eps, f3 o, f3 d, bool any, uint32_t& cur, float& t, int& prim,
                      bool& pop) {
    const uint32_t w = fbits(a.w);
    bool done = false;
    if (tri_test(o, d, t, xyz(a), xyz(b), xyz(c), eps)) {
        prim = (int)(w & ~kLastInLeaf);
        done = any;
    }
    pop = (w & kLastInLeaf) != 0u;
    ++cur;
    return done;
}

// One step of a lane's ray: the node test or the triangle test of the item
// `cur` (a node, or kLeafBit | triangle record), which then becomes the next
// item.  Returns true when the ray is done: any hit found, stack empty or
// overflowed.
//
// What bounds the loop is the chain of dependent steps of a ray, each a round
// trip to memory (about 900 cycles) plus the instructions of the tests.  A
// wave holds lanes at nodes and lanes at triangles; testing the one kind and
// then the other, each after its own loads, costs a wave two round trips per
// step.  Here every lane loads the first three rows of whatever its item is
// from one selected address, and the node lanes' remaining rows follow before
// anything waits, so a step is one round trip.  The next item stays in a
// register when it is the nearest child just tested, instead of going through
// the LDS stack.
template <int ACCEL, bool COUNT>
CT_DEV bool trav_step(const DevScene& sc, float eps, f3 o, f3 d, f3 inv, bool fast, bool any, bool sort, uint32_t& cur,
                      float& t, int& prim, LaneStack& st, TravCount& cnt, const float4 (&n)[7], int kind) {
    bool pop = false, done = false;
    if (kind < 0) {
        if (COUNT) {
            if (any) ++cnt.stris;
            else ++cnt.tris;
        }
        done = leaf_step(n[0], n[1], n[2], eps, o, d, any, cur, t, prim, pop);
    } else {
        if (COUNT) {
            const uint32_t boxes = ACCEL == 2 ? 2u : 1u;
            if (any) cnt.snodes += boxes;
            else cnt.nodes += boxes;
        }
        // any-hit rays visit children nearest first too, like
        // traverseMBVHShadow (MBVHNode.cuh:165-205): in a two-queue launch
        // every lane then runs one code path (slot order for any-hit lanes
        // measured 2% slower)
        if constexpr (ACCEL == 4) {
            if (fast) {
                pop = !node4_fast(sc.nodes4f, (uint32_t)kind, n, o, inv, t, st, cur);
            } else {
                // an opaque copy of the origin: the slab values that both
                // tests compute would otherwise be hoisted above the branch,
                // 24 registers live through it
                f3 oo = o;
                __asm__ volatile("" : "+v"(oo.x), "+v"(oo.y), "+v"(oo.z));
                pop = !node4_step(n, oo, inv, t, st, cur);
            }
        } else if constexpr (ACCEL == kTreeCompact) {
            if (fast) {
                pop = !cnode4_step(n, o, inv, t, st, cur);
            } else {
                float4 full[7];
                for (int k = 0; k < 7; ++k) full[k] = sc.nodes4f[8 * (size_t)(uint32_t)kind + k];
                pop = !node4_step(full, o, inv, t, st, cur);
            }
        } else if constexpr (ACCEL == 8) {
            pop = !fnode8_step(sort, n, o, inv, t, st, cur);
        } else {
            pop = !node2_step(n, o, inv, fast, st, cur);
        }
    }
    if (pop) {
        if (st.empty()) done = true;
        else cur = st.top_pop();
    }
    if constexpr (ACCEL == 2) {
        while (!done && cur == kEmptyLeaf) {
            if (st.empty()) done = true;
            else cur = st.top_pop();
        }
    }
    return done || st.overflow;
}

// The loads of a step.  kind: the item, opaque to the compiler: otherwise the
// uses of the item's kind before and after the loads merge, and each kind
// gets its own loads and its own wait again.
template <int ACCEL>
CT_DEV void load_item(const DevScene& sc, uint32_t cur, float4 (&n)[7], int& kind) {
    using F = NodeFmt<ACCEL>;
    const bool leaf = (int)cur < 0;
    const gptr base = leaf ? (gptr)sc.tris : (gptr)F::base(sc);
    const gptr p = base + (uint64_t)(cur & ~kLeafBit) * (leaf ? 48u : (uint32_t)F::kStride);
#pragma unroll
    for (int k = 0; k < 3; ++k) n[k] = load_row(p + 16 * k);
    kind = (int)cur;
    __asm__ volatile("" : "+v"(kind));
    if (!leaf) {
#pragma unroll
        for (int k = 3; k < F::kRows; ++k) n[k] = load_row(p + 16 * k);
    }
    // One wait for all of them (vmcnt(0)).  Left to the compiler the rows of
    // whichever kind the wave skips count as in flight around the loop, and
    // the next step's loads wait for the last step's result stores.
    __builtin_amdgcn_s_waitcnt(0x0F70);
}

// Whether a ray takes its tree's fast node test.
template <int ACCEL>
CT_DEV bool ray_is_fast(const DevScene& sc, f3 o, f3 inv) {
    if constexpr (ACCEL == 4) return fast_ray(o, inv, sc.plane_flags);
    else if constexpr (ACCEL == kTreeCompact) return compact_ray(o, inv);
    else if constexpr (ACCEL == 2) return finite_ray(o, inv, sc.plane_flags);
    else return false;
}

// 1 / d as the tree's node test takes it.  The wide tree's gets a large finite K
// for an infinite one: a plane is a grid step s or more outside the box it was
// encoded from, so within the box t runs from below -s * K to above s * K, and
// outside the grid's box the range is empty.  K is a power of two, 2^120 over the
// largest coordinate in play (2^100 at most): every term stays finite, and s * K
// is further than any hit (5e23 for boxes 1e-4 wide at coordinates of 1e6).
// Decided per ray; per node it cost every launch ten spilled registers (1080p
// atrium 4.72 to 5.56 ms).
template <int ACCEL>
CT_DEV f3 ray_inv(const DevScene& sc, f3 o, f3 d) {
    f3 inv = mk3(1.0f / d.x, 1.0f / d.y, 1.0f / d.z);
    if constexpr (ACCEL == 8) {
        const float m = fmaxf(fmaxf(sc.wide_extent, fabsf(o.x)), fmaxf(fabsf(o.y), fabsf(o.z)));
        const float k = __uint_as_float(min(374u - (fbits(m) >> 23), 227u) << 23);
        auto finite = [&](float v) { return fabsf(v) > 3.40282347e38f ? copysignf(k, v) : v; };
        inv = mk3(finite(inv.x), finite(inv.y), finite(inv.z));
    }
    return inv;
}

// The item a ray starts at.
template <int ACCEL>
CT_DEV uint32_t root_item(const DevScene& sc) {
    return ACCEL == 2 ? sc.root2 : 0u;
}

// ------------------------------------------------------ four lanes a ray --
// Once a launch's rays are spread so thin that a wave has at most 16 of them
// (a small launch, or the last rays of a large one), what a ray waits for is
// its own chain of steps: some 300 instructions of one wave and a round trip
// to memory each, with most lanes idle.  trace_quads gives each ray the four
// lanes of a quad instead: lane c tests child c of a node (of a binary tree's
// two children, child c & 1), or triangle c of the next four of a leaf.  The quad makes the steps of the one-lane loop
// (the same entry distances in the reference's float order, the same
// comparators, pushes and visit order; the triangles of a leaf in order, the
// first of equal distances kept), so the results are the same bits.  1,000
// rays: 120 to 87 us per call; 1,048,576 rays, whose last ones took a third of
// the launch: 0.597 to 0.497 ms; the textured atrium 6.5 to 5.9 ms; a frame of
// 65,536 paths through the binary tree 0.93 to 0.75 ms.
template <int CTRL>
CT_DEV uint32_t quad_dpp(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, CTRL, 0xF, 0xF, true);
}
template <int CTRL>
CT_DEV float quad_dpp(float v) {
    return __uint_as_float(quad_dpp<CTRL>(fbits(v)));
}
constexpr int kQuadXor1 = 0xB1, kQuadXor2 = 0x4E;  // quad_perm [1,0,3,2] and [2,3,0,1]

// key with its sign flipped where `flip` is the sign bit: comparing flipped
// keys turns a pair's second lane's view of a comparison into the first's.
CT_DEV float flip_sign(float key, uint32_t flip) { return __uint_as_float(fbits(key) ^ flip); }

// One comparator of the network on lane pairs: swaps as the reference does,
// if the first lane's key is greater.  flip: 0 in a pair's first lane, the
// sign bit in its second.
template <int CTRL>
CT_DEV void quad_comparator(uint32_t flip, bool on, float& key, uint32_t& e) {
    const float ok = quad_dpp<CTRL>(key);
    const uint32_t oe = quad_dpp<CTRL>(e);
    const bool sw = (flip_sign(key, flip) > flip_sign(ok, flip)) & on;
    key = sw ? ok : key;
    e = sw ? oe : e;
}

// The quads' rays (all four lanes of a quad hold the same ray; cur == kDead:
// none), to their ends.  st.top: the ray's stack, in the column of one of the
// wave's lanes.  t and prim end as the ray's result (prim -1: none, -2: the
// stack bound was exceeded); lane 0 of the quad gives it to sink as well.
template <int ACCEL, class Sink>
CT_DEV void trace_quads(const DevScene& sc, float eps, f3 o, f3 d, f3 inv, bool fast, bool any, uint32_t ray,
                        uint32_t cur, float& t, int& prim, LaneStack& st, uint32_t* err, Sink sink) {
    const uint32_t c = lane_id() & 3u, qbase = lane_id() & 60u;
    const uint32_t flip1 = (c & 1u) << 31, flip2 = (c & 2u) << 30;
    while (__ballot(cur != kDead) != 0) {
        if (cur == kDead) continue;
        const uint32_t idx = cur & ~kLeafBit;
        // a triangle's rows; a binary child's rows; a quad child's six planes
        // (a, b.xy) and entry (e.z); or a compact node's grid (a), offsets
        // (b, e.xy) and the child's entry (e.z)
        float4 a, b, e;
        const bool packed = ACCEL == kTreeCompact && fast;
        if ((int)cur < 0) {
            // records past the leaf's end are read (within the array) and ignored
            const gptr p = (gptr)sc.tris + (uint64_t)min(idx + c, sc.n_tris - 1u) * 48u;
            a = load_row(p);
            b = load_row(p + 16);
            e = load_row(p + 32);
        } else if constexpr (ACCEL == 2) {
            // lanes 0 and 2 the left child, 1 and 3 the right
            const gptr p = (gptr)sc.nodes2 + (uint64_t)(idx + (c & 1u)) * 32u;
            a = load_row(p);
            b = load_row(p + 16);
        } else if (packed) {
            const uint4* n = sc.cnodes + 4 * (size_t)idx;
            a = *reinterpret_cast<const float4*>(n);
            b = *reinterpret_cast<const float4*>(n + 1);
            const float2 z = *reinterpret_cast<const float2*>(n + 2);
            e.x = z.x;
            e.y = z.y;
            e.z = reinterpret_cast<const float*>(n + 3)[c];
        } else {
            const float* n = reinterpret_cast<const float*>(sc.nodes4f) + 32 * (size_t)idx + c;
            a = make_float4(n[0], n[4], n[8], n[12]);
            b.x = n[16];
            b.y = n[20];
            e.z = n[24];
        }
        int kind = (int)cur;
        __asm__ volatile("" : "+v"(kind));
        __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0), see load_item
        bool done = false, pop = false;
        if (kind < 0) {
            const uint32_t w = fbits(a.w);
            const uint32_t last = (uint32_t)(__ballot((w & kLastInLeaf) != 0u) >> qbase) & 15u;
            float tt = t;
            const bool hit = tri_test(o, d, tt, xyz(a), xyz(b), xyz(e), eps) & ((last & ((1u << c) - 1u)) == 0u);
            tt = hit ? tt : t;
            uint32_t pp = hit ? (w & ~kLastInLeaf) : (uint32_t)prim;
            // the least distance, of equal ones the first triangle's
            const float t1 = quad_dpp<kQuadXor1>(tt);
            const uint32_t p1 = quad_dpp<kQuadXor1>(pp);
            const bool k1 = (t1 < tt) | ((t1 == tt) & ((c & 1u) != 0u));
            tt = k1 ? t1 : tt;
            pp = k1 ? p1 : pp;
            const float t2 = quad_dpp<kQuadXor2>(tt);
            const uint32_t p2 = quad_dpp<kQuadXor2>(pp);
            const bool k2 = (t2 < tt) | ((t2 == tt) & ((c & 2u) != 0u));
            tt = k2 ? t2 : tt;
            pp = k2 ? p2 : pp;
            done = any & (tt < t);
            t = tt;
            prim = (int)pp;
            pop = last != 0u;
            cur += 4u;
        } else if constexpr (ACCEL == 2) {
            float n1;
            bool h;
            if (fast) h = box2_fast(a, b, o, inv, n1);
            else h = box2(a, b, o, inv, n1);
            const uint32_t it = item2(a, b), oi = quad_dpp<kQuadXor1>(it);
            const float n2 = quad_dpp<kQuadXor1>(n1);
            const uint32_t hm = (uint32_t)(__ballot(h) >> qbase) & 3u;  // bit 0: left, bit 1: right
            const uint32_t il = flip1 ? oi : it, ir = flip1 ? it : oi;
            // both hit: the strictly nearer is pushed, the other is next
            const bool near_left = flip_sign(n1, flip1) < flip_sign(n2, flip1);
            pop = hm == 0u;
            if (hm == 3u) {
                if (c == 0u) st.put(st.top, near_left ? il : ir);
                st.top += st.stride4;
                cur = near_left ? ir : il;
            } else if (!pop) {
                cur = (hm & 1u) ? il : ir;
            }
            if (!pop && st.top >= st.max_end) st.overflow = true;
        } else {
            float mn, mx;
            const uint32_t ent = fbits(e.z);
            if (packed) {
                const uint4 ch = ubits4(a), cq = ubits4(b);
                const uint2 cz = make_uint2(fbits(e.x), fbits(e.y));
                const uint32_t sh = 8u * c;
                const float ax = __uint_as_float((ch.w & 0xFFu) << 23) * inv.x;
                const float ay = __uint_as_float(((ch.w >> 8) & 0xFFu) << 23) * inv.y;
                const float az = __uint_as_float(((ch.w >> 16) & 0xFFu) << 23) * inv.z;
                const float bx = (__uint_as_float(ch.x) - o.x) * inv.x, by = (__uint_as_float(ch.y) - o.y) * inv.y,
                            bz = (__uint_as_float(ch.z) - o.z) * inv.z;
                const float lx = fmaf((float)((cq.x >> sh) & 0xFFu), ax, bx), hx = fmaf((float)((cq.y >> sh) & 0xFFu), ax, bx);
                const float ly = fmaf((float)((cq.z >> sh) & 0xFFu), ay, by), hy = fmaf((float)((cq.w >> sh) & 0xFFu), ay, by);
                const float lz = fmaf((float)((cz.x >> sh) & 0xFFu), az, bz), hz = fmaf((float)((cz.y >> sh) & 0xFFu), az, bz);
                mn = fmaxf(fmaxf(fminf(lx, hx), fminf(ly, hy)), fminf(lz, hz));
                mx = fminf(fminf(fmaxf(lx, hx), fmaxf(ly, hy)), fmaxf(lz, hz));
            } else {
                const float ax = (a.x - o.x) * inv.x, bx = (a.y - o.x) * inv.x;
                const float ay = (a.z - o.y) * inv.y, by = (a.w - o.y) * inv.y;
                const float az = (b.x - o.z) * inv.z, bz = (b.y - o.z) * inv.z;
                if (ACCEL == 4 && fast) {
                    // node4_fast's arithmetic
                    const float nx = fminf(ax, bx), ny = fminf(ay, by), nz = fminf(az, bz);
                    mn = fmaxf(fmaxf(nx, ny), nz);
                    mx = fminf(fminf(fmaxf(ax, bx), fmaxf(ay, by)), fmaxf(az, bz));
                    if (mn == 0.0f) mn = gmax(gmax(nx, ny), nz);
                } else {
                    mn = gmax(gmax(gmin(ax, bx), gmin(ay, by)), gmin(az, bz));
                    mx = gmin(gmin(gmax(ax, bx), gmax(ay, by)), gmax(az, bz));
                }
            }
            float key = tag(mn, c);
            uint32_t x = ((mx > 0.0f) & (key <= mx) & (key < t)) ? ent : kNoEntry;
            quad_comparator<kQuadXor1>(flip1, true, key, x);  // (0,1) (2,3)
            quad_comparator<kQuadXor2>(flip2, true, key, x);  // (0,2) (1,3)
            // (2,3), which swaps only where a key is NaN (see node4_fast)
            if (!fast) quad_comparator<kQuadXor1>(flip1, c >= 2u, key, x);
            // the lane holds sorted position c: positions 3, 2, 1, 0 are
            // pushed in this order, the last stays as the next item
            const uint32_t vm = (uint32_t)(__ballot(x != kNoEntry) >> qbase) & 15u;
            const uint32_t x0 = quad_dpp<0x00>(x), x1 = quad_dpp<0x55>(x), x2 = quad_dpp<0xAA>(x), x3 = quad_dpp<0xFF>(x);
            pop = vm == 0u;
            if (!pop) {
                const uint32_t n = (uint32_t)__popc(vm);
                if (x != kNoEntry && (vm & ((1u << c) - 1u)) != 0u) st.put(st.top + st.stride4 * (uint32_t)__popc(vm >> (c + 1u)), x);
                if (st.top + st.stride4 * n >= st.max_end + st.stride4) st.overflow = true;
                st.top += st.stride4 * (n - 1u);
                cur = (vm & 1u) ? x0 : ((vm & 2u) ? x1 : ((vm & 4u) ? x2 : x3));
            }
        }
        if (pop) {
            if (st.empty()) done = true;
            else cur = st.top_pop();
        }
        if constexpr (ACCEL == 2) {
            while (!done && cur == kEmptyLeaf) {
                if (st.empty()) done = true;
                else cur = st.top_pop();
            }
        }
        if (done || st.overflow) {
            if (st.overflow) prim = -2;
            if (c == 0u) {
                if (st.overflow) raise(err);
                sink(ray, any, t, prim);
            }
            cur = kDead;
        }
    }
}

// Idle lanes of a wave from which it claims new rays.  12, 24, 32, 48 and 56
// idle lanes: 16 uneven views of the small box on the binary tree 64.3, 64.5,
// 65.1, 67.6 and 75.5 ms; the atrium frame 3.70, 3.66, 3.67, 3.65 and 3.65,
// the 7.24M-triangle 4K frame 8.08, 8.00, 8.01, 7.97 and 7.98 ms (spread 1%).
constexpr uint32_t kRefillIdle = 24;

// n rays of the first queue and, with MODE kDual, n2 any-hit rays of the
// second.  src(i, any, o, d, t) loads ray i of its queue, sink(i, any, t, prim) takes the
// result: prim = the hit primitive, -1 none, -2 stack overflow (the error
// flag is raised and the ray stops).
//
// A refill costs the wave no wait of its own: the claim's result is read a
// step later, and the new rays' origins and directions are loaded together
// with the other lanes' nodes and triangles.
template <int ACCEL, int MODE, bool COUNT, class Source, class Sink>
CT_DEV void trace_persistent(const DevScene& sc, float eps, uint32_t n, uint32_t n2, uint32_t* fetch, LaneStack& st,
                             TravCount& cnt, uint32_t* err, Source src, Sink sink) {
    bool exhausted = false, fast = false;
    bool any = MODE == kAny;  // the lane's ray is an any-hit query
    uint32_t ray = 0, cur = kDead, isnew = 0;
    f3 o = mk3(0, 0, 0), d = mk3(0, 0, 0), inv = mk3(0, 0, 0);
    float t = 0.0f;
    int prim = -1;
    Fetcher fe;
    fe.base = fetch;
    fe.n = n;
    fe.n2 = MODE == kDual ? n2 : 0u;
    fe.range = (int)(blockIdx.x % kFetchRanges);
    fe.left = gridDim.x < (uint32_t)kFetchRanges ? kFetchRanges - 1 : 0;
    fe.open();
    constexpr bool kQuads = ACCEL != 8 && !COUNT;
    if constexpr (kQuads) {
        // a small launch: the range's rays shared out evenly over its waves,
        // at most 16 each, without claims
        const uint32_t wpb = blockDim.x >> 6, waves = (gridDim.x / (uint32_t)kFetchRanges) * wpb;
        if (waves != 0u && fe.total <= waves * 16u) {
            const uint32_t per = (fe.total + waves - 1u) / waves, q = lane_id() >> 2;
            const uint32_t v = ((blockIdx.x / (uint32_t)kFetchRanges) * wpb + (threadIdx.x >> 6)) * per + q;
            st.reset();
            if (q < per && v < fe.total) {
                if (MODE == kDual) any = v >= fe.nfirst;
                ray = (MODE == kDual && any) ? fe.lo2 + (v - fe.nfirst) : fe.lo + v;
                src(ray, any, o, d, t);
                inv = ray_inv<ACCEL>(sc, o, d);
                fast = ray_is_fast<ACCEL>(sc, o, inv);
                st.top = 4u * (threadIdx.x & ~3u);
                cur = root_item<ACCEL>(sc);
                if (ACCEL == 2 && cur == kEmptyLeaf) {  // a tree without triangles
                    if ((lane_id() & 3u) == 0u) sink(ray, any, t, prim);
                    cur = kDead;
                }
            }
            trace_quads<ACCEL>(sc, eps, o, d, inv, fast, any, ray, cur, t, prim, st, err, sink);
            return;
        }
    }
    while (true) {
        // claim rays for the idle lanes once kRefillIdle of them are idle
        // (wave-uniform); the result is read after this step's tests
        // (a lane whose new ray is on its way is not idle, and idle lanes stay
        // idle until the result is there, so every claimed ray gets a lane)
        const uint32_t want = (uint32_t)__popcll(__ballot(cur == kDead && isnew == 0u));
        const bool refill = !exhausted && want >= kRefillIdle;
        if (exhausted && want >= (kQuads ? 48u : 64u)) break;
        uint32_t got;
        if (refill) got = fe.claim(want);
        bool done = false;
        if (cur != kDead) {
            float4 rows[7];
            int kind;
            load_item<ACCEL>(sc, cur, rows, kind);
            // any-hit lanes of a two-queue launch of the wide tree sort too
            // (one code path per wave)
            done = trav_step<ACCEL, COUNT>(sc, eps, o, d, inv, fast, any, MODE != kAny, cur, t, prim, st, cnt, rows, kind);
        }
        if (isnew) {
            // the ray loaded in the previous step
            prim = -1;
            inv = ray_inv<ACCEL>(sc, o, d);
            fast = ray_is_fast<ACCEL>(sc, o, inv);
            st.reset();
            isnew = 0u;
            cur = root_item<ACCEL>(sc);
            if (ACCEL == 2 && cur == kEmptyLeaf) done = true;  // a tree without triangles
        }
        if (done) {
            if (st.overflow) {
                raise(err);
                prim = -2;
            }
            sink(ray, any, t, prim);
            cur = kDead;
        }
        if (refill) {
            const uint32_t first = __builtin_amdgcn_readfirstlane(got);
            if (first < fe.total) {
                const uint64_t m = __ballot(cur == kDead);
                const uint32_t rank = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
                if (cur == kDead && rank < min(want, fe.total - first)) {
                    const uint32_t v = first + rank;
                    if (MODE == kDual) any = v >= fe.nfirst;
                    ray = (MODE == kDual && any) ? fe.lo2 + (v - fe.nfirst) : fe.lo + v;
                    // loads only, used a step later
                    src(ray, any, o, d, t);
                    isnew = 1u;
                }
            } else {
                exhausted = !fe.next();
            }
        }
    }
    if constexpr (kQuads) {
        // the wave's last rays, at most 16: lane r's alive ray number i moves
        // to quad i (its stack stays where it is)
        const uint64_t alive = __ballot(cur != kDead);
        if (alive == 0) return;
        const uint32_t rank = __builtin_amdgcn_mbcnt_hi((uint32_t)(alive >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)alive, 0u));
        // idle lanes send to lane 1, which no quad reads
        const uint32_t n_alive = (uint32_t)__popcll(alive);
        const uint32_t dst = 4u * (cur != kDead ? rank : 0u);
        const uint32_t from = quad_dpp<0x00>((uint32_t)__builtin_amdgcn_ds_permute((int)(4u * (cur != kDead ? dst : dst + 1u)), (int)lane_id()));
        const bool live = (lane_id() >> 2) < n_alive;
        const int sl = live ? (int)from : 0;
        const uint32_t flags = __shfl((any ? 1u : 0u) | (fast ? 2u : 0u), sl);
        const f3 qo = mk3(__shfl(o.x, sl), __shfl(o.y, sl), __shfl(o.z, sl));
        const f3 qd = mk3(__shfl(d.x, sl), __shfl(d.y, sl), __shfl(d.z, sl));
        const f3 qi = mk3(__shfl(inv.x, sl), __shfl(inv.y, sl), __shfl(inv.z, sl));
        float qt = __shfl(t, sl);
        int qp = __shfl(prim, sl);
        const uint32_t qr = __shfl(ray, sl), qtop = __shfl(st.top, sl), qc = __shfl(cur, sl);
        st.top = qtop;
        st.overflow = false;
        trace_quads<ACCEL>(sc, eps, qo, qd, qi, (flags & 2u) != 0u, (flags & 1u) != 0u, qr, live ? qc : kDead, qt, qp, st,
                           err, sink);
    }
}

// One ray per lane, traced to its end: the step loop of trace_persistent
// (the same node and triangle tests, pushes and visit order, so the same
// result for the ray) for kernels whose lanes each follow a ray of their own
// (k_paths).  t: in, the ray's extent; out, the closest hit's distance.
// Returns the hit primitive, -1 for none, -2 when the stack bound was
// exceeded (the error flag is raised).  any: stop at the first hit (a
// per-lane flag, so closest-hit and any-hit lanes step together).
template <int ACCEL>
CT_DEV int trace_single(const DevScene& sc, float eps, f3 o, f3 d, float& t, bool any, LaneStack& st,
                        uint32_t* err) {
    const f3 inv = ray_inv<ACCEL>(sc, o, d);
    const bool fast = ray_is_fast<ACCEL>(sc, o, inv);
    int prim = -1;
    uint32_t cur = root_item<ACCEL>(sc);
    TravCount cnt{0u, 0u, 0u, 0u};
    st.reset();
    if (ACCEL == 2 && cur == kEmptyLeaf) return prim;  // a tree without triangles
    while (true) {
        float4 n[7];
        int kind;
        load_item<ACCEL>(sc, cur, n, kind);
        if (trav_step<ACCEL, false>(sc, eps, o, d, inv, fast, any, true, cur, t, prim, st, cnt, n, kind)) break;
    }
    if (st.overflow) {
        raise(err);
        return -2;
    }
    return prim;
}

}  // namespace ctd
