// rt_wide8.h — 8-entry nodes over a bound tree, for the queue tracer and the primary rays.
//
// The reference tests a triangle exactly when every box on its path from the root passes, so a
// segment is occluded exactly when some triangle is hit by the triangle test AND every box of its
// path passes the box test. The second half has to be known only for triangles that are hit, so
// the walk may test any boxes in any rounding as long as it never skips such a triangle: a hit is
// then confirmed against the reference's own boxes (w8_confirm). That frees the layout: a node
// holds up to 8 entries (internal nodes or triangles) collapsed from the binary tree, with box planes of 11 bits relative to the node, 128 bytes per node against 128 per
// 4 entries with fp32 planes.
//
// Conservative boxes. Every box is grown by s = 192 u C before it is quantised outwards
// (u = 2^-24, C the largest |box coordinate| of the tree), and the walk forms each slab distance as
// t(q) = RN(q S + N), S = 2^e inv (exact), N = RN(RN(p - o) inv), inv the hardware's 1/d (within
// 2u). With |o| <= 16 C the walk's distance differs from the exact one by at most 6u (|q 2^e| +
// |p - o|) / |d| <= 6u (4.01 C + 17.01 C) / |d|, the reference's RN(RN(b - o)/d) by at most 2.01u
// (17 C) / |d|: 161 u C / |d| in all, less than the growth s / |d|. So the walk's near distance of a box is at most,
// and its far distance at least, the reference's for every box inside it, and the walk enters
// every node on the path of a triangle whose path passes. 1/d is clamped to +-K (SceneView::invMax,
// s K >= 4): for |d| < 1/K a segment that starts inside the grown slab keeps near < 0 and far > 1,
// and one that starts outside cannot reach the box itself (its distance exceeds s K), so zero,
// denormal (the hardware's reciprocal is then infinite) and tiny components are covered too. Long
// segments are another matter: the hardware flushes the reciprocal of a component above 2^126 to
// zero, which puts all its distances at 0, and shorter ones leave S and the slack without bits in a
// small scene. With |d| <= min(2^99, 2^96 C) the reciprocal is normal, S is at least 2^-123 (a
// node's step 2^e is at least 2^-27 C) and the slack s / |d| at least 2^-113, far above what N's product
// loses below the normal range.
//
// Far origins. With |o| > 16 C the rounding of p - o and b - o outgrows s. Such a walk sets every
// near distance back and every far one forward by e = 9 u |o| inv, per axis: the distances differ by
// at most u (6 (|q 2^e| + |p - o|) + 2.01 |b - o|) / |d| <= u (32.2 C + 8.01 |o|) / |d|, one rounding
// more than above included, less than (s + e) / |d|. All
// distances stay finite up to |o| = 2^24 C (2^24 C K < 2^125), where C is an ulp of o. A batch's tracer
// walks these segments as it takes them (occluded_far): 300,000 from 100 times the scene's size take 0.11
// ms, through the binary tree 0.40. Its own visits have no slack: 4 million segments took 0.78
// ms, for 0.74, with a choice in every visit. The passes' rays start on surfaces.
//
// Segments that are longer, from farther away or have a non-finite component walk the binary tree
// (occluded_slow). The same holds for unbounded rays (the primary rays) of unit
// direction, whose boxes all lie within 31 C of the origin: s K >= 31 C.
#pragma once

#include "rt_traverse.h"

namespace rt {

constexpr int kW8Stack = 16;  // entries of a lane's stack: trees of at most 17 levels of 8-entry nodes
constexpr float kW8Grow = 192.0f * 5.9604645e-8f;  // s / C
constexpr float kW8Reach = 16.0f;                  // |o| / C at most, without the slack of far origins
constexpr float kW8Far = 0x1p24f;                  // and with it
constexpr float kW8FarSlack = 9.0f * 5.9604645e-8f;
// Trees whose largest |box coordinate| C keeps every product of the walk finite and its slack normal
__host__ __device__ inline bool w8_covers(float c) { return c > 1e-18f && c < 1e18f; }
constexpr float kW8Long = 0x1p96f, kW8Longest = 0x1p99f;  // |d| / C and |d| at most

struct alignas(128) W8Node {
    float p[3];         // the node's corner: plane q of axis a lies at p[a] + q 2^e[a]
    uint32_t child;     // first internal child's index (23 bits) << 8 | mask of the internal entries:
                        // they take the lowest slots, and the child of slot k is node (child >> 8) + k
    uint32_t exps;      // signed byte a < 3: e[a]; byte 3: mask of the triangle entries
    uint32_t triBase;   // the triangle of slot k is triBase + k
    uint32_t axis;      // the internal entries are in descending order of their centres on this axis
    uint32_t pad;
    uint16_t plane[3][2][8];  // per axis: low and high planes of the 8 slots (halves, 0..2047)
};
static_assert(sizeof(W8Node) == 128, "one 128-byte line per node");

typedef _Float16 h8 __attribute__((ext_vector_type(8)));

// A segment for the 8-entry walk.
struct W8Seg {
    f3 o, d, inv;
    uint32_t ox, oy, oz;  // byte offset of an axis's near planes: 0 for d > 0, else 16
};
// Which walk covers a segment: the plain one, the one with slack for its origin, or none. w is filled in any case.
enum class W8Cover { near, far, none };
__device__ __forceinline__ W8Cover make_w8seg(W8Seg &w, f3 o, f3 d, float maxCoord, float invMax) {
    w.o = o;
    w.d = d;
    const f3 inv{__builtin_amdgcn_rcpf(d.x), __builtin_amdgcn_rcpf(d.y), __builtin_amdgcn_rcpf(d.z)};
    w.inv = f3{fminf(fmaxf(inv.x, -invMax), invMax), fminf(fmaxf(inv.y, -invMax), invMax),
               fminf(fmaxf(inv.z, -invMax), invMax)};
    w.ox = w.inv.x > 0.0f ? 0u : 16u;
    w.oy = w.inv.y > 0.0f ? 0u : 16u;
    w.oz = w.inv.z > 0.0f ? 0u : 16u;
    const float reach = kW8Reach * maxCoord, longest = fminf(kW8Long * maxCoord, kW8Longest);
    // comparisons are false for NaN
    if (!(fabsf(d.x) <= longest && fabsf(d.y) <= longest && fabsf(d.z) <= longest)) return W8Cover::none;
    if (fabsf(o.x) <= reach && fabsf(o.y) <= reach && fabsf(o.z) <= reach) return W8Cover::near;
    const float far = kW8Far * maxCoord;
    return fabsf(o.x) <= far && fabsf(o.y) <= far && fabsf(o.z) <= far ? W8Cover::far : W8Cover::none;
}

// What a visit leaves: the child word with only the internal entries that are passed left in the
// mask, and the mask of the triangle entries that are passed (slot k: triangle triBase + k). With
// kOrder also the node's axis, and the slot of the nearest internal entry that is passed.
struct W8Visit {
    uint32_t child, tris, triBase, axis, nearest;
};
// Visits `node` on [0, tMax]. 12 VALU per box: 6 FMA with half operands, max3, min3, the clamp to
// the segment, a subtraction whose sign is shifted into the mask. kFar: with the slack of far origins.
// kPass: what may be scheduled across the end of the loads (sched_barrier's mask; 0 or 1, as measured).
template <bool kOrder, bool kFar = false, int kPass = 0>
__device__ __forceinline__ W8Visit w8_visit(const W8Seg &w, const W8Node *__restrict__ nodes, uint32_t node,
                                            float tMax) {
    const char *base = reinterpret_cast<const char *>(nodes);
    const uint32_t row = node << 7;
    const float4 h0 = *reinterpret_cast<const float4 *>(base + row);
    uint3 h1{0u, 0u, 0u};
    if (kOrder) {
        h1 = *reinterpret_cast<const uint3 *>(base + row + 16);
    } else {
        const uint2 v = *reinterpret_cast<const uint2 *>(base + row + 16);
        h1.x = v.x;
        h1.y = v.y;
    }
    const h8 nx = *reinterpret_cast<const h8 *>(base + (row + w.ox) + 32);
    const h8 fx = *reinterpret_cast<const h8 *>(base + (row + (w.ox ^ 16u)) + 32);
    const h8 ny = *reinterpret_cast<const h8 *>(base + (row + w.oy) + 64);
    const h8 fy = *reinterpret_cast<const h8 *>(base + (row + (w.oy ^ 16u)) + 64);
    const h8 nz = *reinterpret_cast<const h8 *>(base + (row + w.oz) + 96);
    const h8 fz = *reinterpret_cast<const h8 *>(base + (row + (w.oz ^ 16u)) + 96);
    // the eight loads under way together: left to itself the compiler may wait for one after another (4
    // million segments 0.88 ms instead of 0.74, depending on the code around)
    __builtin_amdgcn_sched_barrier(kPass);
    const int32_t e = static_cast<int32_t>(h1.x);
    const float sx = ldexpf(w.inv.x, (e << 24) >> 24), sy = ldexpf(w.inv.y, (e << 16) >> 24),
                sz = ldexpf(w.inv.z, (e << 8) >> 24);
    const float bx = (h0.x - w.o.x) * w.inv.x, by = (h0.y - w.o.y) * w.inv.y, bz = (h0.z - w.o.z) * w.inv.z;
    f3 nb{bx, by, bz}, fb = nb;
    if (kFar) {
        const f3 slack{kW8FarSlack * fabsf(w.o.x * w.inv.x), kW8FarSlack * fabsf(w.o.y * w.inv.y),
                       kW8FarSlack * fabsf(w.o.z * w.inv.z)};
        nb = nb - slack;
        fb = fb + slack;
    }
    const uint32_t inner = __float_as_uint(h0.w);
    uint32_t miss = 0, near = 0xffffffffu;
#pragma unroll
    for (int k = 7; k >= 0; --k) {
        const float lo = fmaxf(fmaxf(fmaf(static_cast<float>(nx[k]), sx, nb.x), fmaf(static_cast<float>(ny[k]), sy, nb.y)),
                               fmaf(static_cast<float>(nz[k]), sz, nb.z));
        const float hi = fminf(fminf(fmaf(static_cast<float>(fx[k]), sx, fb.x), fmaf(static_cast<float>(fy[k]), sy, fb.y)),
                               fmaf(static_cast<float>(fz[k]), sz, fb.z));
        const float gap = fminf(hi, tMax) - fmaxf(lo, 0.0f);  // negative: the box is missed
        miss = __builtin_amdgcn_alignbit(miss, __float_as_uint(gap), 31);
        if (kOrder) {  // entry distances are not negative: they order as their bits
            const uint32_t key = (__float_as_uint(fmaxf(lo, 0.0f)) & ~7u) | static_cast<uint32_t>(k);
            near = min(near, gap >= 0.0f && ((inner >> k) & 1u) ? key : 0xffffffffu);
        }
    }
    return W8Visit{inner & ~miss, (h1.x >> 24) & ~miss, h1.y, h1.z, near & 7u};
}

// rayTriangleIntersection over given vertices (ray_tri's arithmetic).
__device__ __forceinline__ bool tri_hit(float4 a, float4 b, float4 c, f3 o, f3 d) {
    const f3 p1 = xyz(a);
    const f3 e1 = xyz(b) - p1;
    const f3 e2 = xyz(c) - p1;
    const f3 p = cross(d, e2);
    float f = 1.0f / dot(e1, p);
    const f3 s = o - p1;
    const float bx = f * dot(s, p);
    if (bx < 0.0f || bx > 1.0f) return false;
    const f3 q = cross(s, e1);
    const float by = f * dot(d, q);
    if (by < 0.0f || by + bx > 1.0f) return false;
    f *= dot(e2, q);
    return f > 0.0f && f < 1.0f;
}

__device__ __forceinline__ bool regular_segment(f3 o, f3 d) {
    constexpr float kInf = __builtin_huge_valf();
    return fabsf(d.x) > 0.0f && fabsf(d.y) > 0.0f && fabsf(d.z) > 0.0f && fabsf(d.x) < kInf && fabsf(d.y) < kInf &&
           fabsf(d.z) < kInf && fabsf(o.x) < kInf && fabsf(o.y) < kInf && fabsf(o.z) < kInf;
}

// The box tests of the primary rays (an unbounded ray: no rmin < 1), in the division form.
__device__ __forceinline__ bool ray_box_div_unbounded(f3 o, f3 d, float4 mn, float4 mx) {
    const float ax = (mn.x - o.x) / d.x, ay = (mn.y - o.y) / d.y, az = (mn.z - o.z) / d.z;
    const float bx = (mx.x - o.x) / d.x, by = (mx.y - o.y) / d.y, bz = (mx.z - o.z) / d.z;
    const float rmin = gmax(gmin(ax, bx), gmax(gmin(ay, by), gmin(az, bz)));
    const float rmax = gmin(gmax(ax, bx), gmin(gmax(ay, by), gmax(az, bz)));
    return rmax >= rmin && rmax > 0.0f;
}

// Side `side` of node x: whether its box, as stored, is passed (kSeg: by the segment, else by the
// unbounded ray).
template <bool kSeg>
__device__ __forceinline__ bool side_passes(const Node *__restrict__ nodes, uint32_t x, uint32_t side, f3 o, f3 d) {
    const float4 *p = reinterpret_cast<const float4 *>(nodes + x) + 2 * side;
    return kSeg ? ray_box_div(o, d, p[0], p[1]) : ray_box_div_unbounded(o, d, p[0], p[1]);
}

// Whether the reference tests the triangle stored under `slot` (2 node + side) for this segment:
// every box from that slot up to the root passes. In a nested tree a regular segment that passes a
// box passes every box around it (the slab distances are monotone in the planes), so the slot's
// own box decides.
template <bool kSeg>
__device__ __forceinline__ bool path_passes(const Node *__restrict__ nodes, const uint32_t *__restrict__ parent,
                                            uint32_t slot, f3 o, f3 d, bool leafOnly) {
    for (;;) {
        const uint32_t x = slot >> 1;
        if (!side_passes<kSeg>(nodes, x, slot & 1u, o, d)) return false;
        if (leafOnly || x == 0) return true;
        slot = parent[x];
    }
}

// Confirms a triangle hit (see the file comment). `tight`: every leaf box of the tree is the
// bounding box of its triangle, so the box needs no load. Most confirmations are clear from
// distances formed with the hardware reciprocal (within 4u of the exact quotient of the rounded
// difference, the reference's within u of it: the slack of 16u covers both).
template <bool kSeg>
__device__ __forceinline__ bool w8_confirm(const Node *__restrict__ nodes, const uint32_t *__restrict__ parent,
                                           bool treeNested, bool tight, float4 a, float4 b, float4 c, f3 o, f3 d) {
    const bool leafOnly = treeNested && regular_segment(o, d);
    if (leafOnly && tight) {
        const float4 mn = make_float4(fminf(fminf(a.x, b.x), c.x), fminf(fminf(a.y, b.y), c.y),
                                      fminf(fminf(a.z, b.z), c.z), 0.0f);
        const float4 mx = make_float4(fmaxf(fmaxf(a.x, b.x), c.x), fmaxf(fmaxf(a.y, b.y), c.y),
                                      fmaxf(fmaxf(a.z, b.z), c.z), 0.0f);
        const float ix = __builtin_amdgcn_rcpf(d.x), iy = __builtin_amdgcn_rcpf(d.y), iz = __builtin_amdgcn_rcpf(d.z);
        const float ax = (mn.x - o.x) * ix, ay = (mn.y - o.y) * iy, az = (mn.z - o.z) * iz;
        const float bx = (mx.x - o.x) * ix, by = (mx.y - o.y) * iy, bz = (mx.z - o.z) * iz;
        const float rmin = fmaxf(fmaxf(fminf(ax, bx), fminf(ay, by)), fminf(az, bz));
        const float rmax = fminf(fminf(fmaxf(ax, bx), fmaxf(ay, by)), fmaxf(az, bz));
        constexpr float kRel = 16.0f * 5.9604645e-8f, kAbs = 1e-30f;
        const float big = fmaxf(fmaxf(fmaxf(fabsf(ax), fabsf(bx)), fmaxf(fabsf(ay), fabsf(by))),
                                fmaxf(fabsf(az), fabsf(bz)));  // a flushed or infinite reciprocal fails this test
        const float minHi = rmin + (fabsf(rmin) * kRel + kAbs), maxLo = rmax - (fabsf(rmax) * kRel + kAbs);
        const float dMax = fmaxf(fmaxf(fabsf(d.x), fabsf(d.y)), fabsf(d.z));
        if (big < 1e30f && dMax < 1e30f && (!kSeg || minHi < 1.0f) && maxLo >= minHi && maxLo > 0.0f) return true;
        return kSeg ? ray_box_div(o, d, mn, mx) : ray_box_div_unbounded(o, d, mn, mx);
    }
    return path_passes<kSeg>(nodes, parent, __float_as_uint(a.w), o, d, leafOnly);
}

// The reference's answer for a segment of far origin, by the lane itself; `stk` is its column of kW8Stack
// entries, `stride` apart.
__device__ __forceinline__ bool occluded_far(const W8Seg &w, const W8Node *__restrict__ w8, const float4 *__restrict__ w8Tris,
                                             const Node *__restrict__ nodes, const uint32_t *__restrict__ parent,
                                             bool treeNested, uint32_t *stk, int stride) {
    uint32_t grp = 1u;  // as in the tracer: first child << 8 | mask of the entries to visit
    int top = 0;
    for (;;) {
        if ((grp & 0xffu) == 0) {
            if (top == 0) return false;
            --top;
            grp = stk[top * stride];
        }
        const uint32_t node = (grp >> 8) + static_cast<uint32_t>(__builtin_ctz(grp));
        grp &= grp - 1u;
        const W8Visit v = w8_visit<false, true>(w, w8, node, 1.0f);
        for (uint32_t m = v.tris; m; m &= m - 1u) {
            const float4 *t = w8Tris + 3 * static_cast<size_t>(v.triBase + static_cast<uint32_t>(__builtin_ctz(m)));
            const float4 a = t[0], b = t[1], c = t[2];
            // w8_confirm without its quick form, whose registers the tracer would have to find
            if (tri_hit(a, b, c, w.o, w.d) &&
                path_passes<true>(nodes, parent, __float_as_uint(a.w), w.o, w.d, treeNested && regular_segment(w.o, w.d)))
                return true;
        }
        if (v.child & 0xffu) {
            if (grp & 0xffu) {
                stk[top * stride] = grp;
                ++top;
            }
            grp = v.child;
        }
    }
}

// The reference's answer for any segment, from the binary nodes and their parents, without a stack:
// for the segments the 8-entry walk does not cover. Bit b of `right` is set while the right side of the
// node b levels above the current one is still to visit (trees have at most 64 levels).
__device__ __forceinline__ bool occluded_slow(const Node *__restrict__ nodes, const float4 *__restrict__ tris,
                                              const uint32_t *__restrict__ parent, f3 o, f3 d) {
    const Seg s = make_seg(o, d);
    uint64_t right = 0;
    int32_t x = 0;
    for (;;) {
        const Node nd = load_node(nodes, x);
        const bool l = ray_box(s, nd.lmin, nd.lmax), r = ray_box(s, nd.rmin, nd.rmax);
        if (l && nd.left < 0 && ray_tri(tris, ~nd.left, o, d)) return true;
        if (r && nd.right < 0 && ray_tri(tris, ~nd.right, o, d)) return true;
        const bool goL = l && nd.left >= 0, goR = r && nd.right >= 0;
        if (goL || goR) {
            right = right << 1 | (goL && goR ? 1u : 0u);
            x = goL ? nd.left : nd.right;
            continue;
        }
        if (right == 0) return false;
        for (int up = __builtin_ctzll(right) + 1; up > 0; --up) x = static_cast<int32_t>(parent[x] >> 1);
        right = (right >> __builtin_ctzll(right)) ^ 1ull;
        x = nodes[x].right;
    }
}

}  // namespace rt
