// bvh_build.hip — AabbTree::build (src/aabbTreeBuilder.cpp:52-214) on the GPU: the reference's
// 12-bucket binned-SAH tree, node for node and bit for bit, built one tree level per round of
// launches.
//
// The reference pops index ranges of one primitive-order array from a FIFO, so node ids are
// breadth-first and each tree level is a list of disjoint ranges in position order. Ranges of more
// than kSub primitives are split level by level, one round of launches for all of a level:
//   level              ranks the ranges to split; smaller ones go to the subtree list
//   bounds             centroid and box bounds of each range (and of its halves)
//   bin                bucket of each primitive on the range's longest centroid axis; box and
//                      count per bucket
//   choose             the reference's SAH sweep over the 12 buckets, 16 lanes per range
//   partition          the reference's swap partition, reproduced exactly (below)
// and the host reads back only the number of ranges to split. Each smaller range then becomes a
// whole subtree in one workgroup's LDS (k_bvh_subtrees). A split at position mid makes node mid - 1
// of a temporary array: every inner position is split at once, and position order is the order of a
// level's nodes, so the breadth-first ids are a stable sort of that array by level.
//
// Where the time goes: a level costs its launches (about 5 us each) and its readback, whatever its
// size, and the lower half of a tree's levels holds ranges of a few primitives. 136,000 triangles
// (23 levels): 3.2 ms with every level split that way, in 20 launches each; 1.15 ms with the last 12
// to 13 levels in k_bvh_subtrees (0.22 ms) and 8 launches for each of the others, 1.06 with the 8-entry
// nodes' collapse on 8 lanes a node. 1,200 triangles 1.52 -> 0.39 ms, 2.3 million 18.6 -> 6.4 ms (all
// with the traversal's nodes, bind_tree).
//
// Exact min/max. nv_min(a, b) = a < b ? a : b (nvmath.inl:2414-2420) folded in primitive order
// returns, among equal values, the LAST one; equal floats differ in bits only as +0/-0. Each fold
// is therefore an order-independent atomic min (max) over 64-bit keys: the value in a monotone
// integer code with -0 folded onto +0, then the position (complemented for min) so that the
// later position wins a tie; the winner's own bits are then read back at that position.
//
// Exact partition. The reference swaps every left primitive (bucket <= split) with the first
// element of the right block (aabbTreeBuilder.cpp:178-183). Left primitives keep their order;
// the right block acts as a queue whose front moves to its back whenever a left primitive
// arrives. After the pass, a position p >= mid holds what was placed there at step p: the
// primitive itself if it is a right one, else the front of the block at that step, which sat at
// first + (left primitives before p) and is resolved the same way. That chain only moves to
// smaller positions; it is followed by pointer jumping in place (k_bvh_scatter).
#include <hip/hip_runtime.h>

#include <cfloat>
#include <climits>
#include <cstdint>
#include <cstring>

#include "carve.h"
#include "ctx.h"
#include "kernels.h"
#include "rt_wide8.h"
#include "scan.h"

using namespace rki;

namespace {

constexpr int kBuckets = 12;
constexpr int kBoundWords = 24;                 // centroid lo/hi, box lo/hi keys; the halves' box lo/hi
constexpr int kBinWords = 7;                    // box lo/hi keys + count
constexpr int kAcc = kBoundWords + kBuckets * kBinWords;  // 64-bit words per split range
constexpr int kSlots = 4;  // split ranges a 256-lane group pre-reduces in LDS
// Primitives of a range that one workgroup finishes. 136,000 triangles (2.3 million): with 256 1.21
// (6.94) ms, with 512 1.25 (6.61), with 1024 1.25 (7.12): longer subtrees against more levels.
constexpr uint32_t kSub = 512;
constexpr uint32_t kSubWide = 32;  // and those from which on its 16 lanes fold parts of them, not components
constexpr uint32_t kScanGroup = rscan::kItems;  // positions per block of the partition's prefix sums

struct Seg {  // a range of the level; link = parent node * 2 + side, -1 for the root
    uint32_t first, last;
    int32_t link, pad;
};
struct Split {  // a range being split at this level
    uint32_t first, last, mid;
    uint32_t bucket;      // last bucket of the left side
    uint32_t degenerate;  // the sweep put everything on one side: halved instead
    int32_t link;
    uint32_t pad[2];
};
struct Sub {  // a range of 2..kSub primitives, its level and link
    uint32_t first, last;
    int32_t link;
    uint32_t level;
};
struct Params {
    int32_t axis;
    float lo, width, parentArea;
};
struct Info {
    uint32_t splits;  // ranges to split at this level
    uint32_t subs;    // ranges in the subtree list
    uint32_t bad;     // a vertex coordinate is not finite
    uint32_t depth;   // deepest level of a node
};

using u64 = unsigned long long;

__device__ inline float nv_min(float a, float b) { return a < b ? a : b; }
__device__ inline float nv_max(float a, float b) { return a > b ? a : b; }

__device__ inline uint32_t code(float v) {
    const uint32_t u = __float_as_uint(v == 0.0f ? 0.0f : v);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ inline float uncode(uint32_t c) {
    return __uint_as_float((c & 0x80000000u) ? (c & 0x7fffffffu) : ~c);
}
__device__ inline u64 key_min(float v, uint32_t p) { return (static_cast<u64>(code(v)) << 32) | static_cast<uint32_t>(~p); }
__device__ inline u64 key_max(float v, uint32_t p) { return (static_cast<u64>(code(v)) << 32) | p; }

// word layout of a split range's accumulator: [0,3) centroid lo, [3,6) centroid hi, [6,9) box
// lo, [9,12) box hi, [12,18) box lo, hi of the positions before (first + last) / 2, [18,24) of the
// others; then per bucket b at 24 + 7b: [0,3) box lo, [3,6) box hi, [6] count
__host__ __device__ inline bool is_min_word(int w) { return w < kBoundWords ? ((w / 3) & 1) == 0 : ((w - kBoundWords) % kBinWords) < 3; }
__host__ __device__ inline bool is_count_word(int w) { return w >= kBoundWords && (w - kBoundWords) % kBinWords == 6; }
__device__ inline u64 word_init(int w) { return (!is_count_word(w) && is_min_word(w)) ? ~0ull : 0ull; }

__device__ inline void atomic_key(u64 *a, u64 k, bool isMin) {
    if (isMin) atomicMin(a, k);
    else atomicMax(a, k);
}

// component k of position p's box lo (which 1), box hi (2) or centroid (0)
__device__ inline float element(const uint32_t *idx, const float4 *box, uint32_t p, int which, int k) {
    const uint32_t t = idx[p];
    const float4 lo = box[2 * t], hi = box[2 * t + 1];
    const float l = k == 0 ? lo.x : (k == 1 ? lo.y : lo.z);
    const float h = k == 0 ? hi.x : (k == 1 ? hi.y : hi.z);
    return which == 1 ? l : (which == 2 ? h : 0.5f * (l + h));
}
__device__ inline float decode(u64 key, bool isMin, const uint32_t *idx, const float4 *box, int which, int k) {
    const float v = uncode(static_cast<uint32_t>(key >> 32));
    if (v != 0.0f) return v;
    const uint32_t p = isMin ? ~static_cast<uint32_t>(key) : static_cast<uint32_t>(key);
    return element(idx, box, p, which, k);  // +0 or -0: the winner's own bits
}

__device__ inline float half_area(const float lo[3], const float hi[3]) {  // surfaceAreaHeuristic
    const float sx = hi[0] - lo[0], sy = hi[1] - lo[1], sz = hi[2] - lo[2];
    return sx * sy + sx * sz + sy * sz;
}

// Bucket axis and placement of a range (aabbTreeBuilder.cpp:95-121) from its bounds.
__device__ inline Params make_params(const float cLo[3], const float cHi[3], const float bLo[3], const float bHi[3]) {
    Params q;
    q.parentArea = half_area(bLo, bHi);
    float extent[3];
    for (int k = 0; k < 3; ++k) extent[k] = cHi[k] - cLo[k];
    int axis = extent[0] > extent[1] ? 0 : 1;
    if ((axis == 0 ? extent[0] : extent[1]) < extent[2]) axis = 2;
    q.axis = axis;
    q.lo = axis == 0 ? cLo[0] : axis == 1 ? cLo[1] : cLo[2];
    q.width = (axis == 0 ? extent[0] : axis == 1 ? extent[1] : extent[2]) / static_cast<float>(kBuckets);
    return q;
}
__device__ inline uint32_t bucket_of(const Params &q, float c) {
    float f = (c - q.lo) / q.width;
    f = f < 0.5f ? 0.5f : f;  // nv_clamp(f, 0.5, numBuckets - 0.5)
    f = f > static_cast<float>(kBuckets) - 0.5f ? static_cast<float>(kBuckets) - 0.5f : f;
    // coincident centroids give 0/0 (undefined in the reference): bucket 0
    return f == f ? static_cast<uint32_t>(f) : 0u;
}

// Lane i of a row of 16 gets v of lane i - D (shr) or i + D (shl), `none` where the row ends.
template <int D>
__device__ inline float row_shr(float none, float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(none), __float_as_int(v), 0x110 + D, 0xf, 0xf, false));
}
template <int D>
__device__ inline float row_shl(float none, float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(none), __float_as_int(v), 0x100 + D, 0xf, 0xf, false));
}
struct Bin {  // Bucket (aabbTreeBuilder.cpp:33-50)
    float lo[3], hi[3];
    uint32_t count;
};
__device__ inline Bin bin_empty() {
    return Bin{{FLT_MAX, FLT_MAX, FLT_MAX}, {-FLT_MAX, -FLT_MAX, -FLT_MAX}, 0u};
}
__device__ inline float bin_cost(const Bin &b) { return static_cast<float>(b.count) * half_area(b.lo, b.hi); }
// One step of a row's ordered prefix (suffix) fold. The folds keep the last of equal values, so
// folding blocks of buckets in their order gives what folding the buckets one by one gives.
template <int D>
__device__ inline void fold_left(Bin &b) {
    for (int k = 0; k < 3; ++k) {
        b.lo[k] = nv_min(row_shr<D>(FLT_MAX, b.lo[k]), b.lo[k]);
        b.hi[k] = nv_max(row_shr<D>(-FLT_MAX, b.hi[k]), b.hi[k]);
    }
    b.count += static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(b.count), 0x110 + D, 0xf, 0xf, false));
}
template <int D>
__device__ inline void fold_right(Bin &b) {
    for (int k = 0; k < 3; ++k) {
        b.lo[k] = nv_min(row_shl<D>(FLT_MAX, b.lo[k]), b.lo[k]);
        b.hi[k] = nv_max(row_shl<D>(-FLT_MAX, b.hi[k]), b.hi[k]);
    }
    b.count += static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(b.count), 0x100 + D, 0xf, 0xf, false));
}
// The SAH sweep (aabbTreeBuilder.cpp:131-175) by a row of 16 lanes, lane b holding bucket b (empty
// beyond the last): left and right end as the two sides of a split after bucket b, and the result is
// the first cheapest split, or -1 where no cost is a number below FLT_MAX.
__device__ inline int sah_sweep(Bin &left, Bin &right, float parentArea) {
    const int b = threadIdx.x & 15;
    fold_left<1>(left);
    fold_left<2>(left);
    fold_left<4>(left);
    fold_left<8>(left);
    fold_right<1>(right);
    fold_right<2>(right);
    fold_right<4>(right);
    fold_right<8>(right);
    for (int k = 0; k < 3; ++k) {
        right.lo[k] = row_shl<1>(FLT_MAX, right.lo[k]);
        right.hi[k] = row_shl<1>(-FLT_MAX, right.hi[k]);
    }
    right.count = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(right.count), 0x101, 0xf, 0xf, false));
    float cost = 0.125f + (bin_cost(left) + bin_cost(right)) / parentArea;
    int split = b;
    if (!(b < kBuckets - 1 && cost < FLT_MAX)) {
        cost = INFINITY;
        split = 16;
    }
#pragma unroll
    for (int d = 1; d < 16; d <<= 1) {
        const float c = __shfl_xor(cost, d);
        const int o = __shfl_xor(split, d);
        if (c < cost || (c == cost && o < split)) {
            cost = c;
            split = o;
        }
    }
    return split < 16 ? split : -1;
}

__device__ inline void write_box(float *dst, const float *v) {  // vec4(vec3) sets w = 1
    dst[0] = v[0];
    dst[1] = v[1];
    dst[2] = v[2];
    dst[3] = 1.0f;
}

// ---- kernels ----

// triangles out (w = 1), primitive boxes (aabbForTriangle), the identity order, one root range, its
// accumulator
__global__ __launch_bounds__(256) void k_bvh_prep(uint32_t n, const float *xyz, restir_triangle *tris,
                                                  float4 *box, uint32_t *idx, int32_t *segOf, u64 *acc, Seg *root,
                                                  Info *info) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i < kAcc) acc[i] = word_init(static_cast<int>(i));
    if (i == 0) *root = Seg{0u, n, -1, 0};
    if (i >= n) return;
    float v[9];
    bool finite = true;
    for (int k = 0; k < 9; ++k) {
        v[k] = xyz[9 * static_cast<size_t>(i) + k];
        finite = finite && (v[k] - v[k] == 0.0f);
    }
    if (!finite) atomicOr(&info->bad, 1u);
    restir_triangle t;
    for (int k = 0; k < 3; ++k) {
        t.p1[k] = v[k];
        t.p2[k] = v[3 + k];
        t.p3[k] = v[6 + k];
    }
    t.p1[3] = t.p2[3] = t.p3[3] = 1.0f;
    tris[i] = t;
    float lo[3], hi[3];
    for (int k = 0; k < 3; ++k) {
        lo[k] = v[k];
        hi[k] = v[k];
        lo[k] = nv_min(lo[k], v[3 + k]);
        hi[k] = nv_max(hi[k], v[3 + k]);
        lo[k] = nv_min(lo[k], v[6 + k]);
        hi[k] = nv_max(hi[k], v[6 + k]);
    }
    box[2 * i] = make_float4(lo[0], lo[1], lo[2], 0.0f);
    box[2 * i + 1] = make_float4(hi[0], hi[1], hi[2], 0.0f);
    idx[i] = i;
    segOf[i] = 0;
}

__device__ inline void set_child(restir_aabb_tree_node *tmp, int32_t link, int32_t value) {
    if (link < 0) return;
    restir_aabb_tree_node &parent = tmp[link >> 1];
    if (link & 1) parent.rightChild = value;
    else parent.leftChild = value;
}

// One workgroup: the level's ranges in order. Those to split get consecutive ranks, ranges of one
// primitive become leaves, the others go to the subtree list.
__global__ __launch_bounds__(256) void k_bvh_level(uint32_t S, uint32_t level, const Seg *segs, const uint32_t *idx,
                                                   restir_aabb_tree_node *tmp, int32_t *segRank, Split *splits, Sub *subs,
                                                   Info *info) {
    __shared__ uint32_t waveCount[4];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    uint32_t base = 0;
    for (uint32_t s0 = 0; s0 < S; s0 += 256u) {
        const uint32_t s = s0 + threadIdx.x;
        Seg g{};
        if (s < S) g = segs[s];
        const uint32_t len = g.last - g.first;
        const bool big = len > kSub;
        const uint64_t m = __ballot(big);
        if (lane == 0) waveCount[wave] = static_cast<uint32_t>(__popcll(m));
        __syncthreads();
        uint32_t r = base + static_cast<uint32_t>(__popcll(m & ((1ull << lane) - 1ull)));
        for (uint32_t w = 0; w < 4; ++w) {
            if (w < wave) r += waveCount[w];
            base += waveCount[w];
        }
        __syncthreads();
        if (s >= S) continue;
        segRank[s] = big ? static_cast<int32_t>(r) : -1;
        if (big) splits[r] = Split{g.first, g.last, 0u, 0u, 0u, g.link, {0u, 0u}};
        else if (len == 1) set_child(tmp, g.link, ~static_cast<int32_t>(idx[g.first]));
        else subs[atomicAdd(&info->subs, 1u)] = Sub{g.first, g.last, g.link, level};
    }
    if (threadIdx.x == 0) info->splits = base;
}

// rank of the split range holding position p (-1: a range that is not split any more)
__device__ inline int rank_of(uint32_t p, uint32_t n, const int32_t *segOf, const int32_t *segRank) {
    const int32_t s = p < n ? segOf[p] : -1;
    return s >= 0 ? segRank[s] : -1;
}

// Adds `nw` keys (words w0.. of range r's accumulator) through LDS when r is one of the first
// kSlots ranges present in the group (ranges are position-ordered, so a group's ranks are
// consecutive), else straight to memory. Counts add; other words take min or max.
template <int NW>
struct GroupAcc {
    u64 *sh;  // kSlots * NW words
    int r0;
    __device__ void add(u64 *acc, int r, int w0, const u64 *keys, int nKeys) {
        const int slot = r - r0;
        for (int j = 0; j < nKeys; ++j) {
            const int w = w0 + j;
            if (slot < kSlots) {
                u64 *a = &sh[slot * NW + (w - base)];
                if (is_count_word(w)) atomicAdd(a, keys[j]);
                else atomic_key(a, keys[j], is_min_word(w));
            } else {
                u64 *a = &acc[static_cast<size_t>(r) * kAcc + w];
                if (is_count_word(w)) atomicAdd(a, keys[j]);
                else atomic_key(a, keys[j], is_min_word(w));
            }
        }
    }
    int base;  // first accumulator word the LDS copy mirrors
};

__device__ inline int group_min_rank(int r, int *shR) {
    if (threadIdx.x == 0) *shR = INT_MAX;
    __syncthreads();
    if (r >= 0) atomicMin(shR, r);
    __syncthreads();
    return *shR;
}

// flushes the LDS copies (words base.. base+NW of ranges r0.. r0+kSlots) to memory
template <int NW>
__device__ inline void group_flush(const u64 *sh, int r0, int base, u64 *acc) {
    __syncthreads();
    if (r0 == INT_MAX) return;
    for (int i = threadIdx.x; i < kSlots * NW; i += 256) {
        const int w = base + i % NW;
        const u64 v = sh[i];
        if (v == word_init(w)) continue;  // nothing added (empty min/max word or zero count)
        u64 *a = &acc[static_cast<size_t>(r0 + i / NW) * kAcc + w];
        if (is_count_word(w)) atomicAdd(a, v);
        else atomic_key(a, v, is_min_word(w));
    }
}

// The extreme of v over a wave's lanes (the same on every lane), and from it the key of the last
// lane that holds it: lanes hold consecutive positions, p0 is lane 0's.
template <bool MIN>
__device__ inline u64 wave_key(float v, bool active, uint32_t p0) {
    const float none = MIN ? INFINITY : -INFINITY;
    const float mine = active ? v : none;
    float x = mine;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const float o = __shfl_xor(x, d);
        x = MIN ? (o < x ? o : x) : (o > x ? o : x);
    }
    const uint64_t at = __ballot(active && mine == x);
    const uint32_t p = p0 + 63u - static_cast<uint32_t>(__clzll(static_cast<long long>(at)));
    return MIN ? key_min(x, p) : key_max(x, p);
}

__global__ __launch_bounds__(256) void k_bvh_bounds(uint32_t n, const uint32_t *idx, const int32_t *segOf,
                                                    const int32_t *segRank, const Split *splits, const float4 *box, u64 *acc) {
    __shared__ u64 sh[kSlots * kBoundWords];
    __shared__ int shR;
    const uint32_t p = blockIdx.x * 256u + threadIdx.x;
    const int r = rank_of(p, n, segOf, segRank);
    if (threadIdx.x < kSlots * kBoundWords) sh[threadIdx.x] = word_init(threadIdx.x % kBoundWords);
    const int r0 = group_min_rank(r, &shR);
    float v[kBoundWords / 2] = {};
    bool lower = false;
    if (r >= 0) {
        const uint32_t t = idx[p];
        const float4 lo = box[2 * t], hi = box[2 * t + 1];
        v[0] = v[3] = 0.5f * (lo.x + hi.x);
        v[1] = v[4] = 0.5f * (lo.y + hi.y);
        v[2] = v[5] = 0.5f * (lo.z + hi.z);
        v[6] = lo.x, v[7] = lo.y, v[8] = lo.z;
        v[9] = hi.x, v[10] = hi.y, v[11] = hi.z;
        lower = p < static_cast<uint32_t>((static_cast<uint64_t>(splits[r].first) + splits[r].last) / 2);
    }
    // A wave inside one range and one half of it reduces its keys in registers; LDS atomics of all
    // lanes on the same words would be served one lane at a time.
    const uint64_t in = __ballot(r >= 0);
    if (in) {
        const int lead = __ffsll(static_cast<unsigned long long>(in)) - 1;
        const int rr = __shfl(r, lead), side = __shfl(lower ? 0 : 1, lead);
        const bool same = __ballot(r >= 0 && (r != rr || (lower ? 0 : 1) != side)) == 0;
        GroupAcc<kBoundWords> g{sh, r0, 0};
        if (same) {
            const uint32_t lane = threadIdx.x & 63u;
            u64 mine = 0;
#pragma unroll
            for (uint32_t w = 0; w < 12; ++w) {
                const u64 k = ((w / 3) & 1) == 0 ? wave_key<true>(v[w], r >= 0, p - lane) : wave_key<false>(v[w], r >= 0, p - lane);
                // words 6..11 are also the half's
                if (lane == w || (w >= 6 && lane == w + 6)) mine = k;
            }
            if (lane < 18) g.add(acc, rr, static_cast<int>(lane) + (lane >= 12 ? 6 * side : 0), &mine, 1);
        } else if (r >= 0) {
            u64 keys[12];
#pragma unroll
            for (int w = 0; w < 12; ++w) keys[w] = ((w / 3) & 1) == 0 ? key_min(v[w], p) : key_max(v[w], p);
            g.add(acc, r, 0, keys, 12);
            g.add(acc, r, lower ? 12 : 18, keys + 6, 6);
        }
    }
    group_flush<kBoundWords>(sh, r0, 0, acc);
}

// the bounds of range r as k_bvh_bounds left them
__device__ inline Params params_of(int r, const uint32_t *idx, const float4 *box, const u64 *acc) {
    const u64 *a = acc + static_cast<size_t>(r) * kAcc;
    float cLo[3], cHi[3], bLo[3], bHi[3];
    for (int k = 0; k < 3; ++k) {
        cLo[k] = decode(a[k], true, idx, box, 0, k);
        cHi[k] = decode(a[3 + k], false, idx, box, 0, k);
        bLo[k] = decode(a[6 + k], true, idx, box, 1, k);
        bHi[k] = decode(a[9 + k], false, idx, box, 2, k);
    }
    return make_params(cLo, cHi, bLo, bHi);
}

__global__ __launch_bounds__(256) void k_bvh_bin(uint32_t n, const uint32_t *idx, const int32_t *segOf,
                                                 const int32_t *segRank, const float4 *box, uint8_t *bucket, u64 *acc) {
    constexpr int NW = kBuckets * kBinWords;
    __shared__ u64 sh[kSlots * NW];
    __shared__ int shR;
    const uint32_t p = blockIdx.x * 256u + threadIdx.x;
    const int r = rank_of(p, n, segOf, segRank);
    for (int i = threadIdx.x; i < kSlots * NW; i += 256) sh[i] = word_init(kBoundWords + i % NW);
    const int r0 = group_min_rank(r, &shR);
    if (r >= 0) {
        const Params q = params_of(r, idx, box, acc);
        const uint32_t t = idx[p];
        const float4 lo = box[2 * t], hi = box[2 * t + 1];
        const float c = q.axis == 0 ? 0.5f * (lo.x + hi.x) : (q.axis == 1 ? 0.5f * (lo.y + hi.y) : 0.5f * (lo.z + hi.z));
        const uint32_t b = bucket_of(q, c);
        bucket[p] = static_cast<uint8_t>(b);
        const u64 keys[kBinWords] = {key_min(lo.x, p), key_min(lo.y, p), key_min(lo.z, p), key_max(hi.x, p),
                                     key_max(hi.y, p), key_max(hi.z, p), 1ull};
        GroupAcc<NW> g{sh, r0, kBoundWords};
        g.add(acc, r, kBoundWords + static_cast<int>(b) * kBinWords, keys, kBinWords);
    }
    group_flush<NW>(sh, r0, kBoundWords, acc);
}

// the sweep of one range per 16 lanes, the split point, its node, the next level's two ranges
__global__ __launch_bounds__(256) void k_bvh_choose(uint32_t nSplits, uint32_t level, const uint32_t *idx, const float4 *box,
                                                    const u64 *acc, Split *splits, restir_aabb_tree_node *tmp, uint8_t *levels,
                                                    Seg *next) {
    const uint32_t r = blockIdx.x * 16u + (threadIdx.x >> 4);
    if (r >= nSplits) return;
    const int b = threadIdx.x & 15, row = static_cast<int>(threadIdx.x & 48u);
    const u64 *a = acc + static_cast<size_t>(r) * kAcc;
    Bin left = bin_empty();
    if (b < kBuckets) {
        const u64 *w = a + kBoundWords + b * kBinWords;
        left.count = static_cast<uint32_t>(w[6]);
        if (left.count != 0)
            for (int k = 0; k < 3; ++k) {  // the bucket's fold starts from the empty box
                left.lo[k] = nv_min(FLT_MAX, decode(w[k], true, idx, box, 1, k));
                left.hi[k] = nv_max(-FLT_MAX, decode(w[3 + k], false, idx, box, 2, k));
            }
    }
    Bin right = left;
    const Params q = params_of(static_cast<int>(r), idx, box, acc);
    const int best = sah_sweep(left, right, q.parentArea);
    const int split = best < 0 ? 0 : best;
    Split sp = splits[r];
    uint32_t mid = sp.first + static_cast<uint32_t>(__shfl(static_cast<int>(left.count), row + split));
    const bool degenerate = mid == sp.first || mid == sp.last;
    if (degenerate) mid = static_cast<uint32_t>((static_cast<uint64_t>(sp.first) + sp.last) / 2);
    const uint32_t t = mid - 1;
    restir_aabb_tree_node &node = tmp[t];
    if (b == split) {
        if (degenerate) {
            float v[4][3];
            for (int h = 0; h < 4; ++h)  // left lo, left hi, right lo, right hi
                for (int k = 0; k < 3; ++k) v[h][k] = decode(a[12 + 3 * h + k], (h & 1) == 0, idx, box, (h & 1) ? 2 : 1, k);
            write_box(node.leftAabbMin, v[0]);
            write_box(node.leftAabbMax, v[1]);
            write_box(node.rightAabbMin, v[2]);
            write_box(node.rightAabbMax, v[3]);
        } else {
            const float zero[3] = {0.0f, 0.0f, 0.0f};
            write_box(node.leftAabbMin, best < 0 ? zero : left.lo);
            write_box(node.leftAabbMax, best < 0 ? zero : left.hi);
            write_box(node.rightAabbMin, best < 0 ? zero : right.lo);
            write_box(node.rightAabbMax, best < 0 ? zero : right.hi);
        }
        node._pad[0] = node._pad[1] = 0;
        levels[t] = static_cast<uint8_t>(level);
        set_child(tmp, sp.link, static_cast<int32_t>(t));
        sp.mid = mid;
        sp.bucket = static_cast<uint32_t>(split);
        sp.degenerate = degenerate ? 1u : 0u;
        splits[r] = sp;
        next[2 * r] = Seg{sp.first, mid, static_cast<int32_t>(2 * t), 0};
        next[2 * r + 1] = Seg{mid, sp.last, static_cast<int32_t>(2 * t + 1), 0};
    }
}

__device__ inline bool goes_left(const Split &sp, const uint8_t *bucket, uint32_t p) {
    return !sp.degenerate && bucket[p] <= sp.bucket;
}

// left primitives before each position in its block of kScanGroup positions, and the blocks' totals
__global__ __launch_bounds__(256) void k_bvh_left_count(uint32_t n, const int32_t *segOf, const int32_t *segRank,
                                                        const Split *splits, const uint8_t *bucket, uint32_t *before,
                                                        uint32_t *sums) {
    __shared__ uint32_t waveTotal[4];
    const uint32_t base = blockIdx.x * kScanGroup + threadIdx.x * 4u;
    uint32_t v[4], run = 0;
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) {
        const int r = rank_of(base + i, n, segOf, segRank);
        v[i] = run;
        if (r >= 0 && goes_left(splits[r], bucket, base + i)) ++run;
    }
    const uint32_t incl = rscan::wave_inclusive(run);
    const uint32_t w = threadIdx.x >> 6;
    if ((threadIdx.x & 63u) == 63u) waveTotal[w] = incl;
    __syncthreads();
    uint32_t off = incl - run;
    for (uint32_t k = 0; k < w; ++k) off += waveTotal[k];
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i)
        if (base + i < n) before[base + i] = off + v[i];
    if (threadIdx.x == 255) sums[blockIdx.x] = off + run;
}
// the same over all positions, once `sums` holds the totals' exclusive prefix sums
__device__ inline uint32_t left_before(const uint32_t *before, const uint32_t *sums, uint32_t p) {
    return before[p] + sums[p / kScanGroup];
}

// ptr[p]: the position whose placement position p copies (itself when final)
__global__ __launch_bounds__(256) void k_bvh_chain(uint32_t n, const int32_t *segOf, const int32_t *segRank,
                                                   const Split *splits, const uint8_t *bucket, const uint32_t *before,
                                                   const uint32_t *sums, uint32_t *ptr) {
    const uint32_t p = blockIdx.x * 256u + threadIdx.x;
    if (p >= n) return;
    const int r = rank_of(p, n, segOf, segRank);
    uint32_t q = p;
    if (r >= 0) {
        const Split sp = splits[r];
        if (goes_left(sp, bucket, p)) {
            const uint32_t g = sp.first + (left_before(before, sums, p) - left_before(before, sums, sp.first));
            q = g < p ? g : p;
        }
    }
    ptr[p] = q;
}

// Follows each position's chain to its end by pointer jumping in place, all rounds in one launch:
// ptr[p] always names a position further down p's chain, whatever the order in which the lanes' reads
// and writes land, and the chain ends at a position that names itself. While a lane jumps, the lanes
// whose positions it meets shorten the rest of its chain, so long chains take about log2 of their
// length. Each lane then places what its position holds in the level's new order, notes the
// position's range at the next level, and clears the accumulators of that level's ranges.
__global__ __launch_bounds__(256) void k_bvh_scatter(uint32_t n, uint32_t nSplits, const int32_t *segOf, const int32_t *segRank,
                                                     const Split *splits, const uint8_t *bucket, const uint32_t *before,
                                                     const uint32_t *sums, volatile uint32_t *ptr, const uint32_t *idx,
                                                     uint32_t *idxOut, int32_t *segOut, u64 *acc) {
    const uint32_t p = blockIdx.x * 256u + threadIdx.x;
    if (p >= n) return;
    // fewer words than positions: a split range has more than kSub of them
    static_assert(2 * kAcc < kSub, "a lane clears one word at most");
    if (p < 2 * nSplits * kAcc) acc[p] = word_init(static_cast<int>(p % kAcc));
    const int r = rank_of(p, n, segOf, segRank);
    if (r < 0) {
        idxOut[p] = idx[p];
        segOut[p] = -1;
        return;
    }
    const Split sp = splits[r];
    if (sp.degenerate) {
        idxOut[p] = idx[p];
        segOut[p] = 2 * r + (p >= sp.mid ? 1 : 0);
        return;
    }
    if (goes_left(sp, bucket, p)) {
        const uint32_t q = sp.first + (left_before(before, sums, p) - left_before(before, sums, sp.first));
        idxOut[q] = idx[p];
        segOut[q] = 2 * r;
    }
    uint32_t q = ptr[p];
    for (;;) {
        const uint32_t f = ptr[q];
        if (f == q) break;
        ptr[p] = f;
        q = f;
    }
    if (p >= sp.mid) {
        idxOut[p] = idx[q];
        segOut[p] = 2 * r + 1;
    }
}

// A subtree of at most kSub primitives, level by level, in one workgroup: 16 lanes take a range at a
// time. Bounds: a lane per component folds the primitives in order; bins: a lane per bucket; then the
// sweep of k_bvh_choose and the partition, 16 positions at a time: the chains of a position lead to
// earlier ones, which are resolved already. Everything is read and written in LDS but the nodes.
// Only order within a fold matters, and each fold is one lane's. Bound by the chain of levels: a
// 512-primitive range takes 512 steps of its first fold, its children half of that, and so on.
struct SubQueue {
    uint16_t first, last;
    int32_t link;
};
// a node's four boxes as 16 words
__device__ inline float *box_words(restir_aabb_tree_node &node) { return reinterpret_cast<float *>(&node); }
__global__ __launch_bounds__(256) void k_bvh_subtrees(const Sub *subs, const uint32_t *idx, const float4 *box,
                                                      restir_aabb_tree_node *tmp, uint8_t *levels, Info *info) {
    __shared__ float bx[kSub * 6];
    __shared__ uint32_t prim[kSub];
    __shared__ uint16_t order[2][kSub], ptr[kSub];
    __shared__ uint8_t bucket[kSub];
    __shared__ u64 bins[16][kBuckets * kBinWords];
    __shared__ SubQueue queue[2][kSub / 2];
    __shared__ uint32_t queued[2];
    const Sub sub = subs[blockIdx.x];
    const uint32_t n = sub.last - sub.first;
    for (uint32_t i = threadIdx.x; i < n; i += 256u) {
        const uint32_t t = idx[sub.first + i];
        const float4 lo = box[2 * t], hi = box[2 * t + 1];
        prim[i] = t;
        order[0][i] = static_cast<uint16_t>(i);
        bx[6 * i] = lo.x, bx[6 * i + 1] = lo.y, bx[6 * i + 2] = lo.z;
        bx[6 * i + 3] = hi.x, bx[6 * i + 4] = hi.y, bx[6 * i + 5] = hi.z;
    }
    if (threadIdx.x == 0) {
        queue[0][0] = SubQueue{0, static_cast<uint16_t>(n), sub.link};
        queued[0] = 1;
        queued[1] = 0;
    }
    __syncthreads();
    const uint32_t L = threadIdx.x & 15u;
    const int row = static_cast<int>(threadIdx.x & 48u);
    uint32_t level = sub.level;
    for (uint32_t cur = 0;; cur ^= 1u, ++level) {
        const uint32_t count = queued[cur];
        const uint16_t *ord = order[cur];
        uint16_t *out = order[cur ^ 1u];
        for (uint32_t i = threadIdx.x >> 4; i < count; i += 16u) {
            const uint32_t f = queue[cur][i].first, l = queue[cur][i].last;
            const int32_t link = queue[cur][i].link;
            if (l - f == 2) {  // a pair of leaves
                const uint32_t a = ord[f], b = ord[f + 1], t = sub.first + f;
                restir_aabb_tree_node &node = tmp[t];
                const uint32_t o = L < 8 ? a : b;
                box_words(node)[L] = (L & 3u) == 3u ? 1.0f : bx[6 * o + ((L >> 2) & 1u) * 3 + (L & 3u)];
                if (L == 0) {
                    node.leftChild = ~static_cast<int32_t>(prim[a]);
                    node.rightChild = ~static_cast<int32_t>(prim[b]);
                    node._pad[0] = node._pad[1] = 0;
                    levels[t] = static_cast<uint8_t>(level);
                    set_child(tmp, link, static_cast<int32_t>(t));
                }
                continue;
            }
            float cLo[3], cHi[3], bLo[3], bHi[3];
            const bool wide = l - f > kSubWide;
            if (wide) {  // a lane per sixteenth of the primitives, then the lanes' folds in order
                float v[12];
#pragma unroll
                for (int w = 0; w < 12; ++w) v[w] = ((w / 3) & 1) ? -INFINITY : INFINITY;
                const uint32_t each = (l - f + 15u) / 16u, from = f + L * each, to = from + each < l ? from + each : l;
#pragma unroll 4
                for (uint32_t p = from; p < to; ++p) {
                    const float *e = bx + 6u * ord[p];
#pragma unroll
                    for (int c = 0; c < 3; ++c) {
                        const float lo = e[c], hi = e[c + 3], mid = 0.5f * (lo + hi);
                        v[c] = nv_min(v[c], mid);
                        v[3 + c] = nv_max(v[3 + c], mid);
                        v[6 + c] = nv_min(v[6 + c], lo);
                        v[9 + c] = nv_max(v[9 + c], hi);
                    }
                }
#pragma unroll
                for (int w = 0; w < 12; ++w) {
                    if ((w / 3) & 1) {
                        v[w] = nv_max(v[w], row_shl<1>(-INFINITY, v[w]));
                        v[w] = nv_max(v[w], row_shl<2>(-INFINITY, v[w]));
                        v[w] = nv_max(v[w], row_shl<4>(-INFINITY, v[w]));
                        v[w] = nv_max(v[w], row_shl<8>(-INFINITY, v[w]));
                    } else {
                        v[w] = nv_min(v[w], row_shl<1>(INFINITY, v[w]));
                        v[w] = nv_min(v[w], row_shl<2>(INFINITY, v[w]));
                        v[w] = nv_min(v[w], row_shl<4>(INFINITY, v[w]));
                        v[w] = nv_min(v[w], row_shl<8>(INFINITY, v[w]));
                    }
                    v[w] = __shfl(v[w], row);
                }
#pragma unroll
                for (int c = 0; c < 3; ++c) cLo[c] = v[c], cHi[c] = v[3 + c], bLo[c] = v[6 + c], bHi[c] = v[9 + c];
            } else {
                // lanes 0..2 centroid lo, 3..5 centroid hi, 6..8 box lo, 9..11 box hi
                const uint32_t k = L % 3u, kind = L / 3u;
                float v = (kind & 1u) ? -INFINITY : INFINITY;
                for (uint32_t p = f; p < l; p += 8u) {  // beyond the end: the last one again, which changes nothing
                    float x[8];
#pragma unroll
                    for (uint32_t e = 0; e < 8; ++e) {
                        const uint32_t o = 6u * ord[p + e < l ? p + e : l - 1] + k;
                        const float lo = bx[o], hi = bx[o + 3];
                        x[e] = kind < 2u ? 0.5f * (lo + hi) : kind == 2u ? lo : hi;
                    }
#pragma unroll
                    for (uint32_t e = 0; e < 8; ++e) v = (kind & 1u) ? nv_max(v, x[e]) : nv_min(v, x[e]);
                }
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    cLo[c] = __shfl(v, row + c);
                    cHi[c] = __shfl(v, row + 3 + c);
                    bLo[c] = __shfl(v, row + 6 + c);
                    bHi[c] = __shfl(v, row + 9 + c);
                }
            }
            const Params q = make_params(cLo, cHi, bLo, bHi);
            Bin left = bin_empty();
            if (wide) {  // keys as in k_bvh_bin
                u64 *a = bins[threadIdx.x >> 4];
                for (uint32_t w = L; w < kBuckets * kBinWords; w += 16u) a[w] = word_init(kBoundWords + static_cast<int>(w));
                rk::wave_sync();
                for (uint32_t p = f + L; p < l; p += 16u) {
                    const float *e = bx + 6u * ord[p];
                    const uint32_t b = bucket_of(q, 0.5f * (e[q.axis] + e[q.axis + 3]));
                    bucket[p] = static_cast<uint8_t>(b);
                    u64 *w = a + b * kBinWords;
#pragma unroll
                    for (int c = 0; c < 3; ++c) {
                        atomicMin(&w[c], key_min(e[c], p));
                        atomicMax(&w[3 + c], key_max(e[3 + c], p));
                    }
                    atomicAdd(&w[6], 1ull);
                }
                rk::wave_sync();
                if (L < kBuckets) left.count = static_cast<uint32_t>(a[L * kBinWords + 6]);
                if (left.count != 0)
#pragma unroll
                    for (int c = 0; c < 3; ++c) {
                        const u64 lo = a[L * kBinWords + c], hi = a[L * kBinWords + 3 + c];
                        const float vl = uncode(static_cast<uint32_t>(lo >> 32)), vh = uncode(static_cast<uint32_t>(hi >> 32));
                        left.lo[c] = nv_min(FLT_MAX, vl != 0.0f ? vl : bx[6u * ord[~static_cast<uint32_t>(lo)] + c]);
                        left.hi[c] = nv_max(-FLT_MAX, vh != 0.0f ? vh : bx[6u * ord[static_cast<uint32_t>(hi)] + 3 + c]);
                    }
            } else {
                for (uint32_t p = f + L; p < l; p += 16u) {
                    const uint32_t o = 6u * ord[p] + static_cast<uint32_t>(q.axis);
                    bucket[p] = static_cast<uint8_t>(bucket_of(q, 0.5f * (bx[o] + bx[o + 3])));
                }
                rk::wave_sync();
                // a lane per bucket
                for (uint32_t p = f; p < l; p += 4u) {
                    float x[4][6];
                    bool mine[4];
#pragma unroll
                    for (uint32_t e = 0; e < 4; ++e) {
                        const uint32_t at = p + e < l ? p + e : l - 1, o = 6u * ord[at];
                        mine[e] = p + e < l && bucket[at] == L;
#pragma unroll
                        for (int c = 0; c < 6; ++c) x[e][c] = bx[o + c];
                    }
#pragma unroll
                    for (uint32_t e = 0; e < 4; ++e) {
                        // read in any case, so that the loads of all four are under way together: left
                        // alone the compiler puts each behind a branch on its bucket
#pragma unroll
                        for (int c = 0; c < 6; ++c) asm volatile("" : "+v"(x[e][c]));
                        left.count += mine[e] ? 1u : 0u;
#pragma unroll
                        for (int c = 0; c < 3; ++c) {
                            left.lo[c] = mine[e] ? nv_min(left.lo[c], x[e][c]) : left.lo[c];
                            left.hi[c] = mine[e] ? nv_max(left.hi[c], x[e][3 + c]) : left.hi[c];
                        }
                    }
                }
            }
            Bin right = left;
            const int best = sah_sweep(left, right, q.parentArea);
            const uint32_t split = best < 0 ? 0u : static_cast<uint32_t>(best);
            uint32_t mid = f + static_cast<uint32_t>(__shfl(static_cast<int>(left.count), row + static_cast<int>(split)));
            const bool degenerate = mid == f || mid == l;
            if (degenerate) mid = (f + l) / 2;
            const uint32_t t = sub.first + mid - 1;
            restir_aabb_tree_node &node = tmp[t];
            if (degenerate) {
                // a lane per component of the halves' boxes, in the node's order; w = 1
                const uint32_t c = L & 3u, from = L < 8u ? f : mid, to = L < 8u ? mid : l;
                float x = 1.0f;
                if (c < 3u)
                    for (uint32_t p = from; p < to; ++p) {
                        const float e = bx[6u * ord[p] + ((L >> 2) & 1u) * 3 + c];
                        x = p == from ? e : ((L >> 2) & 1u) ? nv_max(x, e) : nv_min(x, e);
                    }
                box_words(node)[L] = x;
                for (uint32_t p = f + L; p < l; p += 16u) out[p] = ord[p];
            } else {
                if (L == split) {
                    const float zero[3] = {0.0f, 0.0f, 0.0f};
                    write_box(node.leftAabbMin, best < 0 ? zero : left.lo);
                    write_box(node.leftAabbMax, best < 0 ? zero : left.hi);
                    write_box(node.rightAabbMin, best < 0 ? zero : right.lo);
                    write_box(node.rightAabbMax, best < 0 ? zero : right.hi);
                }
                uint32_t run = f;  // the next left primitive's place
                for (uint32_t p0 = f; p0 < l; p0 += 16u) {
                    const uint32_t p = p0 + L;
                    const bool in = p < l, goes = in && bucket[p] <= split;
                    const uint32_t m = static_cast<uint32_t>(__ballot(goes) >> row) & 0xffffu;
                    const uint32_t g = run + static_cast<uint32_t>(__popc(m & ((1u << L) - 1u)));
                    uint32_t at = p;
                    if (goes) {
                        out[g] = ord[p];
                        at = g < p ? g : p;
                    }
                    if (in) ptr[p] = static_cast<uint16_t>(at);
                    rk::wave_sync();
                    if (in)
                        for (uint32_t to = ptr[at]; to != at; to = ptr[at]) at = to;
                    rk::wave_sync();
                    if (in) {
                        ptr[p] = static_cast<uint16_t>(at);
                        if (p >= mid) out[p] = ord[at];
                    }
                    run += static_cast<uint32_t>(__popc(m));
                }
            }
            rk::wave_sync();
            if (L == 0) {
                node._pad[0] = node._pad[1] = 0;
                levels[t] = static_cast<uint8_t>(level);
                set_child(tmp, link, static_cast<int32_t>(t));
            }
            if (L < 2) {
                const uint32_t a = L == 0 ? f : mid, b = L == 0 ? mid : l;
                const int32_t to = static_cast<int32_t>(2 * t + L);
                if (b - a == 1) set_child(tmp, to, ~static_cast<int32_t>(prim[out[a]]));
                else queue[cur ^ 1u][atomicAdd(&queued[cur ^ 1u], 1u)] = SubQueue{static_cast<uint16_t>(a), static_cast<uint16_t>(b), to};
            }
        }
        __syncthreads();
        if (queued[cur ^ 1u] == 0) break;
        __syncthreads();
        if (threadIdx.x == 0) queued[cur] = 0;
        __syncthreads();
    }
    if (threadIdx.x == 0) atomicMax(&info->depth, level);
}

// Breadth-first ids: the temporary nodes, sorted by level, in their order within one. Nodes of each
// level in each block of 256 ...
__global__ __launch_bounds__(256) void k_bvh_level_counts(uint32_t nNodes, uint32_t depth, const uint8_t *levels,
                                                          uint32_t *counts) {
    __shared__ uint32_t sh[64];
    const uint32_t t = blockIdx.x * 256u + threadIdx.x;
    if (threadIdx.x < 64) sh[threadIdx.x] = 0;
    __syncthreads();
    if (t < nNodes) atomicAdd(&sh[levels[t] - 1u], 1u);
    __syncthreads();
    if (threadIdx.x < depth) counts[threadIdx.x * gridDim.x + blockIdx.x] = sh[threadIdx.x];
}
// ... then, from their exclusive prefix sums (level after level), each node's id.
__global__ __launch_bounds__(256) void k_bvh_ids(uint32_t nNodes, const uint8_t *levels, const uint32_t *counts, uint32_t *ids) {
    __shared__ uint32_t sh[4][64];
    const uint32_t t = blockIdx.x * 256u + threadIdx.x, wave = threadIdx.x >> 6, lane = threadIdx.x & 63u;
    sh[wave][lane] = 0;
    __syncthreads();
    const uint32_t l = t < nNodes ? levels[t] - 1u : 0u;
    uint64_t same = __ballot(t < nNodes);
#pragma unroll
    for (int b = 0; b < 6; ++b) {
        const uint64_t m = __ballot((l >> b) & 1u);
        same &= ((l >> b) & 1u) ? m : ~m;
    }
    const uint32_t before = static_cast<uint32_t>(__popcll(same & ((1ull << lane) - 1ull)));
    if (t < nNodes && before == 0) sh[wave][l] = static_cast<uint32_t>(__popcll(same));
    __syncthreads();
    if (t >= nNodes) return;
    uint32_t id = counts[l * gridDim.x + blockIdx.x] + before;
    for (uint32_t w = 0; w < wave; ++w) id += sh[w][l];
    ids[t] = id;
}
__global__ __launch_bounds__(256) void k_bvh_write(uint32_t nNodes, const restir_aabb_tree_node *tmp, const uint32_t *ids,
                                                   restir_aabb_tree_node *nodes) {
    const uint32_t t = blockIdx.x * 256u + threadIdx.x;
    if (t >= nNodes) return;
    restir_aabb_tree_node node = tmp[t];
    if (node.leftChild >= 0) node.leftChild = static_cast<int32_t>(ids[node.leftChild]);
    if (node.rightChild >= 0) node.rightChild = static_cast<int32_t>(ids[node.rightChild]);
    nodes[ids[t]] = node;
}

inline uint32_t groups(uint64_t n) { return static_cast<uint32_t>((n + 255) / 256); }

inline size_t align_up(size_t x) { return (x + 255) & ~static_cast<size_t>(255); }

struct Layout {
    size_t box, idx0, idx1, seg0, seg1, bucket, before, ptr, temp32, segs0, segs1, segRank, splits, subs, acc, tmp, levels,
        counts, info, total;
};

Layout layout(uint32_t n) {
    const size_t maxSplits = n / (kSub + 1) + 1, maxSegs = 2 * maxSplits + 1;
    const size_t sums = (static_cast<size_t>(n) + kScanGroup - 1) / kScanGroup, counts = 64ull * groups(n);
    Layout L{};
    size_t o = 0;
    auto take = [&o](size_t bytes) {
        const size_t at = o;
        o = align_up(o + bytes);
        return at;
    };
    L.box = take(sizeof(float4) * 2 * n);
    L.idx0 = take(4ull * n);
    L.idx1 = take(4ull * n);
    L.seg0 = take(4ull * n);
    L.seg1 = take(4ull * n);
    L.bucket = take(n);
    L.before = take(4ull * n);
    L.ptr = take(4ull * n);  // then the nodes' ids
    L.temp32 = take(4 * (sums + rscan::temp_items(static_cast<uint32_t>(sums)) + rscan::temp_items(static_cast<uint32_t>(counts))));
    L.segs0 = take(sizeof(Seg) * maxSegs);
    L.segs1 = take(sizeof(Seg) * maxSegs);
    L.segRank = take(4 * maxSegs);
    L.splits = take(sizeof(Split) * maxSplits);
    L.subs = take(sizeof(Sub) * (n / 2 + 1));
    L.acc = take(8ull * kAcc * (2 * maxSplits));
    L.tmp = take(sizeof(restir_aabb_tree_node) * n);
    L.levels = take(n);
    L.counts = take(4 * counts);
    L.info = take(sizeof(Info));
    L.total = o;
    return L;
}

}  // namespace

// ------------------------------------------------------------ 4-entry nodes of a bound tree --
namespace {

__device__ inline bool finite_box(float4 mn, float4 mx) {
    constexpr float kInf = __builtin_huge_valf();
    return fabsf(mn.x) < kInf && fabsf(mn.y) < kInf && fabsf(mn.z) < kInf && fabsf(mx.x) < kInf &&
           fabsf(mx.y) < kInf && fabsf(mx.z) < kInf && mn.x <= mx.x && mn.y <= mx.y && mn.z <= mx.z;
}
__device__ inline float box_max(float4 v) { return fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fabsf(v.z)); }
__device__ inline bool inside(float4 mn, float4 mx, float4 outerMn, float4 outerMx) {
    return outerMn.x <= mn.x && outerMn.y <= mn.y && outerMn.z <= mn.z && mx.x <= outerMx.x &&
           mx.y <= outerMx.y && mx.z <= outerMx.z;
}

// One thread per reference node x: its WNode (see rt_traverse.h), and the check that both boxes
// stored in x are finite and ordered and that each internal child's two boxes lie inside the box
// x stores for it (info[0] != 0 otherwise). Every box is stored in exactly one node, so the
// threads together check every box and every parent-child pair; info[1] gets the bits of the
// largest |coordinate| of any box (non-negative floats order as their bit patterns; a NaN orders
// above every number).
// It also writes the parent slot (2 node + side) of each internal child (unless parent is null), and
// sets info[2] when a box is not finite and ordered, info[3] when a leaf's box is not the bounding box
// of its triangle.
__global__ __launch_bounds__(256) void k_wide_build(const rt::Node *__restrict__ nodes, uint32_t nNodes,
                                                    const float4 *__restrict__ tris,
                                                    rt::WNode *__restrict__ wide, uint32_t *__restrict__ parent,
                                                    uint32_t *__restrict__ info) {
    const uint32_t x = blockIdx.x * 256u + threadIdx.x;
    if (x >= nNodes) return;
    const rt::Node b = rt::load_node(nodes, static_cast<int32_t>(x));
    bool ok = finite_box(b.lmin, b.lmax) && finite_box(b.rmin, b.rmax);
    if (!ok) atomicOr(&info[2], 1u);
    bool tight = true;
    float4 mn[4], mx[4];
    int32_t id[4], grp[2];
    for (int side = 0; side < 2; ++side) {
        const int32_t c = side ? b.right : b.left;
        const float4 smn = side ? b.rmin : b.lmin, smx = side ? b.rmax : b.lmax;
        if (c < 0) {
            mn[2 * side] = smn;
            mx[2 * side] = smx;
            id[2 * side] = c;
            mn[2 * side + 1] = mx[2 * side + 1] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            id[2 * side + 1] = rt::kNoEntry;
            grp[side] = -1;
            const float4 *t = tris + 3 * static_cast<size_t>(~c);
            const float4 v0 = t[0], v1 = t[1], v2 = t[2];
            tight = tight && smn.x == fminf(fminf(v0.x, v1.x), v2.x) && smn.y == fminf(fminf(v0.y, v1.y), v2.y) &&
                    smn.z == fminf(fminf(v0.z, v1.z), v2.z) && smx.x == fmaxf(fmaxf(v0.x, v1.x), v2.x) &&
                    smx.y == fmaxf(fmaxf(v0.y, v1.y), v2.y) && smx.z == fmaxf(fmaxf(v0.z, v1.z), v2.z);
        } else {
            if (parent) parent[c] = 2u * x + static_cast<uint32_t>(side);
            const rt::Node cn = rt::load_node(nodes, c);
            mn[2 * side] = cn.lmin;
            mx[2 * side] = cn.lmax;
            id[2 * side] = cn.left;
            mn[2 * side + 1] = cn.rmin;
            mx[2 * side + 1] = cn.rmax;
            id[2 * side + 1] = cn.right;
            grp[side] = c;
            ok = ok && inside(cn.lmin, cn.lmax, smn, smx) && inside(cn.rmin, cn.rmax, smn, smx);
        }
    }
    float4 *o = reinterpret_cast<float4 *>(wide + x);
    o[0] = make_float4(mn[0].x, mn[1].x, mn[2].x, mn[3].x);
    o[1] = make_float4(mn[0].y, mn[1].y, mn[2].y, mn[3].y);
    o[2] = make_float4(mn[0].z, mn[1].z, mn[2].z, mn[3].z);
    o[3] = make_float4(mx[0].x, mx[1].x, mx[2].x, mx[3].x);
    o[4] = make_float4(mx[0].y, mx[1].y, mx[2].y, mx[3].y);
    o[5] = make_float4(mx[0].z, mx[1].z, mx[2].z, mx[3].z);
    reinterpret_cast<int4 *>(o)[6] = make_int4(id[0], id[1], id[2], id[3]);
    // entry masks: bit k set when entry k exists, bit 4 + k when it is a triangle leaf
    uint32_t masks = 0;
    for (int k = 0; k < 4; ++k) {
        if (id[k] != rt::kNoEntry) masks |= 1u << k;
        if (id[k] != rt::kNoEntry && id[k] < 0) masks |= 16u << k;
    }
    reinterpret_cast<int4 *>(o)[7] = make_int4(grp[0], grp[1], static_cast<int32_t>(masks), 0);
    if (!ok) atomicOr(&info[0], 1u);
    if (!tight) atomicOr(&info[3], 1u);
    const float m = fmaxf(fmaxf(fmaxf(box_max(b.lmin), box_max(b.lmax)), box_max(b.rmin)), box_max(b.rmax));
    const bool nan = b.lmin.x != b.lmin.x || b.lmin.y != b.lmin.y || b.lmin.z != b.lmin.z || b.lmax.x != b.lmax.x ||
                     b.lmax.y != b.lmax.y || b.lmax.z != b.lmax.z || b.rmin.x != b.rmin.x || b.rmin.y != b.rmin.y ||
                     b.rmin.z != b.rmin.z || b.rmax.x != b.rmax.x || b.rmax.y != b.rmax.y || b.rmax.z != b.rmax.z;
    atomicMax(&info[1], nan ? 0x7fc00000u : __float_as_uint(m));
}

// ---- 8-entry nodes (rt_wide8.h), collapsed top-down from the binary tree, one level of 8-entry
// nodes per launch: 8 lanes make one node, an entry each. The entries start as the two sides of the
// binary node; while fewer than 8, the largest internal entry (by box area) is replaced by its own two
// sides. Children of one node are consecutive; the order of the nodes of a level is the order of
// the atomics and changes no answer. One triangle per leaf entry: groups of up to 2, 3 and 4 made
// the tracer 0-1%, 5% and 12% slower (more triangle tests than boxes saved). Latency bound (a node's
// expansions wait for one node after another): a lane per node, which
// chose, ordered and rounded its entries one after another, took the builds of 1,200, 136,000 and 2.3
// million triangles 0.49, 1.25 and 6.62 ms, this 0.39, 1.06 and 6.40.
constexpr int kW8Levels = rt::kW8Stack + 1;
// Trees of at most this many nodes (1,120 triangles) take one launch: a launch a level took 300 triangles
// 101 us to bind, 1,000 103, this 70 and 94; 1,200 triangles 104 and 106, 2,000 116 and 130.
constexpr uint32_t kW8OneGroup = 640;
struct W8Info {
    uint32_t nodes[kW8Levels + 1];  // nodes per level; [0] = 1
    uint32_t tris, overflow;
};

// kAll: all levels, `levels` at most, by one workgroup. Else level `level0` alone.
template <bool kAll>
__global__ __launch_bounds__(512) void k_w8_collapse(const rt::Node *__restrict__ nodes,
                                                     const float4 *__restrict__ tris, uint32_t level0,
                                                     uint32_t levels, uint32_t maxNodes, uint32_t maxTris,
                                                     const uint32_t *__restrict__ bounds, rt::W8Node *__restrict__ out,
                                                     float4 *__restrict__ outTris, uint32_t *__restrict__ work,
                                                     W8Info *__restrict__ info) {
    __shared__ __align__(16) rt::W8Node made[64];
    __shared__ uint2 reserve[9];
    __shared__ uint32_t below, spilled;  // kAll: nodes of the next level; whether a node found no room
    const uint32_t lane = threadIdx.x & 63u, k = lane & 7u;
    const int row = static_cast<int>(lane & 56u);
    const float maxCoord = __uint_as_float(bounds[1]);
    const double grow = static_cast<double>(rt::kW8Grow) * static_cast<double>(maxCoord);
    // A box is not finite, or too large or small: no 8-entry nodes. Areas are finite in this range; from about
    // 1.7e38 on a flat box's would be inf * 0, and no lane's NaN agrees with another's choice. Nor is there
    // anything to do below a level that found no room: not every node counted there has its work entry. The
    // three words are read together, one wait for all.
    const uint32_t spilledAbove = kAll ? 0u : info->overflow;
    if ((bounds[2] | spilledAbove) != 0 || !rt::w8_covers(maxCoord)) return;
    uint32_t begin = 0, n = 1;
    if (!kAll) {
        for (uint32_t l = 0; l < level0; ++l) begin += info->nodes[l];
        n = info->nodes[level0];
    }
    for (uint32_t level = level0; n != 0; ++level) {
    const uint32_t next = begin + n;
    if (kAll && threadIdx.x == 0) below = spilled = 0;  // read before the last barrier
    for (uint32_t i0 = blockIdx.x * 64u; i0 < n; i0 += gridDim.x * 64u) {
        const uint32_t i = i0 + (threadIdx.x >> 3), me = begin + i;
        const bool on = i < n && me < maxNodes;  // the same for a node's 8 lanes
        uint32_t cnt = 0;
        float mn[3] = {}, mx[3] = {};  // this lane's entry: its box,
        int32_t ref = 0;               // >= 0 internal node, < 0 ~triangle,
        uint32_t slot = 0;             // where it is stored: 2 node + side,
        float area = -2.0f;            // and its box's area, -2 unless it is internal
        const auto put = [&](float4 lo, float4 hi, int32_t c, uint32_t from) {
            mn[0] = lo.x, mn[1] = lo.y, mn[2] = lo.z;
            mx[0] = hi.x, mx[1] = hi.y, mx[2] = hi.z;
            const float sx = hi.x - lo.x, sy = hi.y - lo.y, sz = hi.z - lo.z;
            area = c >= 0 ? sx * sy + sx * sz + sy * sz : -2.0f;
            ref = c;
            slot = from;
        };
        if (on) {
            int32_t x = level == 0 ? 0 : static_cast<int32_t>(work[me]);
            uint32_t at = 0;
            for (;;) {  // entry `at` becomes the left side of node x, a new entry its right side
                const rt::Node nd = rt::load_node(nodes, x);
                const uint32_t add = cnt == 0 ? 1u : cnt;
                if (k == at) put(nd.lmin, nd.lmax, nd.left, 2u * static_cast<uint32_t>(x));
                if (k == add) put(nd.rmin, nd.rmax, nd.right, 2u * static_cast<uint32_t>(x) + 1u);
                cnt = add + 1u;
                if (cnt == 8) break;
                float best = area;  // the first of the largest
                at = k;
#pragma unroll
                for (int d = 1; d < 8; d <<= 1) {
                    const float v = __shfl_xor(best, d);
                    const uint32_t o = static_cast<uint32_t>(__shfl_xor(static_cast<int>(at), d));
                    if (v > best || (v == best && o < at)) {
                        best = v;
                        at = o;
                    }
                }
                if (best == -2.0f) break;
                x = __shfl(ref, row + static_cast<int>(at));
            }
        }
        const bool internal = k < cnt && ref >= 0, leaf = k < cnt && ref < 0;
        const uint32_t intMask = static_cast<uint32_t>(__ballot(internal) >> row) & 0xffu;
        const uint32_t triMask = static_cast<uint32_t>(__ballot(leaf) >> row) & 0xffu;
        const uint32_t nInt = static_cast<uint32_t>(__popc(intMask)), nTri = static_cast<uint32_t>(__popc(triMask));
        // slots: internal entries first, then the triangles.
        // The internal entries along the axis on which their centres spread most, the largest
        // centre first: the primary rays take them from the side they come from. The shadow rays
        // take them in this order (1-11% faster on the terrains than the other way round)
        uint32_t axis = 0;
        float spread = -1.0f;
#pragma unroll
        for (uint32_t a = 0; a < 3; ++a) {
            const float c = mn[a] + mx[a];
            float lo = internal ? c : __builtin_huge_valf(), hi = internal ? c : -__builtin_huge_valf();
#pragma unroll
            for (int d = 1; d < 8; d <<= 1) {
                lo = fminf(lo, __shfl_xor(lo, d));
                hi = fmaxf(hi, __shfl_xor(hi, d));
            }
            if (hi - lo > spread) {
                spread = hi - lo;
                axis = a;
            }
        }
        const float centre = axis == 0 ? mn[0] + mx[0] : axis == 1 ? mn[1] + mx[1] : mn[2] + mx[2];
        uint32_t rank = k;  // an empty entry keeps its place at the end
        if (leaf) rank = nInt + static_cast<uint32_t>(__popc(triMask & ((1u << k) - 1u)));
        uint32_t before = 0;
#pragma unroll
        for (uint32_t o = 0; o < 8; ++o) {
            const float c = __shfl(centre, row + static_cast<int>(o));
            if (((intMask >> o) & 1u) && (c > centre || (c == centre && o < k))) ++before;
        }
        if (internal) rank = before;
        // room in the next level and among the triangles, one atomic pair per workgroup (an atomic is
        // served in 11 ns: one per wave, of 8 nodes, made 2.3 million triangles 0.7 ms slower)
        const uint32_t inclInt = rscan::wave_inclusive(k == 0 ? nInt : 0u);
        const uint32_t inclTri = rscan::wave_inclusive(k == 0 ? nTri : 0u);
        const uint32_t wave = threadIdx.x >> 6;
        if (lane == 63) reserve[wave] = make_uint2(inclInt, inclTri);
        __syncthreads();
        if (threadIdx.x == 0) {
            uint2 sum = make_uint2(0u, 0u);
            for (uint32_t v = 0; v < 8; ++v) {
                const uint2 t = reserve[v];
                reserve[v] = sum;
                sum.x += t.x;
                sum.y += t.y;
            }
            if (kAll) below += sum.x;
            if (sum.x) sum.x = atomicAdd(&info->nodes[level + 1], sum.x);
            if (sum.y) sum.y = atomicAdd(&info->tris, sum.y);
            reserve[8] = sum;
        }
        __syncthreads();
        const uint32_t baseInt = next + reserve[8].x + reserve[wave].x + inclInt - nInt;
        const uint32_t baseTri = reserve[8].y + reserve[wave].y + inclTri - nTri;
        if (!on) continue;
        if (baseInt + nInt > maxNodes || baseTri + nTri > maxTris) {
            if (k == 0) atomicOr(&info->overflow, 1u);
            if (kAll) spilled = 1;
            continue;
        }
        if (internal) work[baseInt + rank] = static_cast<uint32_t>(ref);
        // per axis, by a lane each: the origin p below the node's planes, and e, the smallest step 2^e
        // (down to 2^-100) whose 2047 multiples span the node
        float least[3], most[3];
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            least[a] = k < cnt ? mn[a] : __builtin_huge_valf();
            most[a] = k < cnt ? mx[a] : -__builtin_huge_valf();
#pragma unroll
            for (int d = 1; d < 8; d <<= 1) {
                least[a] = fminf(least[a], __shfl_xor(least[a], d));
                most[a] = fmaxf(most[a], __shfl_xor(most[a], d));
            }
        }
        const double lo = static_cast<double>(k == 0 ? least[0] : k == 1 ? least[1] : least[2]) - grow;
        const double hi = static_cast<double>(k == 0 ? most[0] : k == 1 ? most[1] : most[2]) + grow;
        float p = static_cast<float>(lo);
        if (static_cast<double>(p) > lo) p = nextafterf(p, -__builtin_huge_valf());
        const double ext = hi - static_cast<double>(p);
        int e = -100;
        if (ext > 0.0) {
            const int f = ilogb(ext) - 11;
            if (f > e) e = f;
        }
        while (ext > 2047.0 * ldexp(1.0, e)) ++e;
        rt::W8Node &w = made[threadIdx.x >> 3];
        uint32_t exps = (((1u << cnt) - 1u) & ~((1u << nInt) - 1u)) << 24;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            const float pa = __shfl(p, row + a);
            const int ea = __shfl(e, row + a);
            exps |= (static_cast<uint32_t>(ea) & 0xffu) << (8 * a);
            const double inv = ldexp(1.0, -ea);
            double ql = 0.0, qh = 0.0;
            if (k < cnt) {
                ql = floor((static_cast<double>(mn[a]) - grow - static_cast<double>(pa)) * inv);
                qh = ceil((static_cast<double>(mx[a]) + grow - static_cast<double>(pa)) * inv);
                ql = fmin(fmax(ql, 0.0), 2047.0);
                qh = fmin(fmax(qh, 0.0), 2047.0);
            }
            w.plane[a][0][rank] = __builtin_bit_cast(uint16_t, static_cast<_Float16>(static_cast<float>(ql)));
            w.plane[a][1][rank] = __builtin_bit_cast(uint16_t, static_cast<_Float16>(static_cast<float>(qh)));
            if (k == 0) w.p[a] = pa;
        }
        if (k == 0) {
            w.child = (baseInt << 8) | ((1u << nInt) - 1u);
            w.triBase = baseTri - nInt;
            w.exps = exps;
            w.axis = axis;
            w.pad = 0;
        }
        rk::wave_sync();
        // the node by way of LDS: 16 bytes a lane
        static_assert(sizeof(rt::W8Node) == 128, "8 lanes store a node");
        reinterpret_cast<float4 *>(out + me)[k] = reinterpret_cast<const float4 *>(&w)[k];
        rk::wave_sync();
        if (leaf) {
            const size_t t = static_cast<size_t>(~ref), to = baseTri + rank - nInt;
            const float4 v0 = tris[3 * t], v1 = tris[3 * t + 1], v2 = tris[3 * t + 2];
            outTris[3 * to] = make_float4(v0.x, v0.y, v0.z, __uint_as_float(slot));
            outTris[3 * to + 1] = make_float4(v1.x, v1.y, v1.z, __int_as_float(static_cast<int32_t>(t)));
            outTris[3 * to + 2] = make_float4(v2.x, v2.y, v2.z, 0.0f);
        }
    }
    if (!kAll) return;
    __syncthreads();  // the level's work entries and its children's number are whole
    begin = next;
    n = level + 1 < levels && !spilled ? below : 0u;
    __syncthreads();
    }
}

__global__ void k_w8_clear(uint32_t *flags, W8Info *info) {
    uint32_t *w = reinterpret_cast<uint32_t *>(info);
    const uint32_t t = threadIdx.x;
    if (t < sizeof(W8Info) / 4) w[t] = t == 0 ? 1u : 0u;
    if (t < 4) flags[t] = 0u;
}

}  // namespace

namespace rki {
// Binds a validated tree (nNodes = nTris - 1, every index in range, depth <= 64) to the context
// and builds its 4-entry and 8-entry nodes. Waits for the device first: work still in flight may
// read the previous tree's nodes, which share the context buffer.
int bind_tree(restir_ctx *ctx, const void *nodes, uint32_t nNodes, const void *tris, uint32_t depth, hipStream_t s) {
    auto hip = [&](hipError_t e, const char *what) { return e == hipSuccess ? RESTIR_OK : hip_fail(ctx, e, what); };
    if (int r = hip(hipDeviceSynchronize(), "bind tree: wait for work in flight")) return r;
    // 8-entry nodes: every node with an internal child has 8 entries, so T triangles need at most
    // 4 T / 7 + 1 nodes (each of them with two-triangle nodes below), usually less than half of that.
    // Node indices take 23 bits of a child word, triangles 26 bits of a tracer's list entry; a tree
    // that turns out to need more nodes, or for which there is no memory, keeps its 4-entry nodes.
    const uint32_t nTris = nNodes + 1;
    const uint64_t most = 4ull * nTris / 7 + 8;
    const uint32_t maxW8 = static_cast<uint32_t>(most < (1u << 23) ? most : 1u << 23);
    bool w8Fits = nTris <= (1u << 26);
    const auto carve = [&](void *base, size_t *bytes) {
        struct {
            rt::WNode *wide;
            rt::W8Node *w8;
            float4 *tris;
            uint32_t *parent, *work, *flags;
            W8Info *info;
        } p{};
        rk::Carver c(base);
        p.wide = c.take<rt::WNode>(sizeof(rt::WNode) * static_cast<size_t>(nNodes));
        p.flags = c.take<uint32_t>(16 + sizeof(W8Info));  // 4 flag words, then the counters
        if (w8Fits) {
            p.w8 = c.take<rt::W8Node>(sizeof(rt::W8Node) * static_cast<size_t>(maxW8));
            p.tris = c.take<float4>(48 * static_cast<size_t>(nTris));
            p.parent = c.take<uint32_t>(4 * static_cast<size_t>(nNodes));
            p.work = c.take<uint32_t>(4 * static_cast<size_t>(maxW8));
        }
        p.info = reinterpret_cast<W8Info *>(p.flags + 4);
        if (bytes) *bytes = c.end();
        return p;
    };
    size_t bytes = 0;
    carve(nullptr, &bytes);
    int held = ensure(ctx, &ctx->wide, &ctx->wideBytes, bytes);
    if (held != RESTIR_OK && w8Fits) {  // the 4-entry nodes alone take half
        (void)hipGetLastError();
        ctx->error.clear();
        w8Fits = false;
        carve(nullptr, &bytes);
        held = ensure(ctx, &ctx->wide, &ctx->wideBytes, bytes);
    }
    if (held != RESTIR_OK) return held;
    const auto p = carve(ctx->wide, nullptr);
    const auto *bn = static_cast<const rt::Node *>(nodes);
    const auto *bt = static_cast<const float4 *>(tris);
    RK_LAUNCH("k_w8_clear", k_w8_clear, dim3(1), dim3(64), 0, s, p.flags, p.info);
    RK_LAUNCH("k_wide_build", k_wide_build, dim3(groups(nNodes)), dim3(256), 0, s, bn, nNodes, bt, p.wide, p.parent,
              p.flags);
    // a level of 8-entry nodes covers at least one level of the tree
    const uint32_t levels = depth < static_cast<uint32_t>(kW8Levels) ? depth : static_cast<uint32_t>(kW8Levels);
    struct {
        uint32_t flags[4];
        W8Info w8;
    } host{{1u, 0x7fc00000u, 1u, 1u}, {}};
    static_assert(sizeof host == 16 + sizeof(W8Info), "flags and counters are copied together");
    // Usually 8-entry levels are about a third as many: after the first launches the counters say
    // whether there are more (an empty launch takes 4 us, 13 of them in a tree of 23 levels).
    // A small tree's are made by one workgroup in one launch.
    uint32_t done = 0;
    if (w8Fits && maxW8 <= kW8OneGroup) {
        RK_LAUNCH("k_w8_collapse", k_w8_collapse<true>, dim3(1), dim3(512), 0, s, bn, bt, 0u, levels, maxW8, nTris, p.flags,
                  p.w8, p.tris, p.work, p.info);
        done = levels;
    }
    for (uint32_t batch = 4 + (32u - static_cast<uint32_t>(__builtin_clz(nTris))) / 3;; batch = 4) {
        const uint32_t end = !w8Fits ? 0u : (done + batch < levels ? done + batch : levels);
        for (; done < end; ++done)
            RK_LAUNCH("k_w8_collapse", k_w8_collapse<false>, dim3(1024), dim3(512), 0, s, bn, bt, done, 1u, maxW8, nTris,
                      p.flags, p.w8, p.tris, p.work, p.info);
        if (int r = hip(hipMemcpyAsync(&host, p.flags, sizeof host, hipMemcpyDeviceToHost, s), "bind tree: read")) return r;
        if (int r = hip(hipStreamSynchronize(s), "bind tree: finish")) return r;
        if (!w8Fits || done == levels || host.w8.nodes[done] == 0) break;
    }
    float maxCoord;
    std::memcpy(&maxCoord, &host.flags[1], sizeof maxCoord);
    ctx->scene.nodes = bn;
    ctx->scene.tris = bt;
    ctx->scene.wide = p.wide;
    ctx->scene.treeNested = host.flags[0] == 0 ? 1 : 0;
    ctx->scene.maxCoord = maxCoord;
    ctx->scene.quickCoord = nNodes <= (1u << 25) ? maxCoord : __builtin_nanf("");
    ctx->scene.parent = p.parent;
    ctx->scene.w8 = p.w8;
    ctx->scene.w8Tris = p.tris;
    ctx->scene.treeTight = host.flags[3] == 0 ? 1 : 0;
    ctx->scene.w8Ok = w8Fits && host.flags[2] == 0 && host.w8.overflow == 0 && host.w8.nodes[done] == 0 &&
                              host.w8.tris == nTris && rt::w8_covers(maxCoord)
                          ? 1
                          : 0;
    ctx->scene.w8Grid = ctx->cus * rk::kTrace8PerCu;
    ctx->scene.invMax = 1e30f / fmaxf(maxCoord, 1.0f);
    // a walk defers at most one sibling per internal level below the root: depth - 1 entries
    ctx->stack = depth <= 24 ? 24 : (depth <= 32 ? 32 : 64);
    ctx->persistentBlocks = persistent_blocks(ctx->cus, ctx->stack);
    ctx->treeDepth = depth;
    ctx->treeTris = nTris;
    ctx->bvhSet = true;
    return RESTIR_OK;
}
}  // namespace rki

extern "C" int restir_build_bvh(restir_ctx *ctx, const float *triXyz, uint32_t nTris, restir_aabb_tree_node *nodes,
                                restir_triangle *tris, uint32_t *depthOut, void *stream) {
    if (!ctx) return RESTIR_E_INVALID_ARGUMENT;
    ctx->bvhSet = false;
    if (!triXyz || !nodes || !tris) return fail(ctx, RESTIR_E_INVALID_ARGUMENT, "build_bvh: NULL buffer");
    if (nTris < 2) return fail(ctx, RESTIR_E_INVALID_ARGUMENT, "build_bvh: %u triangles (need >= 2)", nTris);
    if (nTris > (1u << 30)) return fail(ctx, RESTIR_E_INVALID_ARGUMENT, "build_bvh: %u triangles > 2^30", nTris);
    const size_t xyzBytes = 36ull * nTris, nodeBytes = sizeof(restir_aabb_tree_node) * (nTris - 1ull),
                 triBytes = sizeof(restir_triangle) * static_cast<size_t>(nTris);
    if (overlaps(triXyz, xyzBytes, nodes, nodeBytes) || overlaps(triXyz, xyzBytes, tris, triBytes) ||
        overlaps(nodes, nodeBytes, tris, triBytes))
        return fail(ctx, RESTIR_E_ALIASING, "build_bvh: vertex, node and triangle buffers must not overlap");
    if (int r = use_device(ctx)) return r;
    const Layout L = layout(nTris);
    if (int r = ensure(ctx, &ctx->bvhScratch, &ctx->bvhScratchBytes, L.total)) return r;
    if (!ctx->bvhInfoHost) {
        const hipError_t e = hipHostMalloc(&ctx->bvhInfoHost, sizeof(Info), hipHostMallocDefault);
        if (e != hipSuccess) {
            ctx->bvhInfoHost = nullptr;
            return hip_fail(ctx, e, "build_bvh: hipHostMalloc");
        }
    }
    char *base = static_cast<char *>(ctx->bvhScratch);
    float4 *box = reinterpret_cast<float4 *>(base + L.box);
    uint32_t *idx[2] = {reinterpret_cast<uint32_t *>(base + L.idx0), reinterpret_cast<uint32_t *>(base + L.idx1)};
    int32_t *segOf[2] = {reinterpret_cast<int32_t *>(base + L.seg0), reinterpret_cast<int32_t *>(base + L.seg1)};
    uint8_t *bucket = reinterpret_cast<uint8_t *>(base + L.bucket);
    uint32_t *before = reinterpret_cast<uint32_t *>(base + L.before);
    uint32_t *ptr = reinterpret_cast<uint32_t *>(base + L.ptr), *ids = ptr;
    Seg *segs[2] = {reinterpret_cast<Seg *>(base + L.segs0), reinterpret_cast<Seg *>(base + L.segs1)};
    int32_t *segRank = reinterpret_cast<int32_t *>(base + L.segRank);
    Split *splits = reinterpret_cast<Split *>(base + L.splits);
    Sub *subs = reinterpret_cast<Sub *>(base + L.subs);
    u64 *acc = reinterpret_cast<u64 *>(base + L.acc);
    restir_aabb_tree_node *tmp = reinterpret_cast<restir_aabb_tree_node *>(base + L.tmp);
    uint8_t *levels = reinterpret_cast<uint8_t *>(base + L.levels);
    uint32_t *counts = reinterpret_cast<uint32_t *>(base + L.counts);
    Info *info = reinterpret_cast<Info *>(base + L.info);
    Info *host = static_cast<Info *>(ctx->bvhInfoHost);
    const hipStream_t s = static_cast<hipStream_t>(stream);
    const uint32_t n = nTris, nSums = (n + kScanGroup - 1) / kScanGroup;
    uint32_t *sums = reinterpret_cast<uint32_t *>(base + L.temp32), *temp32 = sums + nSums;

    auto hip = [&](hipError_t e, const char *what) { return e == hipSuccess ? RESTIR_OK : hip_fail(ctx, e, what); };
    auto read_info = [&](const char *what) {
        if (int r = hip(hipMemcpyAsync(host, info, sizeof(Info), hipMemcpyDeviceToHost, s), what)) return r;
        return hip(hipStreamSynchronize(s), what);
    };
    if (int r = hip(hipMemsetAsync(info, 0, sizeof(Info), s), "build_bvh: clear")) return r;
    RK_LAUNCH("k_bvh_prep", k_bvh_prep, dim3(groups(n)), dim3(256), 0, s, n, triXyz, tris, box, idx[0], segOf[0], acc,
              segs[0], info);

    uint32_t S = 1, cur = 0;
    for (uint32_t level = 1;; ++level) {
        RK_LAUNCH("k_bvh_level", k_bvh_level, dim3(1), dim3(256), 0, s, S, level, segs[cur], idx[cur], tmp, segRank, splits,
                  subs, info);
        if (int r = read_info("build_bvh: level")) return r;
        if (host->bad) return fail(ctx, RESTIR_E_INVALID_ARGUMENT, "build_bvh: a vertex coordinate is not finite");
        const uint32_t nSplits = host->splits;
        if (nSplits == 0) break;
        RK_LAUNCH("k_bvh_bounds", k_bvh_bounds, dim3(groups(n)), dim3(256), 0, s, n, idx[cur], segOf[cur], segRank, splits,
                  box, acc);
        RK_LAUNCH("k_bvh_bin", k_bvh_bin, dim3(groups(n)), dim3(256), 0, s, n, idx[cur], segOf[cur], segRank, box, bucket,
                  acc);
        RK_LAUNCH("k_bvh_choose", k_bvh_choose, dim3((nSplits + 15) / 16), dim3(256), 0, s, nSplits, level, idx[cur], box,
                  acc, splits, tmp, levels, segs[cur ^ 1]);
        RK_LAUNCH("k_bvh_left_count", k_bvh_left_count, dim3(nSums), dim3(256), 0, s, n, segOf[cur], segRank, splits, bucket,
                  before, sums);
        if (int r = hip(rscan::exclusive_scan<uint32_t>(sums, sums, nSums, temp32, nullptr, s), "build_bvh: scan")) return r;
        RK_LAUNCH("k_bvh_chain", k_bvh_chain, dim3(groups(n)), dim3(256), 0, s, n, segOf[cur], segRank, splits, bucket,
                  before, sums, ptr);
        RK_LAUNCH("k_bvh_scatter", k_bvh_scatter, dim3(groups(n)), dim3(256), 0, s, n, nSplits, segOf[cur], segRank, splits,
                  bucket, before, sums, ptr, idx[cur], idx[cur ^ 1], segOf[cur ^ 1], acc);
        if (int r = hip(hipGetLastError(), "build_bvh: launch")) return r;
        S = 2 * nSplits;
        cur ^= 1;
    }
    // every level ends in smaller ranges: the deepest nodes are theirs
    RK_LAUNCH("k_bvh_subtrees", k_bvh_subtrees, dim3(host->subs), dim3(256), 0, s, subs, idx[cur], box, tmp, levels, info);
    if (int r = read_info("build_bvh: subtrees")) return r;
    const uint32_t depth = host->depth;
    if (depth > 64)
        return fail(ctx, RESTIR_E_BAD_TREE, "build_bvh: tree depth %u exceeds the 64-entry traversal stack", depth);
    const uint32_t nBlocks = groups(n - 1);
    RK_LAUNCH("k_bvh_level_counts", k_bvh_level_counts, dim3(nBlocks), dim3(256), 0, s, n - 1, depth, levels, counts);
    if (int r = hip(rscan::exclusive_scan<uint32_t>(counts, counts, depth * nBlocks, temp32, nullptr, s), "build_bvh: scan"))
        return r;
    RK_LAUNCH("k_bvh_ids", k_bvh_ids, dim3(nBlocks), dim3(256), 0, s, n - 1, levels, counts, ids);
    RK_LAUNCH("k_bvh_write", k_bvh_write, dim3(nBlocks), dim3(256), 0, s, n - 1, tmp, ids, nodes);
    if (int r = hip(hipGetLastError(), "build_bvh: launch")) return r;
    if (depthOut) *depthOut = depth;
    return bind_tree(ctx, nodes, n - 1, tris, depth, s);
}
