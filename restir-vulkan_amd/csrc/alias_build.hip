// alias_build.hip — createAliasTable (src/misc.cpp:418-497) on the device: the reference's table,
// column for column and bit for bit, without a host round trip, so it can sit inside a captured
// graph: in one workgroup and one launch up to kMany lights, above by launches over the device and
// that workgroup for the end of the pairing. The workgroup's body is alias_kernel.h, shared with a CPU build
// (one thread per lane) that runs it under ThreadSanitizer and AddressSanitizer.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "carve.h"
#include "ctx.h"
#include "kernels.h"
#include "scan.h"

#define AK_FN __device__ __forceinline__
#define AK_WAVE_SYNC(g) rk::wave_sync()
#include "alias_kernel.h"

using namespace rki;

namespace {

constexpr uint32_t kLanes = ak::kLanes;

// the workgroup policy of alias_kernel.h on the device
struct DeviceGroup {
    __device__ __forceinline__ uint32_t tid() const { return threadIdx.x; }
    __device__ __forceinline__ void sync() const { __syncthreads(); }
    __device__ __forceinline__ uint32_t shfl_up(uint32_t v, uint32_t d) const {
        return __shfl_up(v, static_cast<unsigned int>(d), 64);
    }
};

__global__ __launch_bounds__(kLanes) void k_alias_build(const restir_point_light *points, const restir_tri_light *triLights,
                                                        uint32_t n, restir_alias_table_column *cols, float *power,
                                                        float *scaled, uint32_t *under, uint32_t *overA,
                                                        uint32_t *overB) {
    __shared__ ak::Shared sh;
    DeviceGroup g;
    ak::build(g, sh, points, triLights, n, cols, power, scaled, under, overA, overB);
}

// ---- many lights (n > kMany): the same steps over the whole device.
// The power sum: each wave takes a segment of kSeg lights (4 consecutive ones per lane). A first
// launch adds each segment in double, which predicts the binade of the sequential float sum at its
// start; a second one forms the segment's increment map for that binade; then one workgroup walks
// the segments, lane 0 applying a map where the prediction holds and the sum stays in the binade,
// and adding a segment's lights one by one elsewhere (about once per binade). Then the columns are
// normalised, the queues filled by a scan, and the first rounds of the pairing run as two launches
// a step (pair; append in pair order), as many steps as bring the queues of ordinary lights down to
// ak::kStep items, each a no-op once they are. The workgroup of k_alias_rest goes on from there.
// Device-driven throughout, so the sequence can be captured. In one workgroup the build is bound by
// the requests of one CU and by one lane's additions: 100,000 lights take 1.31 ms there, 0.23 here;
// 1M lights 13.3 and 0.71. Here it is bound by its 15 to 40 launches (about 4 us each) and the last
// rounds: 4,097 lights take 0.073 ms there and 0.066 here, 10,000 0.148 and 0.093, hence kMany.
constexpr uint32_t kMany = 4096;
constexpr uint32_t kSeg = 256, kPairs = 2048;  // pairs per workgroup and step

struct State {
    uint32_t head, tail, m, k0, mNext;
    uint32_t flip;  // the larges' queues have changed places an odd number of times
    uint32_t done;  // no more steps over the device
    float powerSum;
};

__device__ inline double wave_add(double v) {
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) v += __shfl_xor(v, d);
    return v;
}

__global__ __launch_bounds__(256) void k_alias_power(const restir_point_light *points, const restir_tri_light *triLights,
                                                     uint32_t n, float *power, double *segSum) {
    const uint32_t i0 = (blockIdx.x * 256u + threadIdx.x) * 4u;
    double sum = 0.0;
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k)
        if (i0 + k < n) {
            const float w = ak::power_of(points, triLights, i0 + k);
            power[i0 + k] = w;
            sum += static_cast<double>(w);
        }
    sum = wave_add(sum);
    if ((threadIdx.x & 63u) == 0 && i0 < n) segSum[i0 / kSeg] = sum;
}

// map[s]: {exponent field of the predicted sum, increments of an even and an odd sum}
__global__ __launch_bounds__(256) void k_alias_maps(uint32_t n, const float *power, const double *segSum, uint3 *map) {
    __shared__ double part[4];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint32_t seg0 = blockIdx.x * 4u, seg = seg0 + wave;
    double before = 0.0;
    for (uint32_t j = threadIdx.x; j < seg0; j += 256u) before += segSum[j];
    before = wave_add(before);
    if (lane == 0) part[wave] = before;
    __syncthreads();
    before = ((part[0] + part[1]) + part[2]) + part[3];
    const uint32_t i0 = (blockIdx.x * 256u + threadIdx.x) * 4u;
    if (seg * kSeg >= n) return;  // wave-uniform
    for (uint32_t j = 0; j < wave; ++j) before += segSum[seg0 + j];
    const uint32_t e = __float_as_uint(static_cast<float>(before)) >> 23;
    const bool usable = e >= 27u && e <= 227u;  // a positive normal sum well inside the range
    ak::Inc a{0u, 0u};
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k)
        if (i0 + k < n) a = ak::compose(a, ak::inc_of(power[i0 + k], e));
#pragma unroll
    for (uint32_t d = 1; d < 64; d <<= 1) {
        const ak::Inc o{__shfl_up(a.even, d), __shfl_up(a.odd, d)};
        if (lane >= d) a = ak::compose(o, a);
    }
    if (lane == 63u) map[seg] = usable ? make_uint3(e, a.even, a.odd) : make_uint3(0u, ak::kOver, ak::kOver);
}

// One wave, its state wave-uniform (in scalar registers but for the sum): 64 maps at a time, one per
// lane, are applied in order; the segment that one does not apply to is added light by light from
// four registers per lane.
__global__ __launch_bounds__(64) void k_alias_sum(uint32_t n, const float *power, const uint3 *map, State *state) {
    const uint32_t lane = threadIdx.x, segs = (n + kSeg - 1) / kSeg;
    float sum = 0.0f;
    for (uint32_t base = 0; base < segs; base += 64u) {
        const uint32_t m = segs - base < 64u ? segs - base : 64u;
        const uint3 v = lane < m ? map[base + lane] : make_uint3(0u, ak::kOver, ak::kOver);
        for (uint32_t j = 0; j < m; ++j) {
            const uint32_t bits = __builtin_amdgcn_readfirstlane(__float_as_uint(sum)), e = bits >> 23;
            uint32_t k = (bits & 0x7fffffu) | 0x800000u;  // the sum in ulps
            bool stuck = false;
            for (; j < m; ++j) {
                if (__builtin_amdgcn_readlane(v.x, j) != e || e == 0u) {
                    stuck = true;
                    break;
                }
                const uint32_t even = __builtin_amdgcn_readlane(v.y, j), odd = __builtin_amdgcn_readlane(v.z, j);
                const uint32_t i = (k & 1u) ? odd : even;
                if (k + i >= ak::kOver) {
                    stuck = true;
                    break;
                }
                k += i;
            }
            if (e != 0u && e < 255u) sum = __uint_as_float((e << 23) | (k & 0x7fffffu));
            if (!stuck) break;
            const uint32_t first = (base + j) * kSeg;
            float w[4];
#pragma unroll
            for (uint32_t r = 0; r < 4; ++r) {
                const uint32_t i = first + 64u * r + lane;
                w[r] = i < n ? power[i] : 0.0f;  // adding +0 changes no sum
            }
#pragma unroll
            for (uint32_t r = 0; r < 4; ++r)
#pragma unroll
                for (uint32_t l = 0; l < 64; ++l)
                    sum += __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(w[r]), l));
        }
    }
    if (lane == 0) state[0].powerSum = sum;
}

// columns before the pairing; flags: 1 for a small item, 2^32 for a large one
__global__ __launch_bounds__(256) void k_alias_normalise(uint32_t n, const float *power, const State *state,
                                                         restir_alias_table_column *cols, float *scaled,
                                                         unsigned long long *flags) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i >= n) return;
    const float s = ak::normalised(cols, i, power[i], state[0].powerSum, static_cast<float>(n));
    scaled[i] = s;
    flags[i] = s >= 1.0f ? 1ull << 32 : 1ull;
}

__global__ __launch_bounds__(256) void k_alias_queues(uint32_t n, const float *scaled, const unsigned long long *scan,
                                                      uint32_t *under, uint32_t *overA, State *state) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i >= n) return;
    const uint32_t smalls = static_cast<uint32_t>(scan[i]), larges = static_cast<uint32_t>(scan[i] >> 32);
    const bool large = scaled[i] >= 1.0f;
    if (large) overA[larges] = i;
    else under[smalls] = i;
    if (i == n - 1) {
        State st = state[0];
        st.head = st.k0 = st.mNext = st.flip = 0u;
        st.tail = smalls + (large ? 0u : 1u);
        st.m = larges + (large ? 1u : 0u);
        st.done = st.m == 0 || st.tail == 0 || n <= ak::kStep ? 1u : 0u;
        state[0] = st;
    }
}

__device__ inline uint32_t pairs_of(const State &st) {
    if (st.done) return 0u;
    const uint32_t l = st.m - st.k0, s = st.tail - st.head;
    return l < s ? l : s;
}

// One step: pair the next larges with the next smalls; smalls[b]: how many of workgroup b's larges
// became small.
__global__ __launch_bounds__(256) void k_alias_pair(const State *state, restir_alias_table_column *cols, float *scaled,
                                                    const uint32_t *under, const uint32_t *over0, const uint32_t *over1,
                                                    uint32_t *smalls) {
    __shared__ uint32_t sum;
    const State st = *state;
    const uint32_t c = pairs_of(st), j0 = blockIdx.x * kPairs;
    if (j0 >= c) return;
    const uint32_t *cur = st.flip ? over1 : over0;
    if (threadIdx.x == 0) sum = 0u;
    __syncthreads();
    uint32_t gl[8], l[8], mine = 0;
#pragma unroll
    for (uint32_t k = 0; k < 8; ++k) {
        const uint32_t j = j0 + k * 256u + threadIdx.x;
        gl[k] = j < c ? cur[st.k0 + j] : 0u;
        l[k] = j < c ? under[st.head + j] : 0u;
    }
    float sg[8], sl[8];
#pragma unroll
    for (uint32_t k = 0; k < 8; ++k) {
        sg[k] = scaled[gl[k]];
        sl[k] = scaled[l[k]];
    }
#pragma unroll
    for (uint32_t k = 0; k < 8; ++k) {
        if (j0 + k * 256u + threadIdx.x >= c) continue;
        cols[l[k]].prob = sl[k];
        cols[l[k]].alias = static_cast<int32_t>(gl[k]);
        const float v = (sg[k] + sl[k]) - 1.0f;
        scaled[gl[k]] = v;
        mine += v < 1.0f ? 1u : 0u;
    }
    atomicAdd(&sum, mine);
    __syncthreads();
    if (threadIdx.x == 0) smalls[blockIdx.x] = sum;
}

// The rest of the step: its larges go to the back of the small or the next large queue in pair order;
// workgroup 0 writes the state of the next step.
__global__ __launch_bounds__(256) void k_alias_append(const State *state, State *next, const float *scaled,
                                                      uint32_t *under, uint32_t *over0, uint32_t *over1,
                                                      const uint32_t *smalls) {
    __shared__ uint32_t earlier, total, count[32];
    const State st = *state;
    const uint32_t c = pairs_of(st), j0 = blockIdx.x * kPairs;
    if (j0 >= c) {
        if (blockIdx.x == 0 && threadIdx.x == 0) *next = st;
        return;
    }
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    // smalls of the workgroups before this one, and (workgroup 0) of all
    const uint32_t groups = (c + kPairs - 1) / kPairs;
    uint32_t before = 0, all = 0;
    for (uint32_t b = threadIdx.x; b < (blockIdx.x == 0 ? groups : blockIdx.x); b += 256u) {
        all += smalls[b];
        if (b < blockIdx.x) before += smalls[b];
    }
    if (threadIdx.x == 0) earlier = total = 0u;
    __syncthreads();
    if (before) atomicAdd(&earlier, before);
    if (all) atomicAdd(&total, all);
    __syncthreads();
    before = earlier;
    all = total;
    const uint32_t *cur = st.flip ? over1 : over0;
    uint32_t *nxt = st.flip ? over0 : over1;
    // pair j0 + 256 k + lane: its rank among the smalls from the ballots of all rows and waves
    uint32_t gl[8];
    uint64_t mask[8];
#pragma unroll
    for (uint32_t k = 0; k < 8; ++k) {
        const uint32_t j = j0 + k * 256u + threadIdx.x;
        gl[k] = j < c ? cur[st.k0 + j] : 0u;
    }
#pragma unroll
    for (uint32_t k = 0; k < 8; ++k) {
        mask[k] = __ballot(j0 + k * 256u + threadIdx.x < c && scaled[gl[k]] < 1.0f);
        if (lane == 0) count[4 * k + wave] = static_cast<uint32_t>(__popcll(mask[k]));
    }
    __syncthreads();
    uint32_t run = before;  // smalls before row k's first pair of this wave
#pragma unroll
    for (uint32_t k = 0; k < 8; ++k) {
        uint32_t s = run;
#pragma unroll
        for (uint32_t w = 0; w < 4; ++w) {
            s += w < wave ? count[4 * k + w] : 0u;
            run += count[4 * k + w];
        }
        s += __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(mask[k] >> 32),
                                       __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(mask[k]), 0u));
        const uint32_t j = j0 + k * 256u + threadIdx.x;
        if ((mask[k] >> lane) & 1ull) under[st.tail + s] = gl[k];
        else if (j < c) nxt[st.mNext + (j - s)] = gl[k];
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        State n = st;
        n.head += c;
        n.k0 += c;
        n.tail += all;
        n.mNext += c - all;
        if (n.k0 == n.m) {  // the round is over
            n.m = n.mNext;
            n.k0 = n.mNext = 0u;
            n.flip ^= 1u;
            n.done = n.m + (n.tail - n.head) <= ak::kStep ? 1u : 0u;
        }
        if (n.head == n.tail) n.done = 1u;
        *next = n;
    }
}

__global__ __launch_bounds__(kLanes) void k_alias_rest(const State *state, restir_alias_table_column *cols,
                                                       float *scaled, uint32_t *under, uint32_t *over0,
                                                       uint32_t *over1) {
    __shared__ ak::Shared sh;
    DeviceGroup g;
    const State st = *state;
    ak::Queues q{scaled, under, st.flip ? over1 : over0, st.flip ? over0 : over1, nullptr,
                 st.head, st.tail, st.m, st.k0, st.mNext};
    ak::pair_all(g, sh, cols, q);
}

__global__ __launch_bounds__(256) void k_alias_finish(restir_alias_table_column *cols, uint32_t n) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i < n) ak::finish(cols, i);
}

// steps of the pairing over the device: the queues of ordinary lights shrink by about a quarter to a
// third per round
uint32_t device_steps(uint32_t n) {
    uint32_t s = 0;
    while (s < 7 && (ak::kStep << s) < n) ++s;
    return 2 * s;
}

}  // namespace

extern "C" int restir_build_alias_table_device(restir_ctx *ctx, const restir_point_light *points, uint32_t nPoint,
                                               const restir_tri_light *triLights, uint32_t nTri,
                                               restir_alias_table_column *columns, void *stream) {
    if (!ctx) return RESTIR_E_INVALID_ARGUMENT;
    const uint32_t n = nPoint > 0 ? nPoint : nTri;
    if (n == 0) return RESTIR_OK;
    if (!columns || (nPoint > 0 && !points) || (nPoint == 0 && !triLights))
        return fail(ctx, RESTIR_E_INVALID_ARGUMENT, "build_alias_table_device: NULL buffer");
    if (n > (1u << 30)) return fail(ctx, RESTIR_E_INVALID_ARGUMENT, "build_alias_table_device: %u lights > 2^30", n);
    const size_t colBytes = sizeof(restir_alias_table_column) * static_cast<size_t>(n);
    const void *in = nPoint > 0 ? static_cast<const void *>(points) : static_cast<const void *>(triLights);
    const size_t inBytes = nPoint > 0 ? sizeof(restir_point_light) * static_cast<size_t>(n)
                                      : sizeof(restir_tri_light) * static_cast<size_t>(n);
    if (overlaps(columns, colBytes, in, inBytes))
        return fail(ctx, RESTIR_E_ALIASING, "build_alias_table_device: columns overlap the light records");
    if (int r = use_device(ctx)) return r;
    const hipStream_t s = static_cast<hipStream_t>(stream);
    const restir_point_light *pts = nPoint > 0 ? points : nullptr;
    const restir_tri_light *tls = nPoint > 0 ? nullptr : triLights;
    const uint32_t segs = (n + kSeg - 1) / kSeg, groups = (n + kPairs - 1) / kPairs;
    struct {
        float *power, *scaled;
        uint32_t *under, *overA, *overB, *smalls;
        double *segSum;
        uint3 *map;
        unsigned long long *flags, *temp;
        State *state;
    } p;
    const auto carve = [&](void *base, bool many) {
        rk::Carver c(base);
        p.power = c.take<float>(4ull * n);
        p.scaled = c.take<float>(4ull * n);
        p.under = c.take<uint32_t>(4ull * n);
        p.overA = c.take<uint32_t>(4ull * n);
        p.overB = c.take<uint32_t>(4ull * n);
        if (many) {
            p.smalls = c.take<uint32_t>(4ull * groups);
            p.segSum = c.take<double>(8ull * segs);
            p.map = c.take<uint3>(12ull * segs);
            p.flags = c.take<unsigned long long>(8ull * n);
            p.temp = c.take<unsigned long long>(8ull * rscan::temp_items(n));
            p.state = c.take<State>(sizeof(State) * (device_steps(n) + 1));
        }
        return c.end();
    };
    // the device-wide steps, unless the larger scratch cannot be had under capture
    bool many = n > kMany;
    size_t bytes = carve(nullptr, many);
    if (many && bytes > ctx->aliasScratchBytes && in_capture(s)) {
        many = false;
        bytes = carve(nullptr, many);
    }
    if (int r = ensure_kept(ctx, &ctx->aliasScratch, &ctx->aliasScratchBytes, &ctx->aliasInGraph, bytes, s)) return r;
    carve(ctx->aliasScratch, many);
    if (!many) {
        RK_LAUNCH("k_alias_build", k_alias_build, dim3(1), dim3(kLanes), 0, s, pts, tls, n, columns, p.power, p.scaled,
                  p.under, p.overA, p.overB);
    } else {
        const dim3 all((n + 255) / 256), quads((n + 1023) / 1024), block(256);
        RK_LAUNCH("k_alias_power", k_alias_power, quads, block, 0, s, pts, tls, n, p.power, p.segSum);
        RK_LAUNCH("k_alias_maps", k_alias_maps, quads, block, 0, s, n, p.power, p.segSum, p.map);
        RK_LAUNCH("k_alias_sum", k_alias_sum, dim3(1), dim3(64), 0, s, n, p.power, p.map, p.state);
        RK_LAUNCH("k_alias_normalise", k_alias_normalise, all, block, 0, s, n, p.power, p.state, columns, p.scaled,
                  p.flags);
        const hipError_t es = rscan::exclusive_scan<unsigned long long>(p.flags, p.flags, n, p.temp, nullptr, s);
        if (es != hipSuccess) return hip_fail(ctx, es, "build_alias_table_device scan");
        RK_LAUNCH("k_alias_queues", k_alias_queues, all, block, 0, s, n, p.scaled, p.flags, p.under, p.overA, p.state);
        const uint32_t steps = device_steps(n);
        for (uint32_t k = 0; k < steps; ++k) {
            RK_LAUNCH("k_alias_pair", k_alias_pair, dim3(groups), block, 0, s, p.state + k, columns, p.scaled, p.under,
                      p.overA, p.overB, p.smalls);
            RK_LAUNCH("k_alias_append", k_alias_append, dim3(groups), block, 0, s, p.state + k, p.state + k + 1,
                      p.scaled, p.under, p.overA, p.overB, p.smalls);
        }
        RK_LAUNCH("k_alias_rest", k_alias_rest, dim3(1), dim3(kLanes), 0, s, p.state + steps, columns, p.scaled, p.under,
                  p.overA, p.overB);
        RK_LAUNCH("k_alias_finish", k_alias_finish, all, block, 0, s, columns, n);
    }
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? RESTIR_OK : hip_fail(ctx, e, "build_alias_table_device launch");
}
