// near_math.hip — the correctly rounded division, reciprocal and square root of csrc/rt_math.h
// against the compiler's IEEE forms, on the device (not part of the library; a shared object that
// tests/test_gpu_near_math_all.py loads). Each check counts operands whose results differ in a bit:
//   near_rcp, near_over_pi  every float in [2^-60, 2^60]
//   near_sqrt               every float in [2^-100, 2^100]
//   near_div                every mantissa of b with `n` mantissas of a from `a0` on, exponents 0:
//                           all 2^46 pairs with a0 = 0, n = 2^23
//   near_range              2^24 x `n` pseudo-random operands over the whole of the ranges that mid_range
//                           and mid_range3 admit, each range's ends among them: quotients, roots, normalize_near
// Returns the count, or -1 after an error of the runtime.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "../csrc/rt_math.h"

namespace {

constexpr uint32_t kOne = 0x3f800000u;

__device__ bool differ(float a, float b) { return __float_as_uint(a) != __float_as_uint(b); }
__device__ uint64_t mix(uint64_t x) {  // splitmix64
    x += 0x9e3779b97f4a7c15ull;
    x = (x ^ (x >> 30)) * 0xbf58476d1ce4e5b9ull;
    x = (x ^ (x >> 27)) * 0x94d049bb133111ebull;
    return x ^ (x >> 31);
}
// a positive float with its bits in [lo, hi]; one in 16 is an end or next to one
__device__ float draw(uint64_t r, uint32_t lo, uint32_t hi) {
    const uint32_t pick = static_cast<uint32_t>(r & 15u), near = static_cast<uint32_t>(r >> 4) & 3u;
    if (pick == 0) return __uint_as_float((r & 64u) ? lo + near : hi - near);
    return __uint_as_float(lo + static_cast<uint32_t>((r >> 8) % (hi - lo + 1u)));
}

template <int WHAT>
__global__ __launch_bounds__(256) void k_all(uint32_t lo, uint32_t hi, unsigned long long *bad) {
    uint32_t c = 0;
    for (uint64_t u = lo + static_cast<uint64_t>(blockIdx.x) * 256u + threadIdx.x; u <= hi; u += gridDim.x * 256ull) {
        const float x = __uint_as_float(static_cast<uint32_t>(u));
        if (WHAT == 0) c += differ(rt::rcp_near(x), 1.0f / x);
        if (WHAT == 1) c += differ(rt::over_pi(x), x / rt::kPi);
        if (WHAT == 2) c += differ(rt::sqrt_near(x), sqrtf(x));
    }
    if (c) atomicAdd(bad, static_cast<unsigned long long>(c));
}

__global__ __launch_bounds__(256) void k_div(uint32_t a0, uint32_t n, unsigned long long *bad) {
    const float b = __uint_as_float(kOne | (blockIdx.x * 256u + threadIdx.x)), y = rt::rcp_near(b);
    uint32_t c = 0;
    for (uint32_t i = 0; i < n; ++i) {
        const float a = __uint_as_float(kOne | (a0 + i));
        c += differ(rt::div_near(a, b, y), a / b);
    }
    if (c) atomicAdd(bad, static_cast<unsigned long long>(c));
}

__global__ __launch_bounds__(256) void k_range(uint32_t n, unsigned long long *bad) {
    constexpr uint32_t kLo = 0x21800000u, kHi = 0x5d800000u;  // 2^-60, 2^60
    uint64_t r = mix(static_cast<uint64_t>(blockIdx.x) * 256u + threadIdx.x);
    uint32_t c = 0;
    for (uint32_t i = 0; i < n; ++i) {
        const float a = draw(r = mix(r), kLo, kHi), b = draw(r = mix(r), kLo, kHi);
        c += !rt::mid_range(a) || !rt::mid_range(b);
        c += differ(rt::div_near(a, b, rt::rcp_near(b)), a / b);
        c += differ(rt::sqrt_near(a), sqrtf(a));
        const auto part = [&]() {  // 2^-48 .. 2^30, of either sign
            const float v = draw(r = mix(r), 0x27800000u, 0x4e800000u);
            return (r >> 60) & 1u ? -v : v;
        };
        const rt::f3 v{part(), part(), part()};
        const float s2 = rt::dot(v, v);
        if (!rt::mid_range3(v, s2)) continue;
        const rt::f3 got = rt::normalize_near(v, s2), want = v / sqrtf(s2);
        c += differ(got.x, want.x) || differ(got.y, want.y) || differ(got.z, want.z);
    }
    if (c) atomicAdd(bad, static_cast<unsigned long long>(c));
}

template <class F>
int64_t counted(F launch) {
    unsigned long long *bad = nullptr, host = 0;
    if (hipMalloc(&bad, sizeof host) != hipSuccess) return -1;
    bool ok = hipMemcpy(bad, &host, sizeof host, hipMemcpyHostToDevice) == hipSuccess;
    if (ok) {
        launch(bad);
        ok = hipGetLastError() == hipSuccess && hipMemcpy(&host, bad, sizeof host, hipMemcpyDeviceToHost) == hipSuccess;
    }
    ok = hipFree(bad) == hipSuccess && ok;
    return ok ? static_cast<int64_t>(host) : -1;
}

}  // namespace

extern "C" {
int64_t near_rcp() {
    return counted([](unsigned long long *bad) { k_all<0><<<8192, 256>>>(0x21800000u, 0x5d800000u, bad); });
}
int64_t near_over_pi() {
    return counted([](unsigned long long *bad) { k_all<1><<<8192, 256>>>(0x21800000u, 0x5d800000u, bad); });
}
int64_t near_sqrt() {
    return counted([](unsigned long long *bad) { k_all<2><<<8192, 256>>>(0x0d800000u, 0x71800000u, bad); });
}
int64_t near_div(uint32_t a0, uint32_t n) {
    return counted([=](unsigned long long *bad) { k_div<<<32768, 256>>>(a0, n, bad); });
}
int64_t near_range(uint32_t n) {
    return counted([=](unsigned long long *bad) { k_range<<<65536, 256>>>(n, bad); });
}
}
