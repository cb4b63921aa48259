// rt_math.h — scalar/vector arithmetic of the ReSTIR path for gfx950 (and the host side of the
// library). Semantics are pinned so that results are reproducible bit for bit:
//   * built with -ffp-contract=off: no FMA contraction; a/b and sqrtf are IEEE correctly rounded
//     (HIP's default correctly-rounded fp32 divide/sqrt is kept);
//   * GLSL min/max/clamp/mix as the GLSL specification writes them;
//   * dot = (x*x' + y*y') + z*z'; normalize(v) = v / sqrt(dot(v, v)) per component;
//   * pow(r, 2.0) of disneyBRDF.glsl:46 is r*r;
//   * sin/cos: quadrant reduction and Taylor polynomials in double, rounded to float.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#define RT_HD __host__ __device__ __forceinline__

namespace rt {

constexpr float kPi = 3.14159265358979323846f;  // M_PI of disneyBRDF.glsl:1 as a float literal

struct f3 {
    float x, y, z;
};
RT_HD f3 make_f3(float x, float y, float z) { return f3{x, y, z}; }
RT_HD f3 operator+(f3 a, f3 b) { return f3{a.x + b.x, a.y + b.y, a.z + b.z}; }
RT_HD f3 operator-(f3 a, f3 b) { return f3{a.x - b.x, a.y - b.y, a.z - b.z}; }
RT_HD f3 operator*(f3 a, float s) { return f3{a.x * s, a.y * s, a.z * s}; }
RT_HD f3 operator*(float s, f3 a) { return f3{s * a.x, s * a.y, s * a.z}; }
RT_HD f3 operator/(f3 a, float s) { return f3{a.x / s, a.y / s, a.z / s}; }
RT_HD f3 neg(f3 a) { return f3{-a.x, -a.y, -a.z}; }
RT_HD float dot(f3 a, f3 b) { return (a.x * b.x + a.y * b.y) + a.z * b.z; }
RT_HD f3 cross(f3 a, f3 b) {
    return f3{a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x};
}
RT_HD f3 xyz(float4 v) { return f3{v.x, v.y, v.z}; }

// ---------------------------------------------------- correctly rounded division and square root
// The same numbers as `/` and sqrtf, from fewer instructions, for operands away from the ends of
// the exponent range. The compiler's IEEE division takes 11 instructions whatever its operands; here
// a divisor's reciprocal is formed once (rcp_near, 3) and each quotient over it takes 3. The square
// root takes 5 instead of about 15.
//   rcp_near(b)     = RN(1 / b):   one Newton step on the hardware's reciprocal
//   div_near(a,b,y) = RN(a / b):   a product and one residual step (Markstein 1990), y = rcp_near(b)
//   sqrt_near(x)    = RN(sqrt(x)): one residual step on the hardware's reciprocal square root
//   over_pi(x)      = RN(x / kPi): as div_near, with 1 / kPi rounded at compile time
// Compared on the MI355X with the IEEE forms for every b in [2^-60, 2^60], every x in [2^-100,
// 2^100], and every one of the 2^46 pairs of mantissas of a and b (probe/near_math.hip): no difference. Scaling by powers of
// two changes no mantissa while nothing under- or overflows, which the bounds below keep away. With
// them, and W formed once instead of per candidate, k_pass_a_ris (VALU bound: 0.82 of the issue
// rate) went from 0.75 to 0.635 ms at 1080p, M = 32.
#ifdef __HIP_DEVICE_COMPILE__
#define RT_NEAR_MATH 1
#endif
__device__ __forceinline__ float rcp_near(float b) {
    const float y = __builtin_amdgcn_rcpf(b);
    return fmaf(fmaf(-b, y, 1.0f), y, y);
}
__device__ __forceinline__ float div_near(float a, float b, float y) {
    const float q = a * y;
    return fmaf(fmaf(-b, q, a), y, q);
}
__device__ __forceinline__ float sqrt_near(float x) {
    const float y = __builtin_amdgcn_rsqf(x), g = x * y;
    return fmaf(fmaf(-g, g, x), 0.5f * y, g);
}
__device__ __forceinline__ float over_pi(float x) {
    constexpr float c = 1.0f / kPi;
    const float q = x * c;
    return fmaf(fmaf(-q, kPi, x), c, q);
}
// x in [2^-60, 2^60]; false for negative numbers, NaN and infinity
__device__ __forceinline__ bool mid_range(float x) {
    return __float_as_uint(x) - 0x21800000u <= 0x5d800000u - 0x21800000u;
}
// Every component of a at least 2^-48 in magnitude and |a|^2 = s2 at most 2^60
__device__ __forceinline__ bool mid_range3(f3 a, float s2) {
    return fminf(fminf(fabsf(a.x), fabsf(a.y)), fabsf(a.z)) >= 0x1p-48f && s2 <= 0x1p60f;
}
// a / sqrt(s2), s2 = dot(a, a) of a mid_range3 vector
__device__ __forceinline__ f3 normalize_near(f3 a, float s2) {
    const float s = sqrt_near(s2), y = rcp_near(s);
    return f3{div_near(a.x, s, y), div_near(a.y, s, y), div_near(a.z, s, y)};
}
RT_HD f3 normalize(f3 a) {
    const float s2 = dot(a, a);
#ifdef RT_NEAR_MATH
    if (mid_range3(a, s2)) return normalize_near(a, s2);
#endif
    return a / sqrtf(s2);
}

// The operations of the BRDF evaluation. Ieee: as written. Near: the forms above; `ok` turns false
// when an operand lies outside their ranges, and the result is then not used.
struct Ieee {
    static constexpr bool ok = true;
    __device__ __forceinline__ float div(float a, float b) { return a / b; }
    __device__ __forceinline__ float rcp(float b) { return 1.0f / b; }
    __device__ __forceinline__ float root(float x) { return sqrtf(x); }
    __device__ __forceinline__ float div_pi(float x) { return x / kPi; }
    __device__ __forceinline__ f3 unit(f3 a, float s2) { return a / sqrtf(s2); }
};
struct Near {
    bool ok = true;
    __device__ __forceinline__ float div(float a, float b) {
        ok = ok && mid_range(a) && mid_range(b);
        return div_near(a, b, rcp_near(b));
    }
    __device__ __forceinline__ float rcp(float b) {
        ok = ok && mid_range(b);
        return rcp_near(b);
    }
    __device__ __forceinline__ float root(float x) {
        ok = ok && mid_range(x);
        return sqrt_near(x);
    }
    __device__ __forceinline__ float div_pi(float x) {  // +0 (a metal) gives +0
        ok = ok && (mid_range(x) || __float_as_uint(x) == 0u);
        return over_pi(x);
    }
    __device__ __forceinline__ f3 unit(f3 a, float s2) {
        ok = ok && mid_range3(a, s2);
        return normalize_near(a, s2);
    }
};

RT_HD float gmin(float x, float y) { return (y < x) ? y : x; }
RT_HD float gmax(float x, float y) { return (x < y) ? y : x; }
RT_HD float gclamp(float x, float lo, float hi) { return gmin(gmax(x, lo), hi); }
RT_HD float gmix(float x, float y, float a) { return x * (1.0f - a) + y * a; }

// ------------------------------------------------------------------------------------ PCG32
// rand.glsl:7-32 — PCG32 XSH-RR, 64-bit state, seeded as pcg32_srandom_r(seed, seq).
struct Pcg {
    uint64_t state, inc;
};
constexpr uint64_t kPcgMul = 6364136223846793005ull;
// The number drawn at state `old` (the output permutation; the state then steps to old * a + inc).
RT_HD uint32_t pcg_output(uint64_t old) {
    const uint32_t xs = static_cast<uint32_t>(((old >> 18u) ^ old) >> 27u);
    const uint32_t rot = static_cast<uint32_t>(old >> 59u);
    return (xs >> rot) | (xs << ((0u - rot) & 31u));
}
RT_HD uint32_t pcg_next(Pcg &r) {
    const uint64_t old = r.state;
    r.state = old * kPcgMul + r.inc;
    return pcg_output(old);
}
// Jump-ahead: k steps after state s the state is a^k s + inc (1 + a + ... + a^(k-1)) (mod 2^64).
constexpr uint64_t pcg_mul_pow(int k) {
    uint64_t m = 1;
    for (int i = 0; i < k; ++i) m *= kPcgMul;
    return m;
}
constexpr uint64_t pcg_mul_sum(int k) {
    uint64_t sum = 0, m = 1;
    for (int i = 0; i < k; ++i) {
        sum += m;
        m *= kPcgMul;
    }
    return sum;
}
RT_HD Pcg pcg_seed(uint64_t seed, uint64_t seq) {
    Pcg r{0ull, (seq << 1u) | 1u};
    (void)pcg_next(r);
    r.state += seed;
    (void)pcg_next(r);
    return r;
}
// u32 -> float rounds to nearest even; the scale by 2^-32 is exact.
RT_HD float pcg_float(Pcg &r) { return static_cast<float>(pcg_next(r)) * 2.3283064365386963e-10f; }
// The float pcg_float draws at state s.
RT_HD float pcg_float_at(uint64_t s) { return static_cast<float>(pcg_output(s)) * 2.3283064365386963e-10f; }

// ---------------------------------------------------------------------------------- sin/cos
RT_HD void sincos_f(float xf, float &s_out, float &c_out) {
    const double x = static_cast<double>(xf);
    const double k = floor(x * 0.63661977236758134308 + 0.5);
    double r = x - k * 1.57079632679489661923;
    r = r - k * 6.12323399573676603587e-17;
    const double r2 = r * r;
    const double s =
        r + r * r2 *
                (-1.0 / 6.0 +
                 r2 * (1.0 / 120.0 +
                       r2 * (-1.0 / 5040.0 +
                             r2 * (1.0 / 362880.0 +
                                   r2 * (-1.0 / 39916800.0 +
                                         r2 * (1.0 / 6227020800.0 + r2 * (-1.0 / 1307674368000.0)))))));
    const double c =
        1.0 + r2 * (-0.5 +
                    r2 * (1.0 / 24.0 +
                          r2 * (-1.0 / 720.0 +
                                r2 * (1.0 / 40320.0 +
                                      r2 * (-1.0 / 3628800.0 +
                                            r2 * (1.0 / 479001600.0 +
                                                  r2 * (-1.0 / 87178291200.0 +
                                                        r2 * (1.0 / 20922789888000.0))))))));
    const long q = static_cast<long>(k) & 3L;
    double sv, cv;
    if (q == 0) { sv = s; cv = c; }
    else if (q == 1) { sv = c; cv = -s; }
    else if (q == 2) { sv = -s; cv = -c; }
    else { sv = -c; cv = s; }
    s_out = static_cast<float>(sv);
    c_out = static_cast<float>(cv);
}
// cos(radians(deg)) of spatialReuse.comp:67
RT_HD float cos_degrees(float deg) {
    float s, c;
    sincos_f(deg * 0.0174532924f, s, c);
    return c;
}

// ------------------------------------------------------------------------------------- BRDF
RT_HD float luminance(float r, float g, float b) {  // common.glsl:7-9
    return 0.2126f * r + 0.7152f * g + 0.0722f * b;
}
RT_HD float schlick(float c) {  // disneyBRDF.glsl:5-10
    const float m = gclamp(1.0f - c, 0.0f, 1.0f);
    const float sm = m * m;
    return sm * sm * m;
}
template <class A>
__device__ __forceinline__ float gtr2(A &m, float ndoth, float a) {  // disneyBRDF.glsl:13-18
    const float a2 = a * a;
    const float t = 1.0f + (a2 - 1.0f) * ndoth * ndoth;
    return m.div(a2, kPi * t * t);
}
template <class A>
__device__ __forceinline__ float smith_g(A &m, float ndotv, float alphaG) {  // disneyBRDF.glsl:20-25
    const float a = alphaG * alphaG;
    const float b = ndotv * ndotv;
    return m.rcp(fabsf(ndotv) + gmax(m.root(a + b - a * b), 0.0001f));
}

// Per-pixel constants of the BRDF that do not depend on the light: alpha, and the terms of
// cosOut. Hoisting them changes no rounding (same operations on the same operands).
struct Surface {
    f3 pos, n, wo;
    float cosOut, albLum, rough, metal;
    float a;          // max(0.001, rough^2)
    float fOut;       // schlick(cosOut)
    float gOut;       // smith_g(cosOut, a)
    float oneMinusMetal;
};
__device__ __forceinline__ Surface make_surface(f3 pos, f3 n, f3 cam, float albLum, float rough, float metal) {
    Surface s;
    s.pos = pos;
    s.n = n;
    s.wo = normalize(cam - pos);
    s.cosOut = dot(n, s.wo);
    s.albLum = albLum;
    s.rough = rough;
    s.metal = metal;
    s.a = gmax(0.001f, rough * rough);
    s.fOut = schlick(s.cosOut);
    Near near;
    s.gOut = smith_g(near, s.cosOut, s.a);
    if (!near.ok) {
        Ieee ieee;
        s.gOut = smith_g(ieee, s.cosOut, s.a);
    }
    s.oneMinusMetal = 1.0f - metal;
    return s;
}

struct LightGeom {
    float cosIn, cosHalf, cosInHalf, geometry;
    bool below;
};
// restirUtils.glsl:7-25 (shared by evaluatePHat and evaluatePHatFull)
template <class A>
__device__ __forceinline__ LightGeom light_geometry(A &m, const Surface &s, f3 L, f3 LN, bool useLN) {
    LightGeom g{};
    f3 wi = L - s.pos;
    if (dot(wi, s.n) < 0.0f) {
        g.below = true;
        return g;
    }
    const float sqrDist = dot(wi, wi);
    wi = m.unit(wi, sqrDist);
    g.cosIn = dot(s.n, wi);
    const f3 hv = wi + s.wo;
    const f3 h = m.unit(hv, dot(hv, hv));
    g.cosHalf = dot(s.n, h);
    g.cosInHalf = dot(wi, h);
    g.geometry = m.div(g.cosIn, sqrDist);
    if (useLN) g.geometry *= fabsf(dot(wi, LN));
    g.below = false;
    return g;
}
// disneyBrdfDiffuseFactor (:27-33) and the specular factor Gs*Ds (:42-55)
template <class A>
__device__ __forceinline__ float diffuse_factor(A &m, const Surface &s, const LightGeom &g) {
    const float fin = schlick(g.cosIn);
    const float fd90 = 0.5f + 2.0f * g.cosInHalf * g.cosInHalf * s.rough;
    const float fd = gmix(1.0f, fd90, fin) * gmix(1.0f, fd90, s.fOut);
    return m.div_pi(fd * s.oneMinusMetal);
}
template <class A>
__device__ __forceinline__ float gs_ds(A &m, const Surface &s, const LightGeom &g) {
    const float ds = gtr2(m, g.cosHalf, s.a);
    float gs = smith_g(m, g.cosIn, s.a);
    gs *= s.gOut;
    return gs * ds;
}
// evaluatePHat, restirUtils.glsl:3-28 with disneyBrdfLuminance (disneyBRDF.glsl:82-90)
template <class A>
__device__ __forceinline__ float eval_phat_as(A &m, const Surface &s, f3 L, f3 LN, bool useLN, float emLum) {
    const LightGeom g = light_geometry(m, s, L, LN, useLN);
    if (g.below) return 0.0f;
    float brdf = 0.0f;
    if (!(g.cosIn < 0.0f)) {
        const float diffuse = s.albLum * diffuse_factor(m, s, g);
        const float fih = schlick(g.cosInHalf);
        const float gsds = gs_ds(m, s, g);
        const float specLum = gmix(0.04f, s.albLum, s.metal);
        const float fs = gmix(specLum, 1.0f, fih);
        brdf = diffuse + fs * gsds;
    }
    return emLum * brdf * g.geometry;
}
__device__ __forceinline__ float eval_phat(const Surface &s, f3 L, f3 LN, bool useLN, float emLum) {
    Near near;
    float p = eval_phat_as(near, s, L, LN, useLN, emLum);
    if (!near.ok) {
        Ieee ieee;
        p = eval_phat_as(ieee, s, L, LN, useLN, emLum);
    }
    return p;
}
// evaluatePHatFull, restirUtils.glsl:30-55 with disneyBrdfColor (disneyBRDF.glsl:73-81)
template <class A>
__device__ __forceinline__ f3 eval_phat_full_as(A &m, const Surface &s, f3 albedo, f3 L, f3 LN, bool useLN, f3 em) {
    const LightGeom g = light_geometry(m, s, L, LN, useLN);
    if (g.below) return f3{0.0f, 0.0f, 0.0f};
    f3 brdf{0.0f, 0.0f, 0.0f};
    if (!(g.cosIn < 0.0f)) {
        const float df = diffuse_factor(m, s, g);
        const float fih = schlick(g.cosInHalf);
        const float gsds = gs_ds(m, s, g);
        const float alb[3] = {albedo.x, albedo.y, albedo.z};
        float out[3];
        for (int c = 0; c < 3; ++c) {
            const float diffuse = alb[c] * df;
            const float sc = gmix(0.04f, alb[c], s.metal);
            const float fs = gmix(sc, 1.0f, fih);
            out[c] = diffuse + fs * gsds;
        }
        brdf = f3{out[0], out[1], out[2]};
    }
    return f3{em.x * brdf.x * g.geometry, em.y * brdf.y * g.geometry, em.z * brdf.z * g.geometry};
}
__device__ __forceinline__ f3 eval_phat_full(const Surface &s, f3 albedo, f3 L, f3 LN, bool useLN, f3 em) {
    Near near;
    f3 p = eval_phat_full_as(near, s, albedo, L, LN, useLN, em);
    if (!near.ok) {
        Ieee ieee;
        p = eval_phat_full_as(ieee, s, albedo, L, LN, useLN, em);
    }
    return p;
}

// ------------------------------------------------------------------------------- reservoirs
// Register-resident reservoir with the fields of restirStructs.glsl:19-34.
struct Res {
    f3 pos;
    float emLum;
    float4 normal;
    int32_t lightIndex;
    float pHat, sumW, w;
    uint32_t M;
};
RT_HD Res res_zero() {
    Res r;
    r.pos = f3{0.0f, 0.0f, 0.0f};
    r.emLum = 0.0f;
    r.normal = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    r.lightIndex = 0;
    r.pHat = r.sumW = r.w = 0.0f;
    r.M = 0u;
    return r;
}
// updateReservoirAt, reservoir.glsl:6-26, in two parts: whether the sample is taken (u: the update's
// uniform draw), and the update, which returns that
__device__ __forceinline__ bool res_takes(Res &r, float weight, float u) {
    r.sumW += weight;
    if (weight == 0.0f) return false;  // u < 0 / sumW never holds
    const float rp = mid_range(weight) && mid_range(r.sumW) ? div_near(weight, r.sumW, rcp_near(r.sumW))
                                                            : weight / r.sumW;
    return u < rp;
}
__device__ __forceinline__ bool res_update_u(Res &r, float weight, f3 pos, float4 n, float emLum, int32_t li, float pHat,
                                             float w, float u) {
    if (res_takes(r, weight, u)) {
        r.pos = pos;
        r.emLum = emLum;
        r.normal = n;
        r.lightIndex = li;
        r.pHat = pHat;
        r.w = w;
        return true;
    }
    return false;
}
__device__ __forceinline__ void res_update(Res &r, float weight, f3 pos, float4 n, float emLum, int32_t li, float pHat,
                                           float w, Pcg &rng) {
    res_update_u(r, weight, pos, n, emLum, li, pHat, w, pcg_float(rng));
}
// addSampleToReservoir, reservoir.glsl:28-42 (u: the update's uniform draw). Its W = sumW / (M
// pHat), of the moment a sample is taken, is left to ris_w: only the last one taken keeps it.
struct RisTaken {
    float sumW = 0.0f;
    uint32_t M = 0u;  // 0: none was taken
};
__device__ __forceinline__ float ris_weight(float pHat, float sampleP) {
    return (mid_range(pHat) || __float_as_uint(pHat) == 0u) && mid_range(sampleP)
               ? div_near(pHat, sampleP, rcp_near(sampleP))
               : pHat / sampleP;
}
__device__ __forceinline__ void res_add_sample_u(Res &r, RisTaken &taken, f3 pos, float4 n, float emLum, int32_t li,
                                                 float pHat, float sampleP, float u) {
    r.M += 1u;
    if (res_update_u(r, ris_weight(pHat, sampleP), pos, n, emLum, li, pHat, 0.0f, u)) {
        taken.sumW = r.sumW;
        taken.M = r.M;
    }
}
// W of the sample taken last (0 when none was)
__device__ __forceinline__ float ris_w(const RisTaken &taken, float pHat) {
    return taken.M ? taken.sumW / (static_cast<float>(taken.M) * pHat) : 0.0f;
}
// combineReservoirs, reservoir.glsl:44-64
__device__ __forceinline__ void res_combine(Res &self, const Res &o, float pHat, Pcg &rng) {
    self.M += o.M;
    const float weight = pHat * o.w * static_cast<float>(o.M);
    if (weight > 0.0f) res_update(self, weight, o.pos, o.normal, o.emLum, o.lightIndex, pHat, o.w, rng);
    if (self.w > 0.0f) self.w = self.sumW / (static_cast<float>(self.M) * self.pHat);
}

}  // namespace rt
