// mlp.hip — the learned light proposal on gfx950 (no reference counterpart).
//
// A 128 -> 128 -> 128 -> 128 -> K ReLU MLP maps per-pixel features (position, normal and view
// direction with 6 sin/cos octaves, 114 values) to a softmax over K light clusters. The proposal
// mixes it with the reference's source distribution (alias table over light power):
//   q(l | x) = (1 - mix) * pi_x(c(l)) * p_within(l) + mix * p_src(l),   mix = 0.1,
// so q > 0 wherever p_src > 0 and RIS stays unbiased. Weights are bf16 (fp32 master copy, Adam);
// every product runs on v_mfma_f32_32x32x16_bf16 with fp32 accumulation.
//
// Kernels:
//   k_propose      fused inference per 2x2 pixel quad: features -> 4 MFMA layers -> softmax ->
//                  M candidates (l, q) for each of its pixels (K <= 256)
//   k_propose_wide the same for K up to 4096: the output layer streamed in 64-cluster blocks
//   k_features     features of listed pixels (bf16), for training and tests
//   k_mlp_forward, k_mlp_backward, k_mlp_grads   training: a tile of samples through all layers and
//                  back, and the weight and bias gradients as partial sums over ranges of samples
//   k_softmax_ce   mean cross-entropy of the logits against target clusters, and dlogits
//   k_sum_partials the partial sums of the gradients and the loss, in fixed order
//   k_adam         Adam step on fp32 master weights, refreshes the bf16 copy
//   k_mlp_init     seeded He-uniform initialisation
#include <algorithm>

#include "../../include/restir_abi.h"
#include "carve.h"
#include "kernels.h"
#include "mlp.h"

namespace rm {

using rt::f3;

// ------------------------------------------------------------------------------ features ---
// Writes the 128 bf16 features of one surface point. The scalars are the position normalised
// to the scene box, the normal and the unit view direction; raw position and normal first, then
// sin/cos(2^k * pi * s) for k = 0..5 (double-angle recurrences from k = 0), zero padding last.
__device__ __forceinline__ void make_features(f3 pos, f3 n, f3 cam, const float *lo, const float *hi,
                                              uint16_t *dst) {
    float s[9];
    const float pp[3] = {pos.x, pos.y, pos.z};
    for (int k = 0; k < 3; ++k) {
        const float c = 0.5f * (lo[k] + hi[k]), h = 0.5f * (hi[k] - lo[k]);
        s[k] = (pp[k] - c) / h;
    }
    s[3] = n.x;
    s[4] = n.y;
    s[5] = n.z;
    f3 v = cam - pos;
    const float vl = sqrtf(rt::dot(v, v));
    v = vl > 0.0f ? v / vl : f3{0.0f, 0.0f, 0.0f};
    s[6] = v.x;
    s[7] = v.y;
    s[8] = v.z;
    // dst is 4-byte aligned and every pair below starts at an even index: one packed
    // conversion and one 32-bit store per pair
    uint32_t *d2 = reinterpret_cast<uint32_t *>(dst);
    for (int k = 0; k < 3; ++k) d2[k] = f2bf2(s[2 * k], s[2 * k + 1]);
    for (int i = 0; i < 9; ++i) {
        float sn, cs;
        sincosf(3.14159265358979f * s[i], &sn, &cs);
        for (int f = 0; f < 6; ++f) {
            d2[3 + 6 * i + f] = f2bf2(sn, cs);
            const float s2 = 2.0f * sn * cs, c2 = (cs - sn) * (cs + sn);
            sn = s2;
            cs = c2;
        }
    }
    for (int k = kFeatures / 2; k < kIn / 2; ++k) d2[k] = 0u;
}

struct FeatArgs {
    rk::GView g;
    f3 cam;
    float lo[3], hi[3];
};

__device__ __forceinline__ bool pixel_features(const FeatArgs &f, uint32_t p, uint16_t *dst) {
    const f3 pos = f3{f.g.pos[p], f.g.pos[f.g.P + p], f.g.pos[2 * f.g.P + p]};
    const f3 n = rk::load_normal(f.g, p);
    make_features(pos, n, f.cam, f.lo, f.hi, dst);
    return rt::dot(n, n) != 0.0f;
}

__global__ __launch_bounds__(256) void k_features(const FeatArgs f, const uint32_t *pixels, uint32_t n,
                                                  uint16_t *out) {
    const uint32_t b = blockIdx.x * 256u + threadIdx.x;
    if (b >= n) return;
    uint16_t *dst = out + static_cast<size_t>(b) * kIn;
    if (pixels[b] < f.g.W * f.g.H) {
        pixel_features(f, pixels[b], dst);
    } else {
        for (int k = 0; k < kIn; ++k) dst[k] = 0;
    }
}

// ----------------------------------------------------------------- forward and backward ------
// Training works on a few thousand samples: what bounds it is the chain of launches and, inside
// one, of memory round trips, not the products (0.9 GFLOP at 4,096 samples and 256 clusters). So a
// workgroup takes 32 samples through all layers, its activations in LDS, each wave with all of a
// layer's weights for its 32 columns under way at once; and the weight gradients of all layers are
// one launch. As 11 launches of a 64x64-tile product (8.6 us each) and 8 others a step of 4,096
// samples took 144 us, now 56: forward 12, backward 14, gradients 13, their sums 8. 4,096 clusters
// 375 -> 277 us, 16,384 samples 320 -> 125, 64 samples 97 -> 40.
constexpr int kMlpRows = 32;     // samples per workgroup
constexpr int kRow = kIn + 8;    // padded LDS row (bf16) against bank conflicts

// the product's operands and result are laid out as mlp.h says; row of a lane's result element i
__device__ __forceinline__ int acc_row(int lane, int i) { return 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3); }
__device__ __forceinline__ f32x16 acc_zero() {
    f32x16 acc;
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
    return acc;
}
// a 32-sample LDS tile to rows of kHidden
__device__ __forceinline__ void store_tile(const uint16_t (*tile)[kRow], uint16_t *dst) {
#pragma unroll
    for (int e = threadIdx.x; e < kMlpRows * (kHidden / 8); e += 256) {
        const int r = e / (kHidden / 8), c = (e % (kHidden / 8)) * 8;
        *reinterpret_cast<uint4 *>(dst + static_cast<size_t>(r) * kHidden + c) = *reinterpret_cast<const uint4 *>(&tile[r][c]);
    }
}

struct ForwardArgs {
    const uint16_t *X, *wbf;
    const float *bias;
    uint16_t *H[3];  // hidden activations
    float *Z;        // logits
    int K, cols;     // clusters; those that a workgroup computes (blockIdx.y-th group, the last may have fewer)
};
// Workgroup (x, y): the hidden layers of samples 32x .. 32x + 31 (kept by y = 0), then their logits
// of the y-th group of clusters: with few samples the output layer of thousands of clusters needs more
// workgroups than there are tiles of samples. Weights are fetched while the results before them are
// written; a load between them and their use (a bias) would wait for them.
__global__ __launch_bounds__(256, 4) void k_mlp_forward(const ForwardArgs a) {
    __shared__ __align__(16) uint16_t act[2][kMlpRows][kRow];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r0 = blockIdx.x * kMlpRows;
    const int row = lane & 31, k8 = 8 * (lane >> 5);
    bf16x8 x[kIn / 16], w[kIn / 16];
    auto load_w = [&](const uint16_t *W, int col) {
#pragma unroll
        for (int s = 0; s < kIn / 16; ++s) w[s] = *reinterpret_cast<const bf16x8 *>(W + static_cast<size_t>(col) * kIn + 16 * s + k8);
    };
#pragma unroll
    for (int s = 0; s < kIn / 16; ++s)
        x[s] = *reinterpret_cast<const bf16x8 *>(a.X + static_cast<size_t>(r0 + row) * kIn + 16 * s + k8);
    load_w(a.wbf + w_off(0), 32 * wave + row);
    const int begin = blockIdx.y * a.cols, end = begin + a.cols < a.K ? begin + a.cols : a.K;
    int at = begin + 32 * wave;  // the wave's 32 clusters
    for (int l = 0; l < 3; ++l) {
        const int col = 32 * wave + row;
        const float bias = a.bias[b_off(l) + col];
        f32x16 acc = acc_zero();
#pragma unroll
        for (int s = 0; s < kIn / 16; ++s) acc = mfma32(x[s], w[s], acc);
        // the next layer's weights while this one's results go through LDS
        if (l < 2 || at < end) load_w(a.wbf + w_off(l + 1), (l < 2 ? 32 * wave : at) + row);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const float v = acc[i] + bias;
            act[l & 1][acc_row(lane, i)][col] = f2bf(v > 0.0f ? v : 0.0f);
        }
        __syncthreads();
#pragma unroll
        for (int s = 0; s < kIn / 16; ++s) x[s] = *reinterpret_cast<const bf16x8 *>(&act[l & 1][row][16 * s + k8]);
        if (blockIdx.y == 0) store_tile(act[l & 1], a.H[l] + static_cast<size_t>(r0) * kHidden);
    }
    for (; at < end; at += 128) {
        const int col = at + row;
        const float bias = a.bias[b_off(3) + col];
        f32x16 acc = acc_zero();
#pragma unroll
        for (int s = 0; s < kIn / 16; ++s) acc = mfma32(x[s], w[s], acc);
        if (at + 128 < end) load_w(a.wbf + w_off(3), col + 128);  // while the logits are stored
#pragma unroll
        for (int i = 0; i < 16; ++i) a.Z[static_cast<size_t>(r0 + acc_row(lane, i)) * a.K + col] = acc[i] + bias;
    }
}

struct BackwardArgs {
    const uint16_t *dZ, *wbf;
    const uint16_t *H[3];
    uint16_t *dH[3];  // gradients at the hidden layers' outputs before their ReLU
    int K;
};
// dIn[b][k] = sum over o of dY[b][o] W[o][k], where the layer below was positive: the output layer's
// weights come through LDS 128 clusters at a time, then the hidden layers' (a wave reads a column of
// them there, eight consecutive o as eight 16-bit reads), the next ones on their way in registers.
__global__ __launch_bounds__(256) void k_mlp_backward(const BackwardArgs a) {
    __shared__ __align__(16) uint16_t wt[kHidden][kRow];
    __shared__ __align__(16) uint16_t dy[kMlpRows][kRow];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r0 = blockIdx.x * kMlpRows;
    const int row = lane & 31, k8 = 8 * (lane >> 5), col = 32 * wave + row;
    const int chunks = (a.K + kHidden - 1) / kHidden;  // of 128 clusters; one of 64 if K = 64
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    u32x4 next[8];
    auto rows_of = [&](int c) { return c < chunks && a.K < kHidden ? a.K : kHidden; };
    auto fetch = [&](int c) {  // chunk c of the output layer, then layers 2 and 1
        const uint16_t *src = c < chunks ? a.wbf + w_off(3) + static_cast<size_t>(c) * kHidden * kIn : a.wbf + w_off(2 - (c - chunks));
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int at = e * 256 + threadIdx.x;
            if (at / (kIn / 8) < rows_of(c)) next[e] = *reinterpret_cast<const u32x4 *>(src + at * 8);
        }
    };
    fetch(0);
    f32x16 acc = acc_zero();
    for (int c = 0; c < chunks + 2; ++c) {
        const int rows = rows_of(c);
        __syncthreads();
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int at = e * 256 + threadIdx.x, r = at / (kIn / 8);
            if (r < rows) *reinterpret_cast<u32x4 *>(&wt[r][(at % (kIn / 8)) * 8]) = next[e];
        }
        __syncthreads();
        if (c + 1 < chunks + 2) fetch(c + 1);
        const int below = c < chunks ? 2 : 1 - (c - chunks);  // the hidden layer that receives the gradient
        const bool ends = c >= chunks - 1;
        uint16_t gate[16];
        if (ends)
#pragma unroll
            for (int i = 0; i < 16; ++i) gate[i] = a.H[below][static_cast<size_t>(r0 + acc_row(lane, i)) * kHidden + col];
        bf16x8 x[kHidden / 16];
#pragma unroll
        for (int s = 0; s < kHidden / 16; ++s)
            if (16 * s < rows)
                x[s] = c < chunks ? *reinterpret_cast<const bf16x8 *>(a.dZ + static_cast<size_t>(r0 + row) * a.K + c * kHidden + 16 * s + k8)
                                  : *reinterpret_cast<const bf16x8 *>(&dy[row][16 * s + k8]);
#pragma unroll
        for (int s = 0; s < kHidden / 16; ++s) {
            if (16 * s >= rows) continue;
            uint32_t d[4];
#pragma unroll
            for (int j = 0; j < 4; ++j)
                d[j] = static_cast<uint32_t>(wt[16 * s + k8 + 2 * j][col]) | (static_cast<uint32_t>(wt[16 * s + k8 + 2 * j + 1][col]) << 16);
            acc = mfma32(x[s], __builtin_bit_cast(bf16x8, make_uint4(d[0], d[1], d[2], d[3])), acc);
        }
        if (!ends) continue;
        __syncthreads();  // the other waves' reads of dy
#pragma unroll
        for (int i = 0; i < 16; ++i) dy[acc_row(lane, i)][col] = bf2f(gate[i]) > 0.0f ? f2bf(acc[i] + 0.0f) : 0;
        acc = acc_zero();
        __syncthreads();
        store_tile(dy, a.dH[below] + static_cast<size_t>(r0) * kHidden);
    }
}

// The gradients of all layers' weights and biases over the samples, as partial sums that
// k_sum_partials adds in a fixed order: gW[o][k] = sum over b of dY[b][o] in[b][k] in `split` ranges
// of b, 64x64 per workgroup, and gb[o] = sum over b of dY[b][o] in ranges of 64.
struct GradLayer {
    const uint16_t *dY, *in;  // [n][N], [n][kIn]
    float *pw, *pb;
    int N, split;
    uint32_t firstW, firstB;  // workgroups before this layer's
};
struct GradArgs {
    GradLayer layer[4];
    int n;
    uint32_t weightGroups;  // workgroups of the weights, then those of the biases
};
// 64x64 outputs per 256-lane workgroup; each wave owns a 32x32 quarter. The samples advance in steps
// of 32 through LDS, both operands transposed on the way in so that every fragment is eight
// consecutive bf16; the next step's are on their way in registers.
__global__ __launch_bounds__(256) void k_mlp_grads(const GradArgs a) {
    __shared__ __align__(16) uint16_t As[64][40];
    __shared__ __align__(16) uint16_t Bt[64][40];
    __shared__ float red[4][64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (blockIdx.x >= a.weightGroups) {
        const uint32_t job = blockIdx.x - a.weightGroups;
        int l = 3;
        while (l > 0 && job >= a.layer[l - 1].firstB) --l;
        const GradLayer &g = a.layer[l];
        const uint32_t local = job - g.firstB, tiles = static_cast<uint32_t>(g.N) / 64u;
        const int c = static_cast<int>(local % tiles) * 64 + lane, chunk = static_cast<int>(local / tiles);
        float sum = 0.0f;
#pragma unroll
        for (int r = 0; r < 16; ++r) sum += bf2f(g.dY[static_cast<size_t>(chunk * 64 + wave + 4 * r) * g.N + c]);
        red[wave][lane] = sum;
        __syncthreads();
        if (wave == 0) g.pb[static_cast<size_t>(chunk) * g.N + c] = ((red[0][lane] + red[1][lane]) + red[2][lane]) + red[3][lane];
        return;
    }
    int l = 3;
    while (l > 0 && blockIdx.x >= a.layer[l - 1].firstW) --l;
    const GradLayer &g = a.layer[l];
    const uint32_t local = blockIdx.x - g.firstW, tiles = 2u * static_cast<uint32_t>(g.N) / 64u;
    const int m0 = static_cast<int>(local % tiles) / 2 * 64, n0 = static_cast<int>(local % 2u) * 64;
    const int part = static_cast<int>(local / tiles), each = a.n / g.split, kBeg = part * each, kEnd = kBeg + each;
    const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
    const int kk = tid >> 3, r = (tid & 7) * 8;
    uint4 va, vb;
    auto fetch = [&](int k0) {
        va = *reinterpret_cast<const uint4 *>(&g.dY[static_cast<size_t>(k0 + kk) * g.N + m0 + r]);
        vb = *reinterpret_cast<const uint4 *>(&g.in[static_cast<size_t>(k0 + kk) * kIn + n0 + r]);
    };
    fetch(kBeg);
    f32x16 acc = acc_zero();
    for (int k0 = kBeg; k0 < kEnd; k0 += 32) {
        const uint32_t wa[4] = {va.x, va.y, va.z, va.w}, wb[4] = {vb.x, vb.y, vb.z, vb.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            As[r + 2 * i][kk] = static_cast<uint16_t>(wa[i] & 0xffffu);
            As[r + 2 * i + 1][kk] = static_cast<uint16_t>(wa[i] >> 16);
            Bt[r + 2 * i][kk] = static_cast<uint16_t>(wb[i] & 0xffffu);
            Bt[r + 2 * i + 1][kk] = static_cast<uint16_t>(wb[i] >> 16);
        }
        __syncthreads();
        if (k0 + 32 < kEnd) fetch(k0 + 32);
#pragma unroll
        for (int ks = 0; ks < 32; ks += 16) {
            const bf16x8 fa = *reinterpret_cast<const bf16x8 *>(&As[wm + (lane & 31)][ks + 8 * (lane >> 5)]);
            const bf16x8 fb = *reinterpret_cast<const bf16x8 *>(&Bt[wn + (lane & 31)][ks + 8 * (lane >> 5)]);
            acc = mfma32(fa, fb, acc);
        }
        __syncthreads();
    }
    float *P = g.pw + static_cast<size_t>(part) * g.N * kIn;
#pragma unroll
    for (int i = 0; i < 16; ++i) P[static_cast<size_t>(m0 + wm + acc_row(lane, i)) * kIn + n0 + wn + (lane & 31)] = acc[i];
}

// ----------------------------------------------------------------------------- loss/grad ----
// dZ = (softmax(z) - onehot(target)) / n_valid for sample b with mask, 0 otherwise (bf16), by the
// 64 lanes of one wave (lanes stride over the K logits, reductions across the wave); returns the
// sample's loss divided by n_valid (0 for a sample that does not train).
__device__ __forceinline__ float softmax_ce_row(const float *Z, int K, const int32_t *target, const uint32_t *mask,
                                                int n, const uint32_t *nValid, uint16_t *dZ, int b, int lane) {
    if (b >= n) return 0.0f;
    const float *z = Z + static_cast<size_t>(b) * K;
    uint16_t *d = dZ + static_cast<size_t>(b) * K;
    const int t = target[b];
    if (!mask[b] || t < 0 || t >= K) {  // an out-of-range target does not train
        for (int c = lane; c < K; c += 64) d[c] = 0;
        return 0.0f;
    }
    const float inv = 1.0f / static_cast<float>(*nValid);
    float mx = -INFINITY;
    for (int c = lane; c < K; c += 64) mx = fmaxf(mx, z[c]);
    for (int off = 32; off > 0; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off));
    float se = 0.0f;
    for (int c = lane; c < K; c += 64) se += expf(z[c] - mx);
    for (int off = 32; off > 0; off >>= 1) se += __shfl_xor(se, off);
    const float rse = 1.0f / se;
    for (int c = lane; c < K; c += 64) d[c] = f2bf((expf(z[c] - mx) * rse - (c == t ? 1.0f : 0.0f)) * inv);
    return -(z[t] - mx - logf(se)) * inv;
}

// The mean cross-entropy's gradient for 4 samples per workgroup (softmax_ce_row); the loss of the
// workgroup's samples, added in sample order, goes to lossPart[blockIdx.x] (k_sum_partials then
// adds the workgroups' sums in order).
__global__ __launch_bounds__(256) void k_softmax_ce(const float *Z, int K, const int32_t *target,
                                                    const uint32_t *mask, int n,
                                                    const uint32_t *nValid, uint16_t *dZ,
                                                    float *lossPart) {
    __shared__ float wl[4];
    const int w = static_cast<int>(threadIdx.x >> 6);
    const int lane = static_cast<int>(threadIdx.x & 63);
    const float sampleLoss = softmax_ce_row(Z, K, target, mask, n, nValid, dZ, blockIdx.x * 4 + w, lane);
    if (lane == 0) wl[w] = sampleLoss;
    __syncthreads();
    if (threadIdx.x == 0) lossPart[blockIdx.x] = ((wl[0] + wl[1]) + wl[2]) + wl[3];
}

// samples that train, by one workgroup
__global__ __launch_bounds__(1024) void k_count_mask(const uint32_t *mask, uint32_t n, uint32_t *count) {
    __shared__ uint32_t waves[16];
    uint32_t c = 0;
    for (uint32_t i = threadIdx.x; i < n; i += 1024u) c += mask[i] != 0u ? 1u : 0u;
    for (int off = 32; off > 0; off >>= 1) c += __shfl_xor(c, off);
    if ((threadIdx.x & 63u) == 0u) waves[threadIdx.x >> 6] = c;
    __syncthreads();
    if (threadIdx.x != 0) return;
    uint32_t sum = 0;
    for (int w = 0; w < 16; ++w) sum += waves[w];
    *count = sum;
}

__global__ void k_copy_f32(const float *src, float *dst) { *dst = *src; }

// 8 reductions in one launch: for segment j, out_j[i] = sum over s < nParts_j of
// part_j[s * count_j + i], in order of s. Lane t of the grid takes element t of the segments laid
// end to end; a last workgroup adds the loss, one number of nLoss parts, through LDS (as one lane's
// loads from memory these took 22 us of 4,096 samples' 1,024).
struct SumSegments {
    const float *part[8];
    float *out[8];
    int nParts[8];
    int64_t count[8];
    const float *lossPart;
    float *loss;
    int nLoss;
};
__global__ __launch_bounds__(256) void k_sum_partials(const SumSegments a) {
    if (blockIdx.x == gridDim.x - 1) {
        __shared__ float v[1024];
        float sum = 0.0f;
        for (int s0 = 0; s0 < a.nLoss; s0 += 1024) {
#pragma unroll
            for (int e = threadIdx.x; e < 1024; e += 256)
                if (s0 + e < a.nLoss) v[e] = a.lossPart[s0 + e];
            __syncthreads();
            if (threadIdx.x == 0) {
                const int end = a.nLoss - s0 < 1024 ? a.nLoss - s0 : 1024;
#pragma unroll 16
                for (int e = 0; e < end; ++e) sum += v[e];
            }
            __syncthreads();
        }
        if (threadIdx.x == 0) *a.loss = sum;
        return;
    }
    int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    int j = 0;
    while (j < 8 && i >= a.count[j]) i -= a.count[j++];
    if (j >= 8) return;
    const float *part = a.part[j];
    const int64_t count = a.count[j];
    float sum = 0.0f;
    // unrolled so that the loads of 16 parts are in flight together; the additions stay in order
#pragma unroll 16
    for (int s = 0; s < a.nParts[j]; ++s) sum += part[s * count + i];
    a.out[j][i] = sum;
}

// --------------------------------------------------------------------------------- Adam -----
struct AdamArgs {
    float *w;          // fp32 master weights (nW), then biases (nB) in `b`
    float *b;
    uint16_t *wbf;     // bf16 copy of the weights
    const float *gw, *gb;
    float *m, *v;      // nW + nB each
    uint32_t nW, nB;
    float lr, b1, b2, eps;
    double b1d, b2d;               // b1, b2 in double for the bias corrections
    uint32_t stepHost;             // step t, unless stepDev is set
    const uint32_t *stepDev;
};

// b^t by binary exponentiation in double (the same products in the same order wherever t is
// read), for the bias corrections 1 - b1^t and 1 - b2^t.
__host__ __device__ inline double pow_step(double b, uint32_t t) {
    double r = 1.0;
    while (t) {
        if (t & 1u) r *= b;
        b *= b;
        t >>= 1;
    }
    return r;
}

// Advances the device step count by one (lane 0; a vector atomic).
__global__ void k_adam_count(uint32_t *step) {
    if (threadIdx.x == 0) atomicAdd(step, 1u);
}

// Adam step; skipped when the batch held no training sample (*nValid == 0; nValid null: always).
__global__ __launch_bounds__(256) void k_adam_guarded(const AdamArgs a, const uint32_t *nValid) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i >= a.nW + a.nB || (nValid && *nValid == 0u)) return;
    const bool isW = i < a.nW;
    const float g = isW ? a.gw[i] : a.gb[i - a.nW];
    const uint32_t t = a.stepDev ? *a.stepDev : a.stepHost;
    const float c1 = static_cast<float>(1.0 - pow_step(a.b1d, t));
    const float c2 = static_cast<float>(1.0 - pow_step(a.b2d, t));
    const float m = a.b1 * a.m[i] + (1.0f - a.b1) * g;
    const float v = a.b2 * a.v[i] + (1.0f - a.b2) * g * g;
    a.m[i] = m;
    a.v[i] = v;
    const float step = a.lr * (m / c1) / (sqrtf(v / c2) + a.eps);
    if (isW) {
        const float w = a.w[i] - step;
        a.w[i] = w;
        a.wbf[i] = f2bf(w);
    } else {
        a.b[i - a.nW] -= step;
    }
}

// He-uniform weights U(-sqrt(6/fan_in), sqrt(6/fan_in)) from PCG32(seed, element index); zero
// biases except the output layer, which starts at `prior` (log cluster power shares) so the
// untrained proposal already samples clusters by power. Adam moments start at zero.
__global__ __launch_bounds__(256) void k_mlp_init(float *w, uint16_t *wbf, float *b, float *m, float *v,
                                                  uint32_t nW, uint32_t nB, uint32_t K, const float *prior,
                                                  uint64_t seed) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i < nW) {
        rt::Pcg r = rt::pcg_seed(seed, i);
        const float u = rt::pcg_float(r) * 2.0f - 1.0f;
        const float val = u * sqrtf(6.0f / static_cast<float>(kIn));
        w[i] = val;
        wbf[i] = f2bf(val);
    }
    if (i < nB) b[i] = (i >= 3u * kHidden) ? prior[i - 3u * kHidden] : 0.0f;
    if (i < nW + nB) {
        m[i] = 0.0f;
        v[i] = 0.0f;
    }
    (void)K;
}

// ------------------------------------------------------------------ training-sample gather --
struct GatherArgs {
    FeatArgs f;
    const restir_reservoir *res;
    const int32_t *lightCluster;
    int32_t nLights;  // lights the clusters cover (the alias table's index space)
    int32_t triBase;  // index of triangle light 0 in that space, -1 if it has none
    uint32_t npx, n, seed;
    uint16_t *X;
    int32_t *target;
    uint32_t *mask, *nValid;
    uint32_t *pixels;
};

// Sample b takes a pseudo-random pixel; it trains (mask = 1) if that pixel's final reservoir
// holds a light of the clustered index space with W > 0, with the light's cluster as the target
// (a reservoir names triangle light t as -1 - t).
__global__ __launch_bounds__(256) void k_train_gather(const GatherArgs a) {
    const uint32_t b = blockIdx.x * 256u + threadIdx.x;
    if (b >= a.n) return;
    rt::Pcg r = rt::pcg_seed(a.seed, b);
    const uint32_t p = rt::pcg_next(r) % a.npx;
    a.pixels[b] = p;
    const bool surface = pixel_features(a.f, p, a.X + static_cast<size_t>(b) * kIn);
    const float4 q2 = reinterpret_cast<const float4 *>(a.res + p)[2];  // lightIndex, pHat, sumW, w
    const int32_t li = __float_as_int(q2.x);
    const int32_t j = li >= 0 ? li : (a.triBase >= 0 ? a.triBase + (-1 - li) : -1);
    const bool ok = surface && j >= 0 && j < a.nLights && q2.w > 0.0f && q2.z > 0.0f;
    a.mask[b] = ok ? 1u : 0u;
    a.target[b] = ok ? a.lightCluster[j] : 0;
    if (ok) atomicAdd(a.nValid, 1u);
}

// ------------------------------------------------------------------- fused inference -------
struct ProposeArgs {
    FeatArgs f;
    const uint16_t *wbf;   // W1..W4 bf16 [out][in]
    const float *bias;
    int K;
    uint32_t npx, M, seed;
    float mix;             // weight of the source distribution
    // proposal tables
    const float4 *alias;   // global alias table (aliasTableColumn)
    int32_t nAlias;
    const int32_t *lightCluster;
    const float *lightPWithin;
    const int32_t *clusterBegin, *clusterCount, *clusterLights;
    const float4 *clusterAlias;  // per-cluster alias columns (alias = local index)
    const float4 *clusterFused;  // per slot: {prob, light, alias light, p_within}, {alias p_within, p_src, alias p_src, 0}
    int32_t *candLight;
    float *candQ;
    uint8_t *slots;      // k_propose_wide: nSlots workgroups' numerators and running sums,
    uint32_t *slotBusy;  // and which of them a workgroup holds
    uint32_t nSlots;
    uint32_t slotBytes;  // (a 64-bit stride: 123 scalars spilled instead of 82, 1,130 us for 1,105)
};


__device__ __forceinline__ void stage_weights(uint16_t *wbuf, const uint16_t *src, int rows) {
    // rows x 128 bf16 from global into LDS rows of kRow, 16 bytes per lane per step
    for (int e = threadIdx.x; e < rows * (kIn / 8); e += blockDim.x) {
        const int r = e / (kIn / 8), c = (e % (kIn / 8)) * 8;
        *reinterpret_cast<uint4 *>(&wbuf[r * kRow + c]) = *reinterpret_cast<const uint4 *>(&src[r * kIn + c]);
    }
}

__device__ __forceinline__ float4 unpack_h4(uint2 v) {  // four fp16 -> float
    const float2 lo = __half22float2(__builtin_bit_cast(__half2, v.x));
    const float2 hi = __half22float2(__builtin_bit_cast(__half2, v.y));
    return make_float4(lo.x, lo.y, hi.x, hi.y);
}

// The pixel whose features stand for quad (qx, qy): its first surface pixel in the order
// (0,0), (1,0), (0,1), (1,1) inside the image, else its top-left pixel.
__device__ __forceinline__ uint32_t quad_pixel(const rk::GView &g, uint32_t qx, uint32_t qy) {
    const uint32_t x0 = 2 * qx, y0 = 2 * qy;
    for (int j = 0; j < 4; ++j) {
        const uint32_t x = x0 + (j & 1), y = y0 + (j >> 1);
        if (x >= g.W || y >= g.H) continue;
        const uint32_t p = y * g.W + x;
        const f3 nq = rk::load_normal(g, p);
        if ((nq.x * nq.x + nq.y * nq.y) + nq.z * nq.z != 0.0f) return p;
    }
    return y0 * g.W + x0;
}

typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

// lanes 32..63 of x change places with lanes 0..31 of y
__device__ __forceinline__ void swap_halves(uint32_t &x, uint32_t &y) {
    const auto r = __builtin_amdgcn_permlane32_swap(x, y, false, false);
    x = r[0];
    y = r[1];
}
__device__ __forceinline__ void swap_halves(float &x, float &y) {
    uint32_t a = __float_as_uint(x), b = __float_as_uint(y);
    swap_halves(a, b);
    x = __uint_as_float(a);
    y = __uint_as_float(b);
}

// a barrier for LDS alone: __syncthreads would also wait for the global stores under way
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// 64 outputs of a layer for the wave's 32 quads: rows of staged weights times the activations, on
// top of the bias. The first half's weights are all read before its products and the second's while
// they run: a read takes as long as four products, and left to itself the compiler puts each read
// right before its product.
__device__ __forceinline__ void wide_blocks(const uint16_t *w, const float *bias, const bf16x8 (&h)[kIn / 16], int lane,
                                            f32x16 &z0, f32x16 &z1) {
    constexpr int kSteps = kIn / 16;
    auto start = [&](f32x16 &z, const float *b) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const float4 v = *reinterpret_cast<const float4 *>(b + 8 * g + 4 * (lane >> 5));
            z[4 * g] = v.x;
            z[4 * g + 1] = v.y;
            z[4 * g + 2] = v.z;
            z[4 * g + 3] = v.w;
        }
    };
    const uint16_t *at = w + (lane & 31) * kRow + 8 * (lane >> 5);
    bf16x8 f0[kSteps], f1[kSteps];
    start(z0, bias);
    start(z1, bias + 32);
#pragma unroll
    for (int s = 0; s < kSteps; ++s) f0[s] = *reinterpret_cast<const bf16x8 *>(at + 16 * s);
#pragma unroll
    for (int s = 0; s < kSteps; ++s) {
        z0 = mfma32(f0[s], h[s], z0);
        f1[s] = *reinterpret_cast<const bf16x8 *>(at + 32 * kRow + 16 * s);
    }
#pragma unroll
    for (int s = 0; s < kSteps; ++s) z1 = mfma32(f1[s], h[s], z1);
    __builtin_amdgcn_sched_group_barrier(0x100, 8 + kSteps, 0);  // LDS reads: both biases, the first half
#pragma unroll
    for (int s = 0; s < kSteps; ++s) {
        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);    // a product
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // a read
    }
    __builtin_amdgcn_sched_group_barrier(0x8, kSteps, 0);
}

// A hidden layer for the wave's 32 quads: its 128 outputs, clamped, as the next layer's operand.
__device__ __forceinline__ void wide_hidden(const uint16_t *w, const float *bias, bf16x8 (&h)[kIn / 16], int lane) {
    bf16x8 out[kIn / 16];
    f32x16 z[2];
#pragma unroll
    for (int nb = 0; nb < kHidden / 32; ++nb) {
        if (nb % 2 == 0) wide_blocks(w + 32 * nb * kRow, bias + 32 * nb, h, lane, z[0], z[1]);
        const f32x16 &acc = z[nb % 2];
        uint32_t d[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float lo = acc[2 * i], hi = acc[2 * i + 1];
            d[i] = f2bf2(lo > 0.0f ? lo : 0.0f, hi > 0.0f ? hi : 0.0f);
        }
        // outputs 8g + 4 * (lane / 32) + 0..3 lie in d[2g], d[2g + 1]; the operand wants
        // 8 * (lane / 32) + 0..7 of each 16
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            swap_halves(d[4 * s], d[4 * s + 2]);
            swap_halves(d[4 * s + 1], d[4 * s + 3]);
            out[2 * nb + s] = __builtin_bit_cast(bf16x8, make_uint4(d[4 * s], d[4 * s + 1], d[4 * s + 2], d[4 * s + 3]));
        }
    }
#pragma unroll
    for (int s = 0; s < kIn / 16; ++s) h[s] = out[s];
}

// One workgroup of 256 lanes (4 waves) proposes for kProposeTile = 128 pixel quads (2x2 pixels
// each): one MLP evaluation per quad, each pixel drawing its own candidates from the quad's
// distribution with its own random stream (q is that distribution, so RIS stays unbiased). A wave
// holds 32 quads in the columns of its products (wide_blocks), so activations and logits stay in
// registers; LDS holds the features and the first layer's weights, then one layer's weights (128
// rows) while the next one's arrive, and last the fp16 softmax numerators [128][K + 4]. 72 KB of LDS
// let two workgroups share a CU, so one's barriers and loads overlap the other's work. 1920x1080,
// K = 256, M = 8: 403 -> 344 us against activations kept in LDS, 208 of them for the draws, which
// wait for the tables.
constexpr int kProposeTile = 128;
template <int KC>
__global__ __launch_bounds__(2 * kProposeTile, 2) void k_propose(const ProposeArgs a) {
    constexpr int T = kProposeTile, kOut = KC < 128 ? KC : 128;  // rows of W4 staged at a time
    __shared__ __align__(16) uint16_t lds[2 * T * kRow];
    __shared__ __align__(16) float bias[3 * kHidden + KC];
    static_assert(T * (KC + 4) <= 2 * T * kRow, "softmax numerators fit the LDS tile");
    static_assert(KC == 64 || KC % 128 == 0, "W4 in whole blocks");
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    // one MLP row per 2x2 pixel quad: the quad's first surface pixel in the order (0,0), (1,0),
    // (0,1), (1,1) stands for it (quad_pixel)
    const uint32_t W = a.f.g.W, H = a.f.g.H, QW = (W + 1) / 2, QH = (H + 1) / 2;
    const uint32_t q0 = blockIdx.x * T;
    // features by the first T lanes while the others stage W1
    for (int e = tid; e < 3 * kHidden + KC; e += 2 * T) bias[e] = a.bias[e];
    if (tid < T) {
        const uint32_t qd = q0 + tid;
        uint16_t *row = lds + tid * kRow;
        if (qd < QW * QH) pixel_features(a.f, quad_pixel(a.f.g, qd % QW, qd / QW), row);
        else for (int k = 0; k < kIn; ++k) row[k] = 0;
    } else {
        for (int e = tid - T; e < kHidden * (kIn / 8); e += T)
            *reinterpret_cast<u32x4 *>(&lds[(T + e / (kIn / 8)) * kRow + e % (kIn / 8) * 8]) =
                *reinterpret_cast<const u32x4 *>(a.wbf + e * 8);
    }
    __syncthreads();
    bf16x8 h[kIn / 16];
#pragma unroll
    for (int s = 0; s < kIn / 16; ++s)
        h[s] = *reinterpret_cast<const bf16x8 *>(&lds[(32 * wave + (lane & 31)) * kRow + 16 * s + 8 * (lane >> 5)]);
    __syncthreads();
    // step L multiplies the weights in buffer (L + 1) & 1 and brings the next ones to the other: the
    // hidden layers, then the output layer 128 clusters at a time
    constexpr int kSteps = 3 + KC / kOut;
    f32x16 acc[KC / 32];
#pragma unroll
    for (int L = 0; L < kSteps; ++L) {
        constexpr int kPer = kHidden * kIn / 8 / (2 * T);  // 16-byte pieces per lane
        u32x4 next[kPer];
        const int rows = L + 1 < 3 ? kHidden : kOut;
        const uint16_t *src = a.wbf + (L + 1 < 3 ? w_off(L + 1) : w_off(3) + static_cast<size_t>(L + 1 - 3) * kOut * kIn);
        if (L + 1 < kSteps)
#pragma unroll
            for (int e = 0; e < kPer; ++e)
                if ((e * 2 * T) / (kIn / 8) < rows) next[e] = *reinterpret_cast<const u32x4 *>(src + (e * 2 * T + tid) * 8);
        const uint16_t *w = lds + ((L + 1) & 1) * T * kRow;
        if (L < 3) {
            wide_hidden(w, bias + b_off(L), h, lane);
        } else {
#pragma unroll
            for (int nb = 0; nb < kOut / 32; nb += 2)
                wide_blocks(w + 32 * nb * kRow, bias + b_off(3) + (L - 3) * kOut + 32 * nb, h, lane,
                            acc[(L - 3) * (kOut / 32) + nb], acc[(L - 3) * (kOut / 32) + nb + 1]);
        }
        if (L + 1 < kSteps)
#pragma unroll
            for (int e = 0; e < kPer; ++e) {
                const int at = e * 2 * T + tid;
                if ((e * 2 * T) / (kIn / 8) < rows)
                    *reinterpret_cast<u32x4 *>(&lds[((L & 1) * T + at / (kIn / 8)) * kRow + at % (kIn / 8) * 8]) = next[e];
            }
        __syncthreads();
    }
    {
        // softmax numerators e = exp(z - rowmax) as fp16 rows of KC + 4 halves; the padding keeps
        // rows 8-byte aligned and spreads these stores and the per-pixel scans below over the banks
        float m = acc[0][0];
#pragma unroll
        for (int nb = 0; nb < KC / 32; ++nb)
#pragma unroll
            for (int i = 0; i < 16; ++i) m = fmaxf(m, acc[nb][i]);
        m = fmaxf(m, __shfl_xor(m, 32));
        __half *row = reinterpret_cast<__half *>(lds) + (32 * wave + (lane & 31)) * (KC + 4) + 4 * (lane >> 5);
#pragma unroll
        for (int nb = 0; nb < KC / 32; ++nb)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const f32x2 e0 = {__expf(acc[nb][4 * g] - m), __expf(acc[nb][4 * g + 1] - m)};
                const f32x2 e1 = {__expf(acc[nb][4 * g + 2] - m), __expf(acc[nb][4 * g + 3] - m)};
                *reinterpret_cast<uint2 *>(row + 32 * nb + 8 * g) =
                    make_uint2(__builtin_bit_cast(uint32_t, __builtin_convertvector(e0, f16x2)),
                               __builtin_bit_cast(uint32_t, __builtin_convertvector(e1, f16x2)));
            }
        __syncthreads();
    }
    // two lanes per quad, each drawing for one row of its 2x2 pixels
    const uint32_t qd = q0 + (tid >> 1);
    if (qd >= QW * QH) return;
    const uint32_t qx = qd % QW, qy = qd / QW;
    // the cluster pmf is e[c] / se with se the sequential sum of the stored fp16 numerators; the
    // inverse-CDF scan below accumulates the same values in the same order, so the sampled
    // distribution and the q written for each candidate agree
    // one 8-byte LDS read yields 4 numerators. Cluster blocks of 32: block sums in registers
    // (sequential inside a block, blocks in order), so a draw picks its block with KC/32
    // compares and scans at most 32 numerators of that block
    const uint2 *row = reinterpret_cast<const uint2 *>(reinterpret_cast<const __half *>(lds) + (tid >> 1) * (KC + 4));
    constexpr int kBlocks = KC / 32;
    // the two lanes of a quad read the same row: each sums every other block (block 2j + lane
    // parity), and the partner's sums come by a lane swap; se then adds the blocks in order
    static_assert(kBlocks % 2 == 0, "block pairs");
    const bool odd = (tid & 1) != 0;
    float bs[kBlocks];
#pragma unroll
    for (int j = 0; j < kBlocks / 2; ++j) {
        const int b = 2 * j + (odd ? 1 : 0);
        float sum = 0.0f;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const float4 f = unpack_h4(row[8 * b + q]);
            sum += f.x;
            sum += f.y;
            sum += f.z;
            sum += f.w;
        }
        const float other = __shfl_xor(sum, 1);
        bs[2 * j] = odd ? other : sum;
        bs[2 * j + 1] = odd ? sum : other;
    }
    float se = 0.0f;
#pragma unroll
    for (int b = 0; b < kBlocks; ++b) se += bs[b];
    const float rse = 1.0f / se;
    // cluster of the draw t in [0, se): the first c whose running sum exceeds t (numerators of
    // zero are never chosen); rounding overflow falls to the last cluster of the block
    auto pick_cluster = [&](float t) {
        int blk = kBlocks - 1;
        float base = 0.0f, cum = 0.0f;
        bool found = false;
#pragma unroll
        for (int b = 0; b < kBlocks; ++b) {
            const float nx = cum + bs[b];
            if (!found && (t < nx || b == kBlocks - 1)) {
                blk = b;
                base = cum;
                found = true;
            }
            cum = nx;
        }
        int c = 32 * blk + 31;
        float run = base;
        bool hit = false;
        // the block's 32 numerators in one batch of LDS reads, then the same sequential sum
        uint2 raw[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) raw[q] = row[8 * blk + q];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const float4 f = unpack_h4(raw[q]);
            const float e4[4] = {f.x, f.y, f.z, f.w};
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                run += e4[k];
                if (!hit && t < run) {
                    c = 32 * blk + 4 * q + k;
                    hit = true;
                }
            }
        }
        return c;
    };
    const int M = static_cast<int>(a.M);
    const FeatArgs &f = a.f;
    const uint32_t py = 2 * qy + static_cast<uint32_t>(tid & 1);
    for (uint32_t px = 2 * qx; px < 2 * qx + 2; ++px) {
    if (px >= W || py >= H) continue;
    const uint32_t p = py * W + px;
    const f3 n = rk::load_normal(f.g, p);
    if (rt::dot(n, n) == 0.0f) continue;  // background: Pass A draws no candidates there
    rt::Pcg rng = rt::pcg_seed(a.seed, p);
    // Candidates in groups of 8, each step's loads issued together (no load waits on another
    // candidate's). Per candidate: one draw for the mixture, one for the cluster (MLP
    // candidates), then two for the alias column.
    for (int j0 = 0; j0 < M; j0 += 8) {
        float r1[8], r2[8], pw[8], ps[8];
        int32_t cl[8], col[8], cnt[8], beg[8], l[8];
        float4 t[8];
#pragma unroll
        for (int jj = 0; jj < 8; ++jj) {
            const int j = j0 + jj;
            cl[jj] = -2;  // beyond M
            if (j < M) {
                const bool src = rt::pcg_float(rng) < a.mix;
                cl[jj] = src ? -1 : pick_cluster(rt::pcg_float(rng) * se);
                r1[jj] = rt::pcg_float(rng);
                r2[jj] = rt::pcg_float(rng);
            }
        }
        // step 1: source candidates read their alias column, MLP candidates their cluster
#pragma unroll
        for (int jj = 0; jj < 8; ++jj) {
            if (cl[jj] == -1) {
                int32_t c = static_cast<int32_t>(static_cast<float>(a.nAlias) * r1[jj]);
                col[jj] = c < a.nAlias - 1 ? c : a.nAlias - 1;
                t[jj] = a.alias[col[jj]];
            } else if (cl[jj] >= 0) {
                cnt[jj] = a.clusterCount[cl[jj]];
                beg[jj] = a.clusterBegin[cl[jj]];
            }
        }
        // step 2: MLP candidates read the fused record of the drawn slot of the cluster's own
        // alias table: the column's and its alias's light, p_within and p_src in 32 bytes
        float4 t2[8];
#pragma unroll
        for (int jj = 0; jj < 8; ++jj) {
            if (cl[jj] >= 0 && cnt[jj] > 0) {
                int32_t c = static_cast<int32_t>(static_cast<float>(cnt[jj]) * r1[jj]);
                col[jj] = c < cnt[jj] - 1 ? c : cnt[jj] - 1;
                const float4 *rec = a.clusterFused + 2 * static_cast<size_t>(beg[jj] + col[jj]);
                t[jj] = rec[0];
                t2[jj] = rec[1];
            }
        }
        // step 3: the light; its probability under the table that drew it comes with the column
        // (oriProb of the column or of its alias, as the alias table stores both), and an MLP
        // candidate's p_src with its record
#pragma unroll
        for (int jj = 0; jj < 8; ++jj) {
            l[jj] = -1;
            if (cl[jj] == -1) {
                const bool keep = t[jj].x > r2[jj];
                l[jj] = keep ? col[jj] : __float_as_int(t[jj].y);
                ps[jj] = keep ? t[jj].z : t[jj].w;
            } else if (cl[jj] >= 0 && cnt[jj] > 0) {
                const bool keep = t[jj].x > r2[jj];
                l[jj] = __float_as_int(keep ? t[jj].y : t[jj].z);
                pw[jj] = keep ? t[jj].w : t2[jj].x;
                ps[jj] = keep ? t2[jj].y : t2[jj].z;
            }
        }
        // step 4: a source candidate's cluster and p_within
#pragma unroll
        for (int jj = 0; jj < 8; ++jj) {
            if (l[jj] >= 0 && cl[jj] == -1) {
                cl[jj] = a.lightCluster[l[jj]];
                pw[jj] = a.lightPWithin[l[jj]];
            }
        }
#pragma unroll
        for (int jj = 0; jj < 8; ++jj) {
            const int j = j0 + jj;
            if (j >= M) continue;
            float q = 0.0f;
            if (l[jj] >= 0) {
                const int c = cl[jj];
                const float pi = __half2float(reinterpret_cast<const __half *>(row)[c]) * rse;
                q = (1.0f - a.mix) * pi * pw[jj] + a.mix * ps[jj];
            }
            a.candLight[static_cast<size_t>(j) * a.npx + p] = l[jj];
            a.candQ[static_cast<size_t>(j) * a.npx + p] = q;
        }
    }
    }  // pixels of this lane
}

// ----------------------------------------------------------- fused inference, many clusters --
// k_propose keeps all K softmax numerators of a quad in LDS, which has room for K <= 256. For
// larger K (a multiple of 128, at most 4096) the output layer streams through LDS in blocks of
// 64 clusters, twice over the same hidden activations:
//   1. the maximum of a quad's logits;
//   2. the numerators e = fp16(exp(z - max)), written to global memory with the running sum after
//      each 32 of them, accumulated as in k_propose: blocks of 32 numerators summed in order,
//      block sums added in cluster order.
// Then each pixel's draws t = u * se select the first block whose running sum exceeds t (the last
// block if rounding leaves none) and the first cluster in it whose running sum from the block's
// start exceeds t (the block's last if none), exactly k_propose's pick_cluster over all K / 32
// blocks; every candidate picks up the numerator of its cluster, whether drawn from the MLP or the
// cluster of a light drawn from the source table. At most kWideCand candidates per pixel.
//
// What bounds it: the matrix cores in the first pass, the exponentials and the 16-bit stores of the
// second. Each wave holds 32 quads in the columns of its products (A = the weights' rows, B = the
// activations): a lane then has 16 logits of one quad, its partner (lane ^ 32) the other 16, the
// maximum stays in the lane, two blocks of 32 are exchanged between the partners' halves and
// summed in order in registers, and a layer's output turns into the next layer's operand by the
// same exchange. LDS holds nothing but two blocks of weights (the next one on its way in registers
// while one is multiplied). Before, activations, logits and draws went through 69.6 KB of LDS, the
// output layer ran a third time to meet the draws, and a lane's draws were searched block by block
// while the other lanes waited. At 1280x720, M = 8: K = 4,096 3.16 -> 1.13 ms, of which the maximum's
// pass takes 0.33 ms, the stores 0.25 and the draws 0.2. Two workgroups on a CU (245 registers, none
// spilled): three are 11% slower, four spill and are slower yet.
//
// The numerators and sums (272 * K bytes a workgroup) live in one of `nSlots` slots. There are at
// most as many workgroups as slots, each taking every gridDim-th tile of quads. A workgroup takes a
// free slot when it starts and gives it back when it ends, so launches on any number of streams
// share them; where they run short, the later workgroups wait for running ones to end.
constexpr int kWideQuads = 128;                 // pixel quads per workgroup: 32 per wave
constexpr int kWideRows = 64;                   // clusters per staged weight block
constexpr int kWideTile = kWideRows * kRow;     // bf16 elements of a staged block
constexpr int kWideResident = 2;                // workgroups on a CU: a wave of each per SIMD
// bytes of a slot: K fp16 numerators and K / 32 running sums for each quad
__host__ __device__ constexpr size_t wide_slot_bytes(int K) {
    return static_cast<size_t>(kWideQuads) * (2 * static_cast<size_t>(K) + static_cast<size_t>(K) / 32 * 4);
}
static_assert(wide_slot_bytes(kMaxClusters) == 272u * kMaxClusters, "the slot size named above");
static_assert(kMaxClusters / kSuper * kWideQuads * 4 <= 2 * kWideTile * 2, "a sum per 128 clusters fits the weight buffers");

__global__ __launch_bounds__(2 * kWideQuads, kWideResident) void k_propose_wide(const ProposeArgs a) {
    __shared__ __align__(16) uint16_t lds[2 * kWideTile];
    __shared__ __align__(16) float bias[2 * kWideRows];
    __shared__ uint32_t slotShared;
    static_assert(kWideQuads * kRow <= 2 * kWideTile && kHidden == 2 * kWideRows, "features and hidden layers fit the weight buffers");
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint32_t W = a.f.g.W, H = a.f.g.H, QW = (W + 1) / 2, QH = (H + 1) / 2;
    const uint16_t *w4 = a.wbf + w_off(3);
    const float *b4 = a.bias + b_off(3);

    if (wave == 0) {  // a slot; an acquire: nothing that an earlier workgroup left of it is read
        const uint32_t chunks = (a.nSlots + 63) / 64;
        uint32_t c = blockIdx.x / 64 % chunks, slot = 0;
        for (bool taken = false; !taken; c = c + 1 < chunks ? c + 1 : 0) {
            const uint32_t i = 64 * c + lane;
            uint32_t busy = 1;
            if (i < a.nSlots) busy = __hip_atomic_load(a.slotBusy + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            uint64_t open = __ballot(busy == 0);
            while (open && !taken) {
                // workgroups start their search at different slots
                const uint64_t later = open >> (blockIdx.x & 63) << (blockIdx.x & 63);
                const int pick = __ffsll(static_cast<unsigned long long>(later ? later : open)) - 1;
                uint32_t was = 1;
                if (lane == pick) was = atomicExch(a.slotBusy + i, 1u);
                taken = __shfl(was, pick) == 0;
                slot = 64 * c + pick;
                open &= ~(1ull << pick);
            }
        }
        if (lane == 0) slotShared = slot;
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    }
    __syncthreads();
    const uint32_t slot = slotShared;
    const uint32_t tiles = (QW * QH + kWideQuads - 1) / kWideQuads;
    for (uint32_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
    const uint32_t q0 = tile * kWideQuads;
    // the quads' features, a lane each, by way of LDS into the B operand of the first layer
    if (tid < kWideQuads) {
        const uint32_t qd = q0 + tid;
        uint16_t *row = lds + tid * kRow;
        if (qd < QW * QH) pixel_features(a.f, quad_pixel(a.f.g, qd % QW, qd / QW), row);
        else for (int k = 0; k < kIn; ++k) row[k] = 0;
    }
    __syncthreads();
    bf16x8 h[kIn / 16];
#pragma unroll
    for (int s = 0; s < kIn / 16; ++s)
        h[s] = *reinterpret_cast<const bf16x8 *>(&lds[(32 * wave + (lane & 31)) * kRow + 16 * s + 8 * (lane >> 5)]);

    // the hidden layers
    for (int L = 0; L < 3; ++L) {
        __syncthreads();
        stage_weights(lds, a.wbf + w_off(L), kHidden);
        if (tid < kHidden) bias[tid] = a.bias[b_off(L) + tid];
        __syncthreads();
        wide_hidden(lds, bias, h, lane);
    }
    __syncthreads();

    // the output layer, 64 clusters at a time: body(step, logits of the first 32, of the second)
    auto sweep = [&](auto &&body) {
        constexpr int kPer = kWideRows * kIn / 8 / (2 * kWideQuads);  // 16-byte pieces per lane
        u32x4 next[kPer];
        float nextBias = 0.0f;
        auto fetch = [&](int step) {
            const u32x4 *src = reinterpret_cast<const u32x4 *>(w4 + static_cast<size_t>(step) * kWideRows * kIn);
#pragma unroll
            for (int e = 0; e < kPer; ++e) next[e] = src[e * 2 * kWideQuads + tid];
            if (tid < kWideRows) nextBias = b4[step * kWideRows + tid];
        };
        auto put = [&](int buf) {
#pragma unroll
            for (int e = 0; e < kPer; ++e) {
                const int at = e * 2 * kWideQuads + tid;
                *reinterpret_cast<u32x4 *>(&lds[buf * kWideTile + at / (kIn / 8) * kRow + at % (kIn / 8) * 8]) = next[e];
            }
            if (tid < kWideRows) bias[buf * kWideRows + tid] = nextBias;
        };
        const int steps = a.K / kWideRows;
        fetch(0);
        put(0);
        __syncthreads();
        for (int step = 0; step < steps; ++step) {
            const int buf = step & 1;
            if (step + 1 < steps) fetch(step + 1);
            const uint16_t *w = lds + buf * kWideTile;
            f32x16 z0, z1;
            wide_blocks(w, bias + buf * kWideRows, h, lane, z0, z1);
            body(step, z0, z1);
            if (step + 1 < steps) put(buf ^ 1);  // read last before the barrier of the step before
            lds_barrier();
        }
    };

    // 1. the maximum
    float zmax = -INFINITY;
    sweep([&](int, const f32x16 &z0, const f32x16 &z1) {
#pragma unroll
        for (int i = 0; i < 16; ++i) zmax = fmaxf(zmax, fmaxf(z0[i], z1[i]));
    });
    zmax = fmaxf(zmax, __shfl_xor(zmax, 32));

    // 2. numerators and running sums. The wave's part of the slot: 16 bytes for each 8
    // clusters of a quad, so placed that the 64 lanes store 1 KB without gaps (a draw then reads its
    // block's 64 bytes in four places, but draws are few: 1.27 -> 1.24 ms, and 1.18 ms with stores
    // that don't stay in the L2; with a block's 64 bytes together those took 2.70 ms); then four
    // running sums per quad and 128 clusters.
    const int quad = lane & 31;
    uint8_t *part = a.slots + static_cast<size_t>(slot) * a.slotBytes + wave * (static_cast<uint32_t>(wide_slot_bytes(a.K)) / 4);
    u32x4 *num = reinterpret_cast<u32x4 *>(part);
    float4 *sums = reinterpret_cast<float4 *>(part + static_cast<size_t>(64) * a.K);
    auto piece = [&](int b, int g) { return static_cast<size_t>(b >> 1) * 256 + 64 * g + 32 * (b & 1) + quad; };
    float se = 0.0f;
    float4 four = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    sweep([&](int step, const f32x16 &z0, const f32x16 &z1) {
        uint32_t p0[8], p1[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const f32x2 e0 = {__expf(z0[2 * i] - zmax), __expf(z0[2 * i + 1] - zmax)};
            const f32x2 e1 = {__expf(z1[2 * i] - zmax), __expf(z1[2 * i + 1] - zmax)};
            p0[i] = __builtin_bit_cast(uint32_t, __builtin_convertvector(e0, f16x2));
            p1[i] = __builtin_bit_cast(uint32_t, __builtin_convertvector(e1, f16x2));
        }
        // lanes 0..31 get all of the first block of their quad, lanes 32..63 all of the second
        float s0 = 0.0f;
        u32x4 *to = num + piece(2 * step, 0) + (lane & 32);
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            swap_halves(p0[2 * g], p1[2 * g]);
            swap_halves(p0[2 * g + 1], p1[2 * g + 1]);
            const u32x4 v = {p0[2 * g], p0[2 * g + 1], p1[2 * g], p1[2 * g + 1]};
            __builtin_nontemporal_store(v, to + 64 * g);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const f16x2 e = __builtin_bit_cast(f16x2, static_cast<uint32_t>(v[k]));
                s0 += static_cast<float>(e[0]);
                s0 += static_cast<float>(e[1]);
            }
        }
        float s1 = s0;
        swap_halves(s0, s1);
        if ((step & 1) == 0) {
            four.x = se + s0;
            four.y = four.x + s1;
            se = four.y;
        } else {
            four.z = se + s0;
            four.w = four.z + s1;
            se = four.w;
            if (lane < 32) sums[(step >> 1) * 32 + quad] = four;
        }
    });
    const float rse = 1.0f / se;
    // the wave's lanes read what its other lanes wrote; the sweep's last barrier freed the weights
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    const int nSuper = a.K / kSuper;
    float *superSum = reinterpret_cast<float *>(lds) + 32 * wave + quad;
    for (int sb = lane >> 5; sb < nSuper; sb += 2) superSum[sb * kWideQuads] = sums[sb * 32 + quad].w;
    __syncthreads();

    // 3. the draws: lane l for row l / 32 of its quad's pixels
    const __half *numh = reinterpret_cast<const __half *>(part);
    auto numerator_at = [&](int c) { return numh[piece(c >> 5, (c >> 3) & 3) * 8 + (c & 7)]; };
    const uint32_t qd = q0 + 32 * wave + quad;
    const int M = static_cast<int>(a.M);
    if (qd < QW * QH) {
        const uint32_t qx = qd % QW, py = 2 * (qd / QW) + static_cast<uint32_t>(lane >> 5);
        for (uint32_t px = 2 * qx; px < 2 * qx + 2; ++px) {
            if (px >= W || py >= H) continue;
            const uint32_t p = py * W + px;
            const f3 n = rk::load_normal(a.f.g, p);
            if (rt::dot(n, n) == 0.0f) continue;  // background: Pass A draws no candidates there
            rt::Pcg rng = rt::pcg_seed(a.seed, p);
            // Each step does all candidates at once, without branches where a load must not wait for
            // another candidate's: one that needs no cluster (a source candidate, one beyond M)
            // searches for t = 0.
            float t[kWideCand], r1[kWideCand], r2[kWideCand];
            int32_t ck[kWideCand], l[kWideCand];  // the cluster; a source candidate's light, else -1
            float pw[kWideCand], ps[kWideCand], ek[kWideCand];
#pragma unroll
            for (int j = 0; j < kWideCand; ++j) {
                t[j] = r1[j] = r2[j] = pw[j] = ps[j] = 0.0f;
                l[j] = -1;
                if (j >= M) continue;
                const bool src = rt::pcg_float(rng) < a.mix;
                if (!src) t[j] = rt::pcg_float(rng) * se;
                r1[j] = rt::pcg_float(rng);
                r2[j] = rt::pcg_float(rng);
                if (src) {
                    const int32_t c = static_cast<int32_t>(static_cast<float>(a.nAlias) * r1[j]);
                    l[j] = c < a.nAlias - 1 ? c : a.nAlias - 1;
                }
            }
            float4 four[kWideCand];
#pragma unroll
            for (int j = 0; j < kWideCand; ++j)
                if (l[j] >= 0) four[j] = a.alias[l[j]];
#pragma unroll
            for (int j = 0; j < kWideCand; ++j) {
                if (l[j] < 0) continue;
                const bool keep = four[j].x > r2[j];
                l[j] = keep ? l[j] : __float_as_int(four[j].y);
                ps[j] = keep ? four[j].z : four[j].w;
            }
#pragma unroll
            for (int j = 0; j < kWideCand; ++j) {
                ck[j] = -1;
                if (l[j] < 0) continue;
                ck[j] = a.lightCluster[l[j]];
                pw[j] = a.lightPWithin[l[j]];
            }
            // the number of running sums, but the last, that t does not lie below: they never fall,
            // so bisection finds it
            int at[kWideCand];
            float base[kWideCand];
#pragma unroll
            for (int j = 0; j < kWideCand; ++j) {
                int sb = 0;
#pragma unroll
                for (int w = kMaxClusters / kSuper / 2; w > 0; w >>= 1) {
                    const int next = sb + w < nSuper ? sb + w : nSuper;  // nSuper: past the last but one
                    const float sum = superSum[(next - 1) * kWideQuads];
                    if (next < nSuper && !(t[j] < sum)) sb = next;
                }
                at[j] = sb;
                base[j] = sb > 0 ? superSum[(sb > 0 ? sb - 1 : 0) * kWideQuads] : 0.0f;
                four[j] = sums[sb * 32 + quad];
            }
#pragma unroll
            for (int j = 0; j < kWideCand; ++j) {
                const bool past0 = !(t[j] < four[j].x), past1 = past0 && !(t[j] < four[j].y), past2 = past1 && !(t[j] < four[j].z);
                base[j] = past2 ? four[j].z : past1 ? four[j].y : past0 ? four[j].x : base[j];
                at[j] = at[j] * (kSuper / 32) + (past0 ? 1 : 0) + (past1 ? 1 : 0) + (past2 ? 1 : 0);
            }
#pragma unroll
            for (int j0 = 0; j0 < kWideCand; j0 += 4) {
                u32x4 raw[4][4];
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int g = 0; g < 4; ++g) raw[j][g] = num[piece(at[j0 + j], g)];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    float run = base[j0 + j];
                    int below = 0;
#pragma unroll
                    for (int g = 0; g < 4; ++g)
#pragma unroll
                        for (int k = 0; k < 4; ++k) {
                            const f16x2 e = __builtin_bit_cast(f16x2, static_cast<uint32_t>(raw[j][g][k]));
                            run += static_cast<float>(e[0]);
                            below += !(t[j0 + j] < run);
                            run += static_cast<float>(e[1]);
                            below += !(t[j0 + j] < run);
                        }
                    if (ck[j0 + j] < 0) ck[j0 + j] = 32 * at[j0 + j] + (below < 31 ? below : 31);
                }
            }
#pragma unroll
            for (int j = 0; j < kWideCand; ++j) ek[j] = __half2float(numerator_at(ck[j]));
            // the light of a cluster's own alias table
            int32_t cnt[kWideCand], beg[kWideCand];
#pragma unroll
            for (int j = 0; j < kWideCand; ++j) {
                cnt[j] = 0;
                if (j >= M || l[j] >= 0) continue;
                cnt[j] = a.clusterCount[ck[j]];
                beg[j] = a.clusterBegin[ck[j]];
            }
#pragma unroll
            for (int j = 0; j < kWideCand; ++j) {
                if (cnt[j] <= 0) continue;
                const int32_t c = static_cast<int32_t>(static_cast<float>(cnt[j]) * r1[j]);
                at[j] = c < cnt[j] - 1 ? c : cnt[j] - 1;
                four[j] = a.clusterAlias[beg[j] + at[j]];
            }
#pragma unroll
            for (int j = 0; j < kWideCand; ++j) {
                if (cnt[j] <= 0) continue;
                const bool keep = four[j].x > r2[j];
                l[j] = a.clusterLights[beg[j] + (keep ? at[j] : __float_as_int(four[j].y))];
                pw[j] = keep ? four[j].z : four[j].w;
            }
#pragma unroll
            for (int j = 0; j < kWideCand; ++j)
                if (cnt[j] > 0) ps[j] = a.alias[l[j]].z;
#pragma unroll
            for (int j = 0; j < kWideCand; ++j) {
                if (j >= M) continue;
                const float q = l[j] >= 0 ? (1.0f - a.mix) * (ek[j] * rse) * pw[j] + a.mix * ps[j] : 0.0f;
                a.candLight[static_cast<size_t>(j) * a.npx + p] = l[j];
                a.candQ[static_cast<size_t>(j) * a.npx + p] = q;
            }
        }
    }
    __syncthreads();  // the next tile's features overwrite the sums
    }  // tiles
    __syncthreads();
    // a release: all writes to the slot are in memory before another workgroup may take it
    if (tid == 0) __hip_atomic_store(a.slotBusy + slot, 0u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
}

}  // namespace rm

// ----------------------------------------------------------------------------- launchers ----
namespace rk {

using rm::kHidden;
using rm::kIn;
using rt::f3;

// Training tensors carved from one scratch allocation.
struct MlpScratch {
    uint16_t *X, *H[3], *dH[3], *dZ;
    float *Z, *gw, *gb, *loss;
    float *part;      // split-K and column-sum partials
    float *lossPart;  // per-workgroup loss sums of k_softmax_ce
    int32_t *target;
    uint32_t *mask, *pixels, *nValid;
};
// split-K of the weight-gradient GEMMs (reduction over the n samples): at most kMaxSplit parts.
// Every layer keeps its own partials (weights: kMaxSplit x rows x kIn, biases: n/64 chunks x rows)
// so that one launch reduces them all after the backward pass.
constexpr int kMaxSplit = 16;
static size_t rows_before(int l) { return static_cast<size_t>(l) * kHidden; }  // output rows of layers < l
static size_t part_floats(int K, uint32_t n) {
    const size_t rows = 3 * static_cast<size_t>(kHidden) + static_cast<size_t>(K);
    return static_cast<size_t>(kMaxSplit) * rows * kIn + static_cast<size_t>(n / 64) * rows;
}
// parts for an M x N (x 64-tiles) gradient over n samples: about 256 workgroups, each K range a
// multiple of 32
static int split_for(int M, int N, int n) {
    const int tiles = (M / 64) * (N / 64);
    int sp = 1;
    while (sp < kMaxSplit && tiles * sp < 256 && (n % (2 * sp * 32)) == 0) sp *= 2;
    return sp;
}
static MlpScratch carve_mlp(void *base, uint32_t n, int K, size_t *bytes = nullptr) {
    Carver c(base);
    const size_t nn = n, kk = static_cast<size_t>(K);
    MlpScratch m;
    m.X = c.take<uint16_t>(2 * nn * kIn);
    for (int l = 0; l < 3; ++l) m.H[l] = c.take<uint16_t>(2 * nn * kHidden);
    for (int l = 0; l < 3; ++l) m.dH[l] = c.take<uint16_t>(2 * nn * kHidden);
    m.dZ = c.take<uint16_t>(2 * nn * kk);
    m.Z = c.take<float>(4 * nn * kk);
    m.target = c.take<int32_t>(4 * nn);
    m.mask = c.take<uint32_t>(4 * nn);
    m.pixels = c.take<uint32_t>(4 * nn);
    m.nValid = c.take<uint32_t>(256);
    m.loss = c.take<float>(256);
    m.gw = c.take<float>(4 * rm::n_weights(K));
    m.gb = c.take<float>(4 * rm::n_bias(K));
    m.part = c.take<float>(4 * part_floats(K, n));
    m.lossPart = c.take<float>(4 * (nn / 4));
    if (bytes) *bytes = c.end();
    return m;
}
size_t mlp_scratch_bytes(uint32_t n, int K) {
    size_t bytes = 0;
    carve_mlp(nullptr, n, K, &bytes);
    return bytes;
}

// forward, keeping the hidden activations for the backward pass
static void mlp_fwd(const restir_mlp &m, const uint16_t *X, uint32_t n, const MlpScratch &t, float *logits,
                    hipStream_t s) {
    const int K = static_cast<int>(m.n_clusters);
    // Groups of clusters: as many as fill the CUs with tiles x groups workgroups, and no more, since each
    // repeats the hidden layers. 128 or 256 clusters a group whatever n was took 16,384 samples 182 us with
    // 4,096 clusters and 288 with 3,968, now 82 and 77; 64 samples 8.3 and 7.2 either way.
    const int tiles = static_cast<int>(n) / rm::kMlpRows, units = (K + 127) / 128;
    const int groups = std::min((256 + tiles - 1) / tiles, units), cols = K < 128 ? K : 128 * ((units + groups - 1) / groups);
    rm::ForwardArgs a{X, m.weights_bf16, m.bias, {t.H[0], t.H[1], t.H[2]}, logits, K, cols};
    RK_LAUNCH("k_mlp_forward", rm::k_mlp_forward, dim3(tiles, (K + cols - 1) / cols), dim3(256), 0, s, a);
}

hipError_t mlp_forward(const restir_mlp &m, const uint16_t *X, uint32_t n, float *logits, void *scratch,
                       hipStream_t s) {
    const MlpScratch t = carve_mlp(scratch, n, static_cast<int>(m.n_clusters));
    mlp_fwd(m, X, n, t, logits, s);
    return hipGetLastError();
}

// mean cross-entropy and its gradient; gw/gb/loss are written (not accumulated)
static void mlp_loss_grad_impl(const restir_mlp &m, const uint16_t *X, const int32_t *target,
                               const uint32_t *mask, uint32_t n, const MlpScratch &t, float *gw, float *gb,
                               float *loss, bool countMask, hipStream_t s) {
    const int K = static_cast<int>(m.n_clusters);
    const int nn = static_cast<int>(n);
    if (countMask)
        RK_LAUNCH("k_count_mask", rm::k_count_mask, dim3(1), dim3(1024), 0, s, mask, n, t.nValid);
    mlp_fwd(m, X, n, t, t.Z, s);
    RK_LAUNCH("k_softmax_ce", rm::k_softmax_ce, dim3((n + 3) / 4), dim3(256), 0, s, t.Z, K, target, mask, nn,
                       t.nValid, t.dZ, t.lossPart);
    const rm::BackwardArgs back{t.dZ, m.weights_bf16, {t.H[0], t.H[1], t.H[2]}, {t.dH[0], t.dH[1], t.dH[2]}, K};
    RK_LAUNCH("k_mlp_backward", rm::k_mlp_backward, dim3(n / rm::kMlpRows), dim3(256), 0, s, back);
    // the gradients' partial sums of all four layers, then each summed in a fixed order, with the
    // loss: the workgroups' sums of k_softmax_ce, in order
    const int chunks = nn / 64;
    float *partB = t.part + static_cast<size_t>(kMaxSplit) * (3 * static_cast<size_t>(kHidden) + K) * kIn;
    rm::GradArgs ga{};
    rm::SumSegments sums{};
    ga.n = nn;
    uint32_t biasGroups = 0;
    int64_t sumCount = 0;
    for (int l = 3; l >= 0; --l) {  // the largest first
        const int j = 3 - l, N = l == 3 ? K : kHidden, sp = split_for(N, kIn, nn);
        float *pw = t.part + static_cast<size_t>(kMaxSplit) * rows_before(l) * kIn;
        float *pb = partB + static_cast<size_t>(chunks) * rows_before(l);
        ga.layer[l] = rm::GradLayer{l == 3 ? t.dZ : t.dH[l], l > 0 ? t.H[l - 1] : X, pw, pb, N, sp, ga.weightGroups, biasGroups};
        ga.weightGroups += static_cast<uint32_t>(kIn / 64 * (N / 64) * sp);
        biasGroups += static_cast<uint32_t>(N / 64 * chunks);
        sums.part[2 * j] = pw;
        sums.nParts[2 * j] = sp;
        sums.count[2 * j] = static_cast<int64_t>(N) * kIn;
        sums.out[2 * j] = gw + rm::w_off(l);
        sums.part[2 * j + 1] = pb;
        sums.nParts[2 * j + 1] = chunks;
        sums.count[2 * j + 1] = N;
        sums.out[2 * j + 1] = gb + rm::b_off(l);
        sumCount += sums.count[2 * j] + N;
    }
    RK_LAUNCH("k_mlp_grads", rm::k_mlp_grads, dim3(ga.weightGroups + biasGroups), dim3(256), 0, s, ga);
    sums.lossPart = t.lossPart;
    sums.loss = loss;
    sums.nLoss = (nn + 3) / 4;
    RK_LAUNCH("k_sum_partials", rm::k_sum_partials, dim3(static_cast<uint32_t>((sumCount + 255) / 256) + 1), dim3(256), 0,
              s, sums);
}

hipError_t mlp_loss_grad(const restir_mlp &m, const uint16_t *X, const int32_t *target, const uint32_t *mask,
                         uint32_t n, float *gw, float *gb, float *loss, void *scratch, hipStream_t s) {
    const MlpScratch t = carve_mlp(scratch, n, static_cast<int>(m.n_clusters));
    mlp_loss_grad_impl(m, X, target, mask, n, t, gw, gb, loss, true, s);
    return hipGetLastError();
}

hipError_t mlp_init(const restir_mlp &m, uint64_t seed, const float *prior, hipStream_t s) {
    const uint32_t K = m.n_clusters;
    const uint32_t nW = static_cast<uint32_t>(rm::n_weights(K)), nB = static_cast<uint32_t>(rm::n_bias(K));
    RK_LAUNCH("k_mlp_init", rm::k_mlp_init, dim3((nW + nB + 255) / 256), dim3(256), 0, s, m.weights, m.weights_bf16,
                       m.bias, m.adam_m, m.adam_v, nW, nB, K, prior, seed);
    return hipGetLastError();
}

hipError_t mlp_features(const GView &g, f3 cam, const float lo[3], const float hi[3], const uint32_t *pixels,
                        uint32_t n, uint16_t *out, hipStream_t s) {
    rm::FeatArgs f{g, cam, {lo[0], lo[1], lo[2]}, {hi[0], hi[1], hi[2]}};
    RK_LAUNCH("k_features", rm::k_features, dim3((n + 255) / 256), dim3(256), 0, s, f, pixels, n, out);
    return hipGetLastError();
}

hipError_t mlp_train(restir_mlp &m, const GView &g, f3 cam, const float lo[3], const float hi[3],
                     const restir_reservoir *res, const int32_t *lightCluster, int32_t nLights,
                     int32_t triBase, uint32_t n, float lr,
                     uint32_t seed, float *lossOut, void *scratch, hipStream_t s) {
    const int K = static_cast<int>(m.n_clusters);
    const MlpScratch t = carve_mlp(scratch, n, K);
    rm::GatherArgs ga{};
    ga.f = rm::FeatArgs{g, cam, {lo[0], lo[1], lo[2]}, {hi[0], hi[1], hi[2]}};
    ga.res = res;
    ga.lightCluster = lightCluster;
    ga.nLights = nLights;
    ga.triBase = triBase;
    ga.npx = g.W * g.H;
    ga.n = n;
    ga.seed = seed;
    ga.X = t.X;
    ga.target = t.target;
    ga.mask = t.mask;
    ga.nValid = t.nValid;
    ga.pixels = t.pixels;
    RK_LAUNCH("k_zero_u32", k_zero_u32, dim3(1), dim3(64), 0, s, t.nValid, 1u);
    RK_LAUNCH("k_train_gather", rm::k_train_gather, dim3((n + 255) / 256), dim3(256), 0, s, ga);
    mlp_loss_grad_impl(m, t.X, t.target, t.mask, n, t, t.gw, t.gb, t.loss, false, s);
    const hipError_t ea = mlp_adam(m, t.gw, t.gb, t.nValid, lr, s);
    if (ea != hipSuccess) return ea;
    if (lossOut) RK_LAUNCH("k_copy_f32", rm::k_copy_f32, dim3(1), dim3(1), 0, s, t.loss, lossOut);
    return hipGetLastError();
}

// One Adam step (beta 0.9 / 0.999, eps 1e-8) from the gradients gw, gb: advances the step count
// (host, and the device copy when set) and updates the fp32 master weights, the moments and the
// bf16 copy. nValid (device, may be null): the step is skipped when it reads 0.
hipError_t mlp_adam(restir_mlp &m, const float *gw, const float *gb, const uint32_t *nValid, float lr,
                    hipStream_t s) {
    const int K = static_cast<int>(m.n_clusters);
    m.adam_step += 1;
    const double b1 = 0.9, b2 = 0.999;
    rm::AdamArgs a{};
    a.w = m.weights;
    a.b = m.bias;
    a.wbf = m.weights_bf16;
    a.gw = gw;
    a.gb = gb;
    a.m = m.adam_m;
    a.v = m.adam_v;
    a.nW = static_cast<uint32_t>(rm::n_weights(K));
    a.nB = static_cast<uint32_t>(rm::n_bias(K));
    a.lr = lr;
    a.b1 = static_cast<float>(b1);
    a.b2 = static_cast<float>(b2);
    a.eps = 1e-8f;
    a.b1d = b1;
    a.b2d = b2;
    a.stepHost = m.adam_step;
    a.stepDev = m.adam_step_device;
    if (m.adam_step_device)
        RK_LAUNCH("k_adam_count", rm::k_adam_count, dim3(1), dim3(64), 0, s, m.adam_step_device);
    RK_LAUNCH("k_adam_guarded", rm::k_adam_guarded, dim3((a.nW + a.nB + 255) / 256), dim3(256), 0, s, a, nValid);
    return hipGetLastError();
}

size_t wide_slot_bytes(uint32_t K) { return rm::wide_slot_bytes(static_cast<int>(K)); }
uint32_t wide_slots(uint32_t cus) { return rm::kWideResident * cus; }

hipError_t mlp_propose(const restir_mlp &m, const GView &g, f3 cam, const float lo[3], const float hi[3],
                       const SceneView &sc, const int32_t *lightCluster, const float *lightPWithin,
                       const int32_t *clusterBegin, const int32_t *clusterCount, const int32_t *clusterLights,
                       const restir_alias_table_column *clusterAlias, const float4 *clusterFused, uint32_t M,
                       float mix, uint32_t seed, const WideSlots &slots, int32_t *candLight, float *candQ,
                       hipStream_t s) {
    rm::ProposeArgs a{};
    a.f = rm::FeatArgs{g, cam, {lo[0], lo[1], lo[2]}, {hi[0], hi[1], hi[2]}};
    a.wbf = m.weights_bf16;
    a.bias = m.bias;
    a.K = static_cast<int>(m.n_clusters);
    a.npx = g.W * g.H;
    a.M = M;
    a.seed = seed;
    a.mix = mix;
    a.alias = sc.alias;
    a.nAlias = sc.nAlias;
    a.lightCluster = lightCluster;
    a.lightPWithin = lightPWithin;
    a.clusterBegin = clusterBegin;
    a.clusterCount = clusterCount;
    a.clusterLights = clusterLights;
    a.clusterAlias = reinterpret_cast<const float4 *>(clusterAlias);
    a.clusterFused = clusterFused;
    a.candLight = candLight;
    a.candQ = candQ;
    const uint32_t quads = ((g.W + 1) / 2) * ((g.H + 1) / 2);
    const dim3 grid((quads + rm::kProposeTile - 1) / rm::kProposeTile), block(2 * rm::kProposeTile);
    const uint32_t tilesW = (quads + rm::kWideQuads - 1) / rm::kWideQuads;
    const dim3 gridW(tilesW < slots.n ? tilesW : slots.n), blockW(2 * rm::kWideQuads);
    a.slots = static_cast<uint8_t *>(slots.base);
    a.slotBusy = slots.busy;
    a.nSlots = slots.n;
    a.slotBytes = static_cast<uint32_t>(slots.each);
    switch (a.K) {
        case 64: RK_LAUNCH("k_propose", (rm::k_propose<64>), grid, block, 0, s, a); break;
        case 128: RK_LAUNCH("k_propose", (rm::k_propose<128>), grid, block, 0, s, a); break;
        case 256: RK_LAUNCH("k_propose", (rm::k_propose<256>), grid, block, 0, s, a); break;
        default: RK_LAUNCH("k_propose_wide", rm::k_propose_wide, gridW, blockW, 0, s, a); break;
    }
    return hipGetLastError();
}

}  // namespace rk
