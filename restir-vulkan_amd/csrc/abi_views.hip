// abi_views.hip — batched-view entry points (restir_*_views): per-view validation with the same
// rules as the single-view entry points, then one launch per pass over all views, or, for the passes that
// trace shadow rays, the queued schedule view after view where that is faster (Route).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <vector>

#include "ctx.h"
#include "kernels.h"

using namespace rki;

namespace {

struct Span {
    const void *p;
    size_t bytes;
};

// every output span against every other span (outputs and inputs of all views)
int check_disjoint(restir_ctx *ctx, const std::vector<Span> &outs, const std::vector<Span> &ins,
                   const char *name) {
    for (size_t i = 0; i < outs.size(); ++i) {
        for (size_t j = 0; j < outs.size(); ++j)
            if (i != j && overlaps(outs[i].p, outs[i].bytes, outs[j].p, outs[j].bytes))
                return fail(ctx, RESTIR_E_ALIASING, "%s: outputs of two views overlap", name);
        for (const Span &in : ins)
            if (overlaps(outs[i].p, outs[i].bytes, in.p, in.bytes))
                return fail(ctx, RESTIR_E_ALIASING, "%s: an output overlaps an input", name);
    }
    return RESTIR_OK;
}

int check_views(restir_ctx *ctx, const restir_view *views, uint32_t n, const char *name) {
    if (!ctx) return RESTIR_E_INVALID_ARGUMENT;
    if (n == 0) return RESTIR_OK;
    if (!views) return fail(ctx, RESTIR_E_INVALID_ARGUMENT, "%s: views is NULL", name);
    if (n > RESTIR_MAX_VIEWS) return fail(ctx, RESTIR_E_INVALID_ARGUMENT, "%s: %u views > %d", name, n, RESTIR_MAX_VIEWS);
    for (uint32_t v = 0; v < n; ++v) {
        const restir_ctx *sc = views[v].scene;
        if (!sc) return fail(ctx, RESTIR_E_INVALID_ARGUMENT, "%s: view %u has no scene context", name, v);
        if (sc->device != ctx->device)
            return fail(ctx, RESTIR_E_INVALID_ARGUMENT, "%s: view %u's scene is on device %d, not %d", name, v,
                        sc->device, ctx->device);
        if (!sc->lightsSet) return fail(ctx, RESTIR_E_NOT_READY, "%s: view %u: lights not set", name, v);
    }
    return RESTIR_OK;
}

int prepare(restir_ctx *ctx, uint32_t n, hipStream_t s) {
    if (int r = use_device(ctx)) return r;
    return ensure_kept(ctx, &ctx->viewTable, &ctx->viewTableBytes, &ctx->viewsInGraph, rk::views_table_bytes(n), s);
}

uint32_t *view_counter(restir_ctx *ctx) { return ctx->counters + 8; }

// The two routes of a pass that traces rays: queued, view after view, or inline, one persistent launch
// over all views with the rays traced in the pixels' lanes. Queued, each view takes a few launches and
// waits for its longest ray; inline, one launch does, but a wave waits for the longest ray of its pixels and
// cannot gather triangle tests. All of it grows with the depth of the trees, L = log2(triangles). In us
//   Pass A:  queued 5.6 L a view more; inline  8.2 L once, 18 (L - 10) - 1.6 (M - 8) a million pixels more
//   Pass C:  queued 5.6 L a view more; inline  4 (k + 2) L once, 14 (k + 1) (L - 7) a million pixels more
// (negative over small trees and with many candidates, where inline costs less per pixel too). Fitted to
// 560 pairs of times for each pass: 1 to 12 views of 64 to 1,080 lines, 34 to 593,000 triangles, M 8 and 32,
// k 3 and 5. What this picks takes at most 1.3 times what the other route takes (4 pairs above 1.15);
// always queued takes up to 8.1 times, always inline up to 6.5. Inline against queued, 138,000 triangles:
//   12 views of      120 lines        240 lines        720 lines       1 view of 120 lines
//   Pass A, M = 32   0.41, 1.62 ms    0.83, 1.85 ms    5.59, 5.86 ms   0.18, 0.13 ms
//   Pass C, k = 5    1.19, 1.33       2.62, 2.08       17.3, 6.58      0.56, 0.11
// Without rays one view takes about as long either way, and more are better inline (12 views of 240 lines:
// Pass A 0.34, 0.75 ms, Pass C 0.18, 0.26).
class Route {
  public:
    // perMpx: what inline costs more per million pixels of a view, from its L
    template <class F>
    void add(const restir_view &w, F perMpx) {
        const restir_uniforms &u = *w.uniforms;
        const double L = std::log2(std::max(2u, w.scene->treeTris));
        ++views_;
        rays_ = rays_ || (u.flags & RESTIR_VISIBILITY_REUSE_FLAG);
        deepest_ = std::max(deepest_, L);
        gain_ += 5.6 * L - 1e-6 * u.screenSize[0] * u.screenSize[1] * perMpx(L);
    }
    // once: what the inline launch costs more, per L
    bool queued(double once) const { return rays_ ? gain_ <= once * deepest_ : views_ == 1; }

  private:
    double gain_ = 0.0, deepest_ = 0.0;
    uint32_t views_ = 0;
    bool rays_ = false;
};

// Whether the views run queued, with this context's scratch (`bytes`: the largest view's) and work
// counters: where that is the faster route (`pays`), unless the caller asks for the inline schedule or
// the scratch is too small and cannot grow (the stream is being captured, or the device is out of memory).
bool queued_views(restir_ctx *ctx, const restir_launch *launch, bool pays, size_t bytes, hipStream_t s) {
    if (!pays || (launch && launch->schedule == RESTIR_SCHEDULE_INLINE)) return false;
    // what the scratch held of a single-view Pass C will be overwritten
    ctx->queuedNpx = 0;
    ctx->surfValid = false;
    if (bytes > ctx->scratchBytes && in_capture(s)) return false;
    if (ensure_scratch(ctx, bytes, s) == RESTIR_OK) return true;
    (void)hipGetLastError();
    ctx->error.clear();
    return false;
}

// The scene of a view as this context's launches see it: a scene may be in use by launches of its
// own context, so the tracer takes its chunks through this context's counters.
rk::SceneView own_counters(const restir_ctx *ctx, rk::SceneView sc) {
    sc.traceHeads = ctx->scene.traceHeads;
    return sc;
}

}  // namespace

extern "C" {

int restir_initial_temporal_views(restir_ctx *ctx, const restir_view *views, uint32_t n,
                                  const restir_launch *launch, void *stream) {
    if (int r = check_views(ctx, views, n, "initial_temporal_views")) return r;
    if (n == 0) return RESTIR_OK;
    int tile;
    if (int r = pick_tile(ctx, launch, &tile)) return r;
    std::vector<rk::ViewA> rec(n);
    std::vector<Span> outs, ins;
    size_t queueBytes = 0;
    Route route;
    int stack = 24;  // the smallest compiled stack; raised to the deepest scene's
    for (uint32_t v = 0; v < n; ++v) {
        const restir_view &w = views[v];
        const restir_uniforms *u = w.uniforms;
        if (int r = check_frame(ctx, u, "initial_temporal_views")) return r;
        const bool vis = (u->flags & RESTIR_VISIBILITY_REUSE_FLAG) != 0;
        const bool temporal = (u->flags & RESTIR_TEMPORAL_REUSE_FLAG) != 0;
        if (vis && !w.scene->bvhSet) return fail(ctx, RESTIR_E_NOT_READY, "initial_temporal_views: view %u: BVH not set", v);
        const uint32_t W = u->screenSize[0], H = u->screenSize[1];
        if (int r = check_gbuffer(ctx, w.cur, W, H, false, "initial_temporal_views cur")) return r;
        if (!w.out) return fail(ctx, RESTIR_E_INVALID_ARGUMENT, "initial_temporal_views: view %u output is NULL", v);
        const size_t bytes = sizeof(restir_reservoir) * W * H;
        if (temporal) {
            if (int r = check_gbuffer(ctx, w.prev, W, H, false, "initial_temporal_views prev")) return r;
            if (!w.in) return fail(ctx, RESTIR_E_INVALID_ARGUMENT, "initial_temporal_views: view %u previous reservoirs are NULL", v);
            ins.push_back({w.in, bytes});
        }
        outs.push_back({w.out, bytes});
        if (w.scene->stack > stack) stack = w.scene->stack;
        queueBytes = std::max(queueBytes, rk::pass_a_queue_bytes(W * H));
        route.add(w, [u](double L) { return 18.0 * (L - 10.0) - 1.6 * (static_cast<double>(u->initialLightSampleCount) - 8.0); });
        rec[v] = rk::ViewA{*u, w.scene->scene, view_of(w.cur), view_of(temporal ? w.prev : nullptr), w.in, w.out};
    }
    if (int r = check_disjoint(ctx, outs, ins, "initial_temporal_views")) return r;
    if (int r = use_device(ctx)) return r;
    const hipStream_t s = static_cast<hipStream_t>(stream);
    if (queued_views(ctx, launch, route.queued(8.2), queueBytes, s)) {
        for (uint32_t v = 0; v < n; ++v) {
            const rk::ViewA &w = rec[v];
            const int st = views[v].scene->stack;
            const hipError_t e = rk::launch_pass_a(tile, st, w.u, own_counters(ctx, w.sc), w.cur, w.prev, w.prevRes,
                                                   w.out, nullptr, nullptr, ctx->scratch,
                                                   persistent_blocks(ctx->cus, st), s,
                                                   light_records(ctx, w.sc, w.u, s));
            if (e != hipSuccess) return hip_fail(ctx, e, "initial_temporal_views launch");
        }
        return RESTIR_OK;
    }
    if (int r = prepare(ctx, n, s)) return r;
    const hipError_t e = rk::launch_pass_a_views(tile, stack, rec.data(), n, ctx->viewTable, view_counter(ctx),
                                                 resident_blocks(ctx->cus, static_cast<uint32_t>(stack) * 1024u), s);
    return e == hipSuccess ? RESTIR_OK : hip_fail(ctx, e, "initial_temporal_views launch");
}

int restir_spatial_views(restir_ctx *ctx, const restir_view *views, uint32_t n, int iter,
                         const restir_launch *launch, void *stream) {
    if (int r = check_views(ctx, views, n, "spatial_views")) return r;
    if (n == 0) return RESTIR_OK;
    int tile;
    if (int r = pick_tile(ctx, launch, &tile)) return r;
    std::vector<rk::ViewB> rec(n);
    std::vector<Span> outs, ins;
    for (uint32_t v = 0; v < n; ++v) {
        const restir_view &w = views[v];
        const restir_uniforms *u = w.uniforms;
        if (int r = check_frame(ctx, u, "spatial_views")) return r;
        const uint32_t W = u->screenSize[0], H = u->screenSize[1];
        if (int r = check_gbuffer(ctx, w.cur, W, H, true, "spatial_views")) return r;
        if (!w.in || !w.out) return fail(ctx, RESTIR_E_INVALID_ARGUMENT, "spatial_views: view %u reservoir buffer is NULL", v);
        const size_t bytes = sizeof(restir_reservoir) * W * H;
        ins.push_back({w.in, bytes});
        outs.push_back({w.out, bytes});
        rec[v] = rk::ViewB{*u, view_of(w.cur), w.in, w.out, rt::cos_degrees(u->spatialNormalThreshold)};
    }
    if (int r = check_disjoint(ctx, outs, ins, "spatial_views")) return r;
    if (int r = prepare(ctx, n, static_cast<hipStream_t>(stream))) return r;
    const hipError_t e = rk::launch_pass_b_views(tile, rec.data(), n, iter, ctx->viewTable, view_counter(ctx),
                                                 ctx->persistentBlocks, static_cast<hipStream_t>(stream));
    return e == hipSuccess ? RESTIR_OK : hip_fail(ctx, e, "spatial_views launch");
}

int restir_unbiased_views(restir_ctx *ctx, const restir_view *views, uint32_t n, int k, int iter,
                          const restir_launch *launch, void *stream) {
    if (int r = check_views(ctx, views, n, "unbiased_views")) return r;
    if (n == 0) return RESTIR_OK;
    if (k < 1 || k > 16) return fail(ctx, RESTIR_E_INVALID_ARGUMENT, "unbiased_views: k=%d outside [1,16]", k);
    int tile;
    if (int r = pick_tile(ctx, launch, &tile)) return r;
    std::vector<rk::ViewC> rec(n);
    std::vector<Span> outs, ins;
    size_t queueBytes = 0;
    Route route;
    bool queueable = true;
    int stack = 24;  // the smallest compiled stack; raised to the deepest scene's
    for (uint32_t v = 0; v < n; ++v) {
        const restir_view &w = views[v];
        const restir_uniforms *u = w.uniforms;
        if (int r = check_frame(ctx, u, "unbiased_views")) return r;
        const bool vis = (u->flags & RESTIR_VISIBILITY_REUSE_FLAG) != 0;
        if (vis && !w.scene->bvhSet) return fail(ctx, RESTIR_E_NOT_READY, "unbiased_views: view %u: BVH not set", v);
        const uint32_t W = u->screenSize[0], H = u->screenSize[1];
        if (int r = check_gbuffer(ctx, w.cur, W, H, false, "unbiased_views")) return r;
        if (!w.in || !w.out) return fail(ctx, RESTIR_E_INVALID_ARGUMENT, "unbiased_views: view %u reservoir buffer is NULL", v);
        const size_t bytes = sizeof(restir_reservoir) * W * H;
        ins.push_back({w.in, bytes});
        outs.push_back({w.out, bytes});
        if (w.scene->stack > stack) stack = w.scene->stack;
        queueBytes = std::max(queueBytes, rk::pass_c_queue_bytes(W * H, k));
        route.add(w, [k](double L) { return 14.0 * (k + 1) * (L - 7.0); });
        // a queued neighbour ray carries its pixel in 27 bits of its tag
        queueable = queueable && static_cast<uint64_t>(W) * H < (1ull << 27);
        rec[v] = rk::ViewC{*u, w.scene->scene, view_of(w.cur), w.in, w.out};
    }
    if (int r = check_disjoint(ctx, outs, ins, "unbiased_views")) return r;
    if (int r = use_device(ctx)) return r;
    const hipStream_t s = static_cast<hipStream_t>(stream);
    if (queued_views(ctx, launch, queueable && route.queued(4.0 * (k + 2)), queueBytes, s)) {
        for (uint32_t v = 0; v < n; ++v) {
            rk::ViewC &w = rec[v];
            w.u.flags &= ~RESTIR_INPUT_VISIBLE_FLAG;  // these calls make no use of the promise
            const int st = views[v].scene->stack;
            const hipError_t e = rk::launch_pass_c(tile, st, w.u, k, iter, own_counters(ctx, w.sc), w.g, w.in, w.out,
                                                   ctx->scratch, persistent_blocks(ctx->cus, st), s);
            if (e != hipSuccess) return hip_fail(ctx, e, "unbiased_views launch");
        }
        return RESTIR_OK;
    }
    if (int r = prepare(ctx, n, s)) return r;
    const hipError_t e = rk::launch_pass_c_views(tile, stack, rec.data(), n, k, iter, ctx->viewTable,
                                                 view_counter(ctx), resident_blocks(ctx->cus, static_cast<uint32_t>(stack) * 1024u),
                                                 s);
    return e == hipSuccess ? RESTIR_OK : hip_fail(ctx, e, "unbiased_views launch");
}

int restir_shade_views(restir_ctx *ctx, const restir_view *views, uint32_t n, float gamma,
                       void *stream) {
    if (int r = check_views(ctx, views, n, "shade_views")) return r;
    if (n == 0) return RESTIR_OK;
    if (!(gamma > 0.0f)) return fail(ctx, RESTIR_E_INVALID_ARGUMENT, "shade_views: gamma must be > 0");
    std::vector<rk::ViewShade> rec(n);
    std::vector<Span> outs, ins;
    for (uint32_t v = 0; v < n; ++v) {
        const restir_view &w = views[v];
        const restir_uniforms *u = w.uniforms;
        if (int r = check_frame(ctx, u, "shade_views")) return r;
        const uint32_t W = u->screenSize[0], H = u->screenSize[1];
        if (int r = check_gbuffer(ctx, w.cur, W, H, false, "shade_views")) return r;
        if (!w.in || !w.rgb) return fail(ctx, RESTIR_E_INVALID_ARGUMENT, "shade_views: view %u needs in and rgb", v);
        if (w.rgb_stride < static_cast<uint64_t>(W) * H)
            return fail(ctx, RESTIR_E_SIZE_MISMATCH, "shade_views: view %u rgb plane stride too small", v);
        ins.push_back({w.in, sizeof(restir_reservoir) * W * H});
        outs.push_back({w.rgb, sizeof(float) * (2 * w.rgb_stride + static_cast<uint64_t>(W) * H)});
        rec[v] = rk::ViewShade{w.scene->scene, rt::f3{u->cameraPos[0], u->cameraPos[1], u->cameraPos[2]},
                               view_of(w.cur), w.in, w.rgb, w.rgb_stride};
    }
    if (int r = check_disjoint(ctx, outs, ins, "shade_views")) return r;
    if (int r = prepare(ctx, n, static_cast<hipStream_t>(stream))) return r;
    const hipError_t e = rk::launch_shade_views(rec.data(), n, gamma, ctx->viewTable, view_counter(ctx),
                                                ctx->persistentBlocks, static_cast<hipStream_t>(stream));
    return e == hipSuccess ? RESTIR_OK : hip_fail(ctx, e, "shade_views launch");
}

}  // extern "C"
