"""The multi-view passes A and C: queued view after view, or one persistent launch with the rays
traced per pixel (inline schedule; or under capture while the scratch is too small). Every route gives
the same reservoirs, and a captured graph stays valid when a later call grows the scratch."""
import ctypes as C

import pytest

from restir_amd import abi, scenes
from restir_amd.pipeline import BatchRenderer

pytestmark = pytest.mark.gpu

K, PASSES = 3, 2


def _views(sizes):
    a = scenes.cornell_box(1)
    b = scenes.terrain(11, grid=48, n_boxes=60, n_point_lights=2000, extent=16.0)
    return [((a, b)[i % 2], w, h) for i, (w, h) in enumerate(sizes)]


class _Passes:
    """Passes A and C of one frame over a BatchRenderer's views through the multi-view entry points."""

    def __init__(self, torch, sizes):
        views = _views(sizes)
        self.b = b = BatchRenderer(views, k=K, M=8)
        b.cur = 0
        self.us, self.gs, self.bufs = [], [], []
        for v, (sc, w, h) in zip(b.views, views):
            cam = sc.camera
            v["ctx"].primary_gbuffer(cam, v["dev"].d_tri_material, v["dev"].d_materials, len(sc.materials),
                                     v["gbuf"][0], w, h)
            self.us.append(abi.make_uniforms(w, h, 1, cam["position"], M=8, flags=abi.VISIBILITY_REUSE_FLAG))
            self.gs.append(b._g(v, 0))
            self.bufs.append([torch.zeros(16 * w * h, dtype=torch.int32, device="cuda") for _ in range(2)])

    def _rec(self, src, dst):
        return [abi.View(v["ctx"].h.value, C.pointer(u), C.pointer(g), C.pointer(g),
                         abi.as_ptr(buf[src]) if src is not None else None, abi.as_ptr(buf[dst]), None, 0)
                for v, u, g, buf in zip(self.b.views, self.us, self.gs, self.bufs)]

    def run(self, launch=None, stream=None):
        self.b.ctx.initial_temporal_views(self._rec(None, 0), launch, stream)
        for j in range(PASSES):
            self.b.ctx.unbiased_views(self._rec(j % 2, 1 - j % 2), K, j, launch, stream)

    def out(self, torch):
        torch.cuda.synchronize()
        return [buf[PASSES % 2].clone() for buf in self.bufs]


@pytest.mark.parametrize("sizes", [[(64, 48)], [(33, 70), (80, 45), (1, 1), (17, 16)]])
def test_routes_agree_and_graphs_survive_growth(sizes):
    import torch
    p = _Passes(torch, sizes)
    inline = abi.Launch(0, 0, abi.SCHEDULE_INLINE)
    p.run(inline)  # no queue scratch yet
    ref = p.out(torch)
    graphs = []
    for step in ("scratch too small", "queued"):
        for buf in p.bufs:
            for t in buf:
                t.zero_()
        s = torch.cuda.Stream()
        s.wait_stream(torch.cuda.current_stream())
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            p.run(stream=s)
        graphs.append(g)
        for rep in range(3):
            g.replay()
            assert all(torch.equal(a, b) for a, b in zip(p.out(torch), ref)), (step, rep)
            p.run(inline)
        p.run()  # eager: grows the scratch, and takes the queued route
        assert all(torch.equal(a, b) for a, b in zip(p.out(torch), ref)), step
    # a larger call on the same context replaces the scratch that the second graph uses
    big = _Passes(torch, [(320, 200)])
    big.b.ctx = p.b.ctx
    big.run()
    torch.cuda.synchronize()
    for g in graphs:
        for buf in p.bufs:
            for t in buf:
                t.zero_()
        g.replay()
        assert all(torch.equal(a, b) for a, b in zip(p.out(torch), ref))


def test_single_view_graph_survives_growth():
    """A graph of single-view passes A and C keeps its ray queues when later eager calls on the same
    context need larger ones: a multi-view call with a larger view, then a larger single view."""
    import torch

    def single(ctx, p, stream=None):
        (u,), (g,), (bufs,) = p.us, p.gs, p.bufs
        ctx.initial_temporal(u, g, g, None, bufs[0], None, stream)
        for j in range(PASSES):
            ctx.unbiased(u, K, j, g, bufs[j % 2], bufs[1 - j % 2], None, stream)

    p, large, larger = (_Passes(torch, [size]) for size in ((200, 120), (320, 200), (900, 700)))
    ctx = p.b.views[0]["ctx"]  # holds the room, the scene of all three
    single(ctx, p)  # eager: sizes the queues
    ref = p.out(torch)[0]
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        single(ctx, p, s)
    large.b.ctx = ctx
    for step in (large.run, lambda: single(ctx, larger)):
        step()
        for _ in range(3):
            for t in p.bufs[0]:
                t.zero_()
            graph.replay()
            assert torch.equal(p.out(torch)[0], ref)
            step()


def test_graph_of_views_keeps_its_table():
    """The per-view records of a captured persistent launch stay its own when a call over more views
    needs a larger table."""
    import torch
    p, more = _Passes(torch, [(64, 48), (33, 21)]), _Passes(torch, [(16 + i, 9) for i in range(12)])
    inline = abi.Launch(0, 0, abi.SCHEDULE_INLINE)
    p.run(inline)
    ref = p.out(torch)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        p.run(inline, s)
    more.run(inline)
    want = more.out(torch)
    more.b.ctx = p.b.ctx
    for _ in range(3):
        more.run(inline)
        assert all(torch.equal(a, b) for a, b in zip(more.out(torch), want))
        for buf in p.bufs:
            for t in buf:
                t.zero_()
        graph.replay()
        assert all(torch.equal(a, b) for a, b in zip(p.out(torch), ref))
