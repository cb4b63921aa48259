"""Pass A over light records (each alias column next to the point lights it can draw) against Pass A
over the tables themselves, which the inline schedule reads: the same reservoirs bit for bit, for
point lights alone, for a union with triangle lights, around the rule's limits, after the tables
changed in place, and from a captured graph that outlives its records."""
import pytest

from restir_amd import abi, scenes
from restir_amd.pipeline import Renderer

pytestmark = pytest.mark.gpu

INLINE = abi.Launch(0, 0, abi.SCHEDULE_INLINE)


class _PassA:
    def __init__(self, torch, lights, lamps, w=521, h=301, M=32, ctx=None, flags=abi.VISIBILITY_REUSE_FLAG):
        self.sc = scenes.terrain(11, grid=24, n_boxes=20, n_point_lights=lights, n_tri_lights=lamps, extent=16.0)
        self.r = r = Renderer(self.sc, w, h, M=M, ctx=ctx)
        r.begin_frame(self.sc.camera)
        self.u = abi.make_uniforms(w, h, 1, self.sc.camera["position"], M=M, flags=flags)
        self.g = r.gstruct(r.cur)
        self.out = torch.zeros(16 * w * h, dtype=torch.int32, device="cuda")

    def run(self, launch=None, stream=None):
        self.r.ctx.initial_temporal(self.u, self.g, self.g, None, self.out, launch, stream)

    def get(self, torch, launch=None):
        self.out.zero_()
        self.run(launch)
        torch.cuda.synchronize()
        return self.out.clone()

    def used(self, ctx):
        ctx.profile_read()
        ctx.profile_enable(True)
        self.run()
        rows = ctx.profile_read()
        ctx.profile_enable(False)
        return "k_light_records" in rows


@pytest.mark.parametrize("lights,lamps,records", [(2047, 0, False), (2048, 0, True), (3000, 1000, True),
                                                  (3000, 1001, False), (0, 3000, False), (5003, 0, True)])
def test_same_reservoirs(lights, lamps, records):
    import torch
    p = _PassA(torch, lights, lamps)
    assert p.used(p.r.ctx) == records
    assert torch.equal(p.get(torch), p.get(torch, INLINE))
    # lights that changed in place
    if lights:
        pts = p.r.dev.d_points.view(torch.float32)
        pts[4:] = pts[4:].roll(8)  # the header stays; every light takes its neighbour's place
        a = p.get(torch)
        assert torch.equal(a, p.get(torch, INLINE))


def test_graph_outlives_its_records():
    import torch
    p = _PassA(torch, 2500, 0, flags=0)
    ref = p.get(torch, INLINE)
    assert torch.equal(p.get(torch), ref)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        p.run(stream=s)
    other = _PassA(torch, 6000, 0, ctx=p.r.ctx, flags=0)  # larger records on the same context
    for _ in range(3):
        assert torch.equal(other.get(torch), other.get(torch, INLINE))
        p.out.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(p.out, ref)
