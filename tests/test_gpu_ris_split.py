"""Pass A with four lanes per pixel (small images, point lights alone, 16 candidates or more) against
the inline schedule, which draws a pixel's candidates one after another: the same reservoirs bit for
bit, and the same random stream afterwards (the second frame's temporal reuse draws from it), for
counts of candidates of every remainder, at the rule's limits and beyond them."""
import pytest

from restir_amd import abi, scenes
from restir_amd.pipeline import Renderer

pytestmark = pytest.mark.gpu

INLINE = abi.Launch(0, 0, abi.SCHEDULE_INLINE)


@pytest.mark.parametrize("w,h,M,lights,lamps,standard,split", [
    (1, 1, 16, 1, 0, False, True), (65, 47, 17, 64, 0, True, True), (33, 90, 18, 500, 0, False, True),
    (256, 256, 19, 1000, 0, False, True), (384, 256, 32, 50, 0, True, True), (385, 256, 32, 50, 0, False, False),
    (64, 64, 15, 50, 0, False, False), (64, 64, 32, 50, 20, False, False), (64, 64, 32, 0, 20, False, False)])
def test_same_reservoirs(w, h, M, lights, lamps, standard, split):
    import torch
    sc = scenes.terrain(11, grid=24, n_boxes=20, n_point_lights=lights, n_tri_lights=lamps, extent=16.0)
    r = Renderer(sc, w, h, M=M)
    r.begin_frame(sc.camera)
    g = r.gstruct(r.cur)
    flags = abi.VISIBILITY_REUSE_FLAG | (abi.STANDARD_WEIGHTS_FLAG if standard else 0)
    res = {}
    for name, launch in (("queued", None), ("inline", INLINE)):
        prev = None
        for frame in (1, 2):
            u = abi.make_uniforms(w, h, frame, sc.camera["position"], M=M,
                                  flags=flags | (abi.TEMPORAL_REUSE_FLAG if prev is not None else 0))
            out = torch.zeros(16 * w * h, dtype=torch.int32, device="cuda")
            r.ctx.profile_read()
            r.ctx.profile_enable(True)
            r.ctx.initial_temporal(u, g, g, prev, out, launch)
            rows = r.ctx.profile_read()
            r.ctx.profile_enable(False)
            if launch is None:
                assert ("k_pass_a_ris_split" in rows) == split
            prev = out
        res[name] = prev.clone()
    assert torch.equal(res["queued"], res["inline"])
