"""Pass A over an image of more than 2^27 pixels: the queued schedule's shadow verdicts reach the
pixels that they belong to (a tag of Pass C's tracer keeps a pixel in 27 bits, Pass A's in 32), single
view and multi-view. Only the first and the last two rows hold surface, so the pass is quick."""
import ctypes as C

import pytest

from restir_amd import abi, scenes
from restir_amd.pipeline import SceneOnDevice

pytestmark = pytest.mark.gpu

W, H = 65536, 2050  # row 2048's first pixel is number 2^27


def test_verdicts_beyond_2_27_pixels():
    import torch
    sc = scenes.cornell_box(1)
    ctx = abi.Context(0)
    dev = SceneOnDevice(ctx, sc, "cuda")
    n = W * H
    assert n > 1 << 27
    planes = torch.zeros(abi.GBUFFER_PLANES, n, dtype=torch.float32, device="cuda")
    g = abi.gbuffer_struct(planes.data_ptr(), W, H)
    # surface points of an ordinary G-buffer of the room, in rows 0, 1 (which the wrong verdicts would
    # reach) and 2048, 2049
    small = torch.zeros(abi.GBUFFER_PLANES * 256 * 256, dtype=torch.float32, device="cuda")
    ctx.primary_gbuffer(sc.camera, dev.d_tri_material, dev.d_materials, len(sc.materials), small, 256, 256)
    small = small.view(abi.GBUFFER_PLANES, -1)
    rows = [0, 1, 2048, 2049]
    gen = torch.Generator(device="cuda").manual_seed(3)
    for y in rows:
        planes[:, y * W:(y + 1) * W] = small[:, torch.randint(256 * 256, (W,), device="cuda", generator=gen)]
    u = abi.make_uniforms(W, H, 1, sc.camera["position"], M=2, flags=abi.VISIBILITY_REUSE_FLAG)
    out = torch.zeros(16 * n, dtype=torch.int32, device="cuda")

    def surface():
        torch.cuda.synchronize()
        return torch.cat([out[16 * y * W:16 * (y + 1) * W] for y in rows]).clone()

    def views(launch):
        v = abi.View(ctx.h.value, C.pointer(u), C.pointer(g), C.pointer(g), None, abi.as_ptr(out), None, 0)
        ctx.initial_temporal_views([v], launch)

    inline = abi.Launch(0, 0, abi.SCHEDULE_INLINE)
    ctx.initial_temporal(u, g, g, None, out, inline)
    ref = surface()
    w = ref.view(torch.float32).view(-1, 16)[:, 11]
    shadowed = (w == 0).view(4, W).sum(dim=1)
    assert (shadowed > W // 20).all() and (shadowed < W).all(), shadowed
    for name, run in (("single", lambda: ctx.initial_temporal(u, g, g, None, out)), ("views", lambda: views(None)),
                      ("views inline", lambda: views(inline))):
        out.zero_()
        run()
        assert torch.equal(surface(), ref), name
