"""The primary rays over the 8-entry nodes against the oracle's brute-force closest hits, bit for
bit: images at the edges of the 16x16 tiles and with a centre column whose rays have a zero
direction component, cameras inside and outside the scene and beyond the reach of the grown boxes
(there the binary walk renders the image)."""
import numpy as np
import pytest

from restir_amd import abi, scenes
from restir_amd.pipeline import Renderer
from rt_helpers import HostScene, floats_equal_nan

pytestmark = pytest.mark.gpu

SIZES = [(1, 1), (15, 17), (16, 16), (33, 31), (65, 48)]


@pytest.mark.parametrize("name", ["cornell", "terrain_small"])
@pytest.mark.parametrize("place", ["own", "inside", "beside", "far"])
def test_primary_hits(name, place):
    import torch
    sc = scenes.cornell_box(1) if name == "cornell" else scenes.terrain(5, grid=24, n_boxes=20, n_point_lights=4)
    hs = HostScene(sc)
    lo, hi = sc.aabb()
    mid, ext = (lo + hi) / 2, hi - lo
    cam = dict(sc.camera)
    if place != "own":
        shift = {"inside": (0.1, 0.3, -0.2), "beside": (3.0, 0.6, 1.0), "far": (40.0, 3.0, 0.0)}[place]
        cam["position"] = tuple(float(v) for v in mid + np.array(shift) * ext.max() / 2)
        cam["lookAt"] = tuple(float(v) for v in mid)
    for W, H in SIZES:
        r = Renderer(sc, W, H, M=1)
        r.render_gbuffer(cam, 0)
        torch.cuda.synchronize()
        got = r.gbuf[0].cpu().numpy()
        ref = hs.oracle_gbuffer(W, H, cam)
        ref = ref[0] if isinstance(ref, tuple) else ref
        bad = ~floats_equal_nan(got[: 13 * W * H], np.asarray(ref).reshape(-1)[: 13 * W * H])
        assert not bad.any(), f"{name} {place} {W}x{H}: {int(bad.sum())} values differ"
