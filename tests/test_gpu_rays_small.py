"""Visibility batches of every size class of the queue tracer (a wave per ray, several rays per wave,
full waves, chunks handed out) against one lane per ray, each verdict, and nothing written beyond the
batch."""
import numpy as np
import pytest

from restir_amd import scenes
from restir_amd.pipeline import Renderer

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def scene():
    import torch
    sc = scenes.terrain(11, grid=64, n_boxes=60, n_point_lights=500, extent=16.0)
    r = Renderer(sc, 64, 64, M=1)
    rng = np.random.default_rng(7)
    n = 330000
    tri = sc.tri_xyz.reshape(-1, 3, 3)[rng.integers(0, len(sc.tri_xyz), n)]
    w = rng.dirichlet((1.0, 1.0, 1.0), n)[:, :, None]
    p = np.ones((2, n, 4), np.float32)
    p[0, :, :3] = (tri * w).sum(1)
    p[1, :, :3] = sc.point_lights["pos"][rng.integers(0, 500, n)][:, :3]
    return r, torch.from_numpy(p[0]).cuda(), torch.from_numpy(p[1]).cuda()


@pytest.mark.parametrize("n", [1, 3, 64, 1279, 1280, 1281, 5001, 40960, 40961, 100003, 327680, 327681])
def test_verdicts(scene, n):
    import torch
    r, p1, p2 = scene
    out = [torch.full((n + 256,), 7, dtype=torch.int32, device="cuda") for _ in range(2)]
    r.ctx.trace_shadow(p1, p2, n, out[0])
    r.ctx.trace_shadow(p1, p2, n, out[1], one_ray_per_lane=True)
    assert torch.equal(out[0], out[1])
    assert bool((out[0][n:] == 7).all()) and bool((out[0][:n] <= 1).all())
