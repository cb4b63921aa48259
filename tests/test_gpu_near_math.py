"""The target function's cheaper divisions and roots at the ends of their operand range: the room
scaled by powers of two (squared distances from 2^-80 to 2^80 leave the range, so pixels take the
IEEE forms), metals (a zero diffuse factor), mirrors, and lights exactly on the axes of their
pixels (zero direction components). Every reservoir and colour equals the oracle's bit for bit."""
import numpy as np
import pytest

from restir_amd import scenes
from restir_amd.pipeline import Renderer
from test_gpu_parity import run_frame_and_compare

pytestmark = pytest.mark.gpu


def _scaled(exp):
    sc = scenes.cornell_box(3, n_lights=24)
    f = np.float32(2.0 ** exp)
    sc.tri_xyz = (sc.tri_xyz * f).astype(np.float32)
    sc.point_lights["pos"][:, :3] *= f
    cam = dict(sc.camera)
    for k in ("position", "lookAt"):
        cam[k] = tuple(float(v * f) for v in cam[k])
    cam["zNear"], cam["zFar"] = cam["zNear"] * float(f), cam["zFar"] * float(f)
    sc.camera = cam
    return sc


@pytest.mark.parametrize("exp", [-40, -30, -24, 24, 30, 40])
def test_scaled_room(exp):
    sc = _scaled(exp)
    r = Renderer(sc, 96, 64, mode="unbiased", k=3, spatial_passes=1, M=8)
    for _ in range(2):
        run_frame_and_compare(r, sc.camera)


@pytest.mark.parametrize("rough,metal", [(0.0, 1.0), (1.0, 1.0), (0.0, 0.0), (0.02, 0.5)])
def test_metals_mirrors_and_aligned_lights(rough, metal):
    sc = scenes.cornell_box(4, n_lights=16)
    sc.materials[:, 4], sc.materials[:, 5] = rough, metal
    W, H = 65, 63  # a centre column and row whose rays have zero components
    r = Renderer(sc, W, H, mode="biased", spatial_passes=1, M=16)
    r.render_gbuffer(sc.camera, 0)
    pos = r.gbuf[0].cpu().numpy()[: 3 * W * H].reshape(3, -1)
    pick = np.linspace(0, W * H - 1, 16).astype(int)  # lights straight above pixels
    sc.point_lights["pos"][:, 0] = pos[0, pick]
    sc.point_lights["pos"][:, 2] = pos[2, pick]
    r = Renderer(sc, W, H, mode="biased", spatial_passes=1, M=16)
    for _ in range(2):
        run_frame_and_compare(r, sc.camera)
