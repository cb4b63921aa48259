"""The device tree build's pointer chains at their longest: `k` primitives that go right stand before
all the others, so the swap partition rotates the right block through the whole range and the
chains of the last `k` positions have about n / k links. Every node must equal the host build's."""
import numpy as np
import pytest

from restir_amd import abi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,k", [(257, 1), (1000, 3), (20000, 1), (300000, 2)])
def test_rotated_partition_with_long_chains(n, k):
    import torch
    rng = np.random.default_rng(n + k)
    c = rng.random((n, 1, 3), dtype=np.float32)
    c[:k, 0, 0] += 1000.0  # the outliers come first and end up on the right
    xyz = (c + 0.01 * rng.random((n, 3, 3), dtype=np.float32)).astype(np.float32).reshape(n, 9)
    nodes, tris, depth = abi.build_aabb_tree(xyz)
    ctx = abi.Context(0)
    d_nodes = torch.zeros(abi.NODE_DTYPE.itemsize * (n - 1), dtype=torch.uint8, device="cuda")
    d_tris = torch.zeros(abi.TRIANGLE_DTYPE.itemsize * n, dtype=torch.uint8, device="cuda")
    got = ctx.build_bvh(torch.from_numpy(xyz).cuda(), n, d_nodes, d_tris)
    assert got == depth
    assert d_nodes.cpu().numpy().tobytes() == nodes.tobytes()
    assert d_tris.cpu().numpy().tobytes() == tris.tobytes()
