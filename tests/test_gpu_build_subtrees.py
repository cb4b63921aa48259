"""The device tree build around the sizes at which ranges change hands: at most 512 triangles become a
subtree in one workgroup, more are split level by level first; inside a subtree, ranges above 32 fold
their bounds and bins another way. Against the host build byte for byte, over triangles with ties in
every coordinate (equal values, and zeros of both signs, of which the last one in order is kept),
coincident ones (halved at every level) and clusters that leave the sweep very uneven sides."""
import numpy as np
import pytest

from restir_amd import abi
from test_gpu_build import _assert_same_tree

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch as t
    assert t.cuda.is_available(), "GPU tests need a HIP device"
    return t


@pytest.fixture(scope="module")
def ctx(torch):
    return abi.Context(0)


def _soup(rng, n):
    return rng.standard_normal((n, 9)).astype(np.float32)


def _ties(rng, n):
    g = rng.integers(-3, 4, size=(n, 9)).astype(np.float32)
    return np.where(g == 0.0, np.where(rng.random((n, 9)) < 0.5, -0.0, 0.0), g).astype(np.float32)


def _coincident(rng, n):
    return np.tile(_soup(rng, 1), (n, 1))


def _uneven(rng, n):
    at = rng.choice([0.0, 1e-3, 1.0, 40.0], p=[0.9, 0.06, 0.03, 0.01], size=(n, 1))
    return (at + 1e-4 * rng.standard_normal((n, 9))).astype(np.float32)


@pytest.mark.parametrize("kind", [_soup, _ties, _coincident, _uneven])
@pytest.mark.parametrize("n", [4, 31, 33, 65, 511, 512, 513, 1025, 2600])
def test_matches_host_build(torch, ctx, kind, n):
    _assert_same_tree(torch, ctx, kind(np.random.default_rng(n), n), f"{kind.__name__} {n}")
