"""The queue tracer's 8-entry nodes (no counts asked for) against the oracle's binary walk.

Every verdict must equal the reference's (oracle_trace_shadow) whatever the segment or the tree:
random segments; segments with zero direction components on box planes (0/0 in the reference's
slabs); tiny and huge components; origins outside the reach of the grown boxes and non-finite
segments (walked through the binary tree); a tree whose boxes are not nested and one whose leaf
boxes are not their triangles' bounds (hits are then confirmed box by box up to the root); a tree
too deep for the 8-entry nodes; the smallest trees (2 triangles up to more than one node's worth).
"""
import numpy as np
import pytest

import oracle
from restir_amd import abi, scenes
from rt_helpers import HostScene, random_segments
from test_gpu_wide import _bind, _plane_segments

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch as t
    assert t.cuda.is_available(), "GPU tests need a HIP device"
    return t


def _check(torch, ctx, osc, p1, p2, name):
    ref, _, _ = oracle.trace_shadow(osc, p1, p2)
    n = len(p1)
    out = torch.full((n,), 7, dtype=torch.int32, device="cuda")
    ctx.trace_shadow(torch.from_numpy(p1).cuda(), torch.from_numpy(p2).cuda(), n, out)
    got = out.cpu().numpy().astype(np.uint32)
    bad = np.flatnonzero(got != ref)
    assert len(bad) == 0, f"{name}: {len(bad)} of {n} verdicts differ, first rays {bad[:4]}"
    return ref


def _odd_segments(rng, lo, hi, n):
    """Segments with tiny, huge, non-finite or far-away coordinates, one kind after another."""
    p1, p2 = random_segments(rng, lo, hi, n)
    ax = rng.integers(3, size=n)
    i = np.arange(n)
    kind = i % 8
    tiny = kind == 0  # a component far below the clamp of 1/d
    p1[i[tiny], ax[tiny]] = 0.0
    p2[i[tiny], ax[tiny]] = np.float32(1e-35)
    far1 = kind == 1  # origins from just inside to far outside the grown boxes' reach
    p1[far1, :3] *= np.float32(2.0) ** rng.integers(2, 12, size=(far1.sum(), 1)).astype(np.float32)
    far2 = kind == 2
    p2[far2, :3] *= np.float32(1e6)
    nan = kind == 3
    p1[i[nan], ax[nan]] = np.nan
    inf = kind == 4
    p2[i[inf], ax[inf]] = np.inf
    point = kind == 5  # no direction at all (0/0 in the shrunk segment)
    p2[point] = p1[point]
    return p1, p2


@pytest.mark.parametrize("name", ["cornell", "terrain_small"])
def test_wide8_verdicts(torch, name):
    sc = scenes.cornell_box(1) if name == "cornell" else scenes.terrain(5, grid=64, n_boxes=100, n_point_lights=10)
    hs = HostScene(sc)
    ctx = abi.Context(0)
    keep = _bind(torch, ctx, hs.nodes, hs.tris)
    lo, hi = sc.aabb()
    rng = np.random.default_rng(21)
    ref = _check(torch, ctx, hs.oracle, *random_segments(rng, lo, hi, 60000), f"{name} random")
    assert 0.05 < ref.mean() < 0.95
    ref = _check(torch, ctx, hs.oracle, *_plane_segments(rng, hs.nodes, lo, hi, 40000), f"{name} plane")
    assert 0.02 < ref.mean() < 0.98
    _check(torch, ctx, hs.oracle, *_odd_segments(rng, lo, hi, 16000), f"{name} odd")
    del keep


@pytest.mark.parametrize("what", ["not nested", "loose leaves"])
def test_wide8_on_a_foreign_tree(torch, what):
    sc = scenes.terrain(5, grid=64, n_boxes=100, n_point_lights=10)
    hs = HostScene(sc)
    nodes = hs.nodes.copy()
    lo, hi = sc.aabb()
    if what == "not nested":  # shrink the boxes stored for some inner subtrees: the reference culls there
        inner = [i for i in range(7, 400) if nodes[i]["left"] > 0]
        for x in inner[::5]:
            ax = int(np.argmax(nodes[x]["lmax"][:3] - nodes[x]["lmin"][:3]))
            ext = nodes[x]["lmax"][ax] - nodes[x]["lmin"][ax]
            nodes[x]["lmax"][ax] = nodes[x]["lmin"][ax] + np.float32(0.3) * ext
    else:  # leaf boxes cut to half their triangle: nested, but not the triangles' bounds
        leaf = np.flatnonzero(nodes["left"] < 0)[::3]
        ext = nodes["lmax"][leaf, :3] - nodes["lmin"][leaf, :3]
        nodes["lmax"][leaf, :3] = nodes["lmin"][leaf, :3] + np.float32(0.5) * ext
    osc = oracle.Scene(nodes, hs.tris, None, None, None)
    ctx = abi.Context(0)
    keep = _bind(torch, ctx, nodes, hs.tris)
    rng = np.random.default_rng(22)
    p1, p2 = random_segments(rng, lo, hi, 60000)
    ref = _check(torch, ctx, osc, p1, p2, what)
    orig, _, _ = oracle.trace_shadow(hs.oracle, p1, p2)
    assert (orig != ref).sum() > 50, "the changed boxes change too few verdicts"
    _check(torch, ctx, osc, *_plane_segments(rng, nodes, lo, hi, 20000), f"{what} plane")
    del keep


@pytest.mark.parametrize("n_tris", [2, 3, 4, 5, 8, 9, 31, 33, 65])
def test_wide8_small_trees(torch, n_tris):
    rng = np.random.default_rng(100 + n_tris)
    xyz = (rng.uniform(-1, 1, size=(n_tris, 1, 3)) + rng.uniform(-0.4, 0.4, size=(n_tris, 3, 3))).astype(np.float32)
    nodes, tris, _ = abi.build_aabb_tree(xyz.reshape(-1, 9))
    osc = oracle.Scene(nodes, tris, None, None, None)
    ctx = abi.Context(0)
    keep = _bind(torch, ctx, nodes, tris)
    lo, hi = np.full(3, -1.4, np.float32), np.full(3, 1.4, np.float32)
    for n in (1, 63, 4097):
        _check(torch, ctx, osc, *random_segments(rng, lo, hi, n), f"{n_tris} triangles, {n} rays")
    del keep


def test_wide8_chain_tree(torch):
    """A chain (one triangle split off per node): 60 levels collapse to 9 levels of 8 entries;
    coincident triangles everywhere keep every box passing."""
    n = 60
    rng = np.random.default_rng(9)
    xyz = np.zeros((n, 9), np.float32)
    for i in range(n):
        xyz[i] = (rng.uniform(-0.2, 0.2, size=(3, 3)) + np.array([i * 0.5, 0, 0])).astype(np.float32).reshape(-1)
    _, tris, _ = abi.build_aabb_tree(xyz)
    v = xyz.reshape(n, 3, 3)
    tmin, tmax = v.min(axis=1), v.max(axis=1)
    nodes = np.zeros(n - 1, dtype=abi.NODE_DTYPE)
    for i in range(n - 1):
        last = i == n - 2
        nodes[i]["lmin"], nodes[i]["lmax"] = [*tmin[i], 1], [*tmax[i], 1]
        nodes[i]["rmin"] = [*tmin[i + 1:].min(axis=0), 1]
        nodes[i]["rmax"] = [*tmax[i + 1:].max(axis=0), 1]
        nodes[i]["left"], nodes[i]["right"] = ~i, (~(n - 1) if last else i + 1)
    osc = oracle.Scene(nodes, tris, None, None, None)
    ctx = abi.Context(0)
    keep = _bind(torch, ctx, nodes, tris)
    lo, hi = np.array([-1, -0.4, -0.4], np.float32), np.array([31, 0.4, 0.4], np.float32)
    ref = _check(torch, ctx, osc, *random_segments(np.random.default_rng(10), lo, hi, 30000), "chain")
    assert 0.02 < ref.mean() < 0.98
    del keep


@pytest.mark.parametrize("levels", [17, 18, 30])
def test_wide8_spine_tree(torch, levels):
    """Each node has a subtree of 8 large triangles and the rest of the tree, half as large: the
    largest entries come first, so every level takes an 8-entry level of its own. 17 levels just
    fit the tracer's stack; deeper trees stay on the 4-entry nodes."""
    rng = np.random.default_rng(levels)
    tri, nodes = [], []

    def box(ids):
        v = np.concatenate([tri[i] for i in ids])
        return [*v.min(axis=0), 1.0], [*v.max(axis=0), 1.0]

    def node(a, b):  # a, b: (child, triangles below)
        n = np.zeros(1, dtype=abi.NODE_DTYPE)[0]
        n["lmin"], n["lmax"] = box(a[1])
        n["rmin"], n["rmax"] = box(b[1])
        n["left"], n["right"] = a[0], b[0]
        nodes.append(n)
        return len(nodes) - 1, a[1] + b[1]

    def eight(scale):
        part = []
        for _ in range(8):
            tri.append((rng.uniform(-1, 1, size=(3, 3)) * scale).astype(np.float32))
            part.append((~(len(tri) - 1), [len(tri) - 1]))
        while len(part) > 1:
            part = [node(part[i], part[i + 1]) for i in range(0, len(part), 2)]
        return part[0]

    rest = eight(0.5 ** (levels - 1))
    for lv in range(levels - 2, -1, -1):
        rest = node(eight(0.5 ** lv), rest)
    arr = np.array(nodes, dtype=abi.NODE_DTYPE)[::-1].copy()  # node 0 is the root
    for side in ("left", "right"):
        inner = arr[side] >= 0
        arr[side][inner] = len(arr) - 1 - arr[side][inner]
    tris = np.ones((len(tri), 3, 4), np.float32)
    tris[:, :, :3] = np.array(tri)
    tris = tris.reshape(-1).view(abi.TRIANGLE_DTYPE)
    osc = oracle.Scene(arr, tris, None, None, None)
    ctx = abi.Context(0)
    keep = _bind(torch, ctx, arr, tris)
    p1, p2 = random_segments(rng, -np.ones(3, np.float32), np.ones(3, np.float32), 20000)
    s = (np.float32(0.5) ** rng.integers(0, levels, size=(20000, 1))).astype(np.float32)
    p1[:, :3] *= s
    p2[:, :3] *= s
    ref = _check(torch, ctx, osc, p1, p2, f"spine of {levels}")
    assert 0.02 < ref.mean() < 0.999
    del keep


def _long_segments(rng, lo, hi, n, reach):
    """Segments from the scene to `reach` times its size and beyond, up to the largest float, along one
    axis, two or all three (whose other components keep the scene's size), through its middle."""
    size = float((hi - lo).max())
    p1, p2 = random_segments(rng, lo, hi, n)
    axes = rng.integers(1, 8, size=n)
    length = np.exp(rng.uniform(np.log(size * reach), np.log(3.3e38), size=n))
    for a in range(3):
        far = (axes >> a) & 1 != 0
        sign = rng.choice((-1.0, 1.0), size=n)
        p2[far, a] = (sign * length * rng.uniform(0.2, 1.0, size=n))[far].astype(np.float32)
    return p1, p2


@pytest.mark.parametrize("size", [1.0, 1e-8, 1e-12])
def test_wide8_long_segments(torch, size):
    """A segment's component above 2^126 has a reciprocal that the hardware flushes to zero, and far
    shorter ones leave a tiny scene's slab distances without bits: the binary walk takes those."""
    sc = scenes.terrain(5, grid=64, n_boxes=100, n_point_lights=10)
    lo, hi = sc.aabb()
    scale = size / float((hi - lo).max())
    xyz = (sc.tri_xyz.reshape(-1, 9).astype(np.float64) * scale).astype(np.float32)
    lo, hi = lo.astype(np.float64) * scale, hi.astype(np.float64) * scale
    nodes, tris, _ = abi.build_aabb_tree(xyz)
    osc = oracle.Scene(nodes, tris, None, None, None)
    ctx = abi.Context(0)
    keep = _bind(torch, ctx, nodes, tris)
    rng = np.random.default_rng(23)
    p1, p2 = _long_segments(rng, lo, hi, 60000, 1e2)
    ref = _check(torch, ctx, osc, p1, p2, f"long, size {size}")
    # what the walk over rounded slab distances gets wrong is occluded segments
    top = np.abs(p2[:, :3] - p1[:, :3]).max(axis=1) > 2.0 ** 126
    assert ref.sum() > 200 and (size != 1.0 or ref[top].sum() > 20), (ref.sum(), ref[top].sum())
    del keep


@pytest.mark.parametrize("how", ["host", "device"])
@pytest.mark.parametrize("size", [1e17, 1e19, 3.3e38])
def test_wide8_enormous_boxes(torch, size, how):
    """Boxes up to the largest float, flat ones among them (whose area would be inf * 0): beyond the
    coordinates that the 8-entry nodes cover, the tree keeps its 4-entry nodes."""
    rng = np.random.default_rng(31)
    n = 300
    xyz = np.zeros((n, 3, 3))
    xyz[:, :, 0] = rng.uniform(-1, 1, size=(n, 1)) + rng.uniform(-0.2, 0.2, size=(n, 3))
    xyz[:, :, 2] = rng.uniform(-1, 1, size=(n, 1)) + rng.uniform(-0.2, 0.2, size=(n, 3))
    xyz[n // 2:, :, 1] = rng.uniform(-1e-3, 1e-3, size=(n - n // 2, 3))  # the first half is flat
    xyz = (np.clip(xyz, -1, 1) * size).astype(np.float32)
    nodes, tris, _ = abi.build_aabb_tree(xyz.reshape(-1, 9))
    osc = oracle.Scene(nodes, tris, None, None, None)
    ctx = abi.Context(0)
    if how == "host":
        keep = _bind(torch, ctx, nodes, tris)
    else:
        keep = (torch.from_numpy(xyz).cuda(), torch.zeros(nodes.nbytes, dtype=torch.uint8, device="cuda"),
                torch.zeros(tris.nbytes, dtype=torch.uint8, device="cuda"))
        ctx.build_bvh(keep[0], n, keep[1], keep[2])
        assert keep[1].cpu().numpy().tobytes() == nodes.tobytes()
    lo, hi = np.array([-1, -1e-3, -1]) * size * 0.5, np.array([1, 1e-3, 1]) * size * 0.5
    _check(torch, ctx, osc, *random_segments(rng, lo, hi, 20000), f"size {size}")
    del keep


@pytest.mark.parametrize("name", ["cornell", "terrain_small"])
def test_wide8_far_origins(torch, name):
    """Origins from inside the reach of the grown boxes, over the far ones whose slab distances get a
    slack per ray, to those that walk the binary tree; each mixed with near ones in its wave."""
    sc = scenes.cornell_box(1) if name == "cornell" else scenes.terrain(5, grid=64, n_boxes=100, n_point_lights=10)
    hs = HostScene(sc)
    ctx = abi.Context(0)
    keep = _bind(torch, ctx, hs.nodes, hs.tris)
    lo, hi = sc.aabb()
    big = max(np.abs(lo).max(), np.abs(hi).max())
    rng = np.random.default_rng(25)
    n = 80000
    p1, p2 = random_segments(rng, lo, hi, n)
    v = rng.normal(size=(n, 3))
    v[::5] = np.eye(3)[rng.integers(3, size=len(v[::5]))] * rng.choice([-1, 1], size=(len(v[::5]), 1))  # axis-parallel
    far = rng.uniform(size=n) < 0.9
    dist = big * 2.0 ** rng.uniform(2, 27, size=n)
    ends = p1[:, :3] + v / np.linalg.norm(v, axis=1, keepdims=True) * dist[:, None]
    p1[far, :3] = ends[far].astype(np.float32)
    # a segment may also start at the far end's light and lead past the scene
    past = rng.uniform(size=n) < 0.3
    p2[past, :3] += (p2[past, :3] - p1[past, :3]) * np.float32(0.5)
    ref = _check(torch, ctx, hs.oracle, p1, p2, f"{name} far")
    for k in range(4, 24, 4):
        some = far & (dist > big * 2.0 ** k) & (dist < big * 2.0 ** (k + 4))
        assert 0.05 < ref[some].mean() < 0.98, k
    del keep


@pytest.mark.parametrize("n_tris", [1119, 1120, 1121, 3000])
def test_wide8_one_workgroup_or_many(torch, n_tris):
    """Up to 640 possible nodes the collapse is one workgroup's; both sides of that, host and device build."""
    rng = np.random.default_rng(n_tris)
    xyz = (rng.uniform(-1, 1, size=(n_tris, 1, 3)) + rng.uniform(-0.1, 0.1, size=(n_tris, 3, 3))).astype(np.float32)
    nodes, tris, _ = abi.build_aabb_tree(xyz.reshape(-1, 9))
    osc = oracle.Scene(nodes, tris, None, None, None)
    lo, hi = np.full(3, -1.1, np.float32), np.full(3, 1.1, np.float32)
    for how in ("host", "device"):
        ctx = abi.Context(0)
        for _ in range(2):  # again over the buffers of the first
            if how == "host":
                keep = _bind(torch, ctx, nodes, tris)
            else:
                keep = (torch.from_numpy(xyz).cuda(), torch.zeros(nodes.nbytes, dtype=torch.uint8, device="cuda"),
                        torch.zeros(tris.nbytes, dtype=torch.uint8, device="cuda"))
                ctx.build_bvh(keep[0], n_tris, keep[1], keep[2])
        ctx.profile_enable(True)
        ref = _check(torch, ctx, osc, *random_segments(rng, lo, hi, 20000), f"{n_tris} triangles, {how}")
        assert "k_zero_counters" not in ctx.profile_read(), "the 8-entry nodes do not cover the tree"
        assert 0.02 < ref.mean() < 0.98
        del keep
