"""Memory of a bound tree of 16 million triangles: the 8-entry nodes are sized by what a tree can have
of them at most, up to what their indices hold, and the count that the build finds decides whether they
cover it; where they cannot be had, the tree is bound over its 4-entry nodes."""
import pytest

from restir_amd import abi

pytestmark = pytest.mark.gpu

GRID = 2830
N = 2 * (GRID - 1) ** 2
HUGE_GRID = 4130  # more than 2^25 triangles


@pytest.fixture(scope="module")
def torch():
    import torch as t
    assert t.cuda.is_available(), "GPU tests need a HIP device"
    return t


def _field(torch, grid):
    """A height field's triangles, and their tree built by a first context."""
    g = torch.Generator(device="cuda").manual_seed(2)
    y = torch.rand(grid, grid, device="cuda", generator=g) * 2e-3
    x, z = torch.meshgrid(*[torch.linspace(-1, 1, grid, device="cuda")] * 2, indexing="ij")
    p = torch.stack([x, y, z], dim=2)
    a, b, c, d = p[:-1, :-1], p[1:, :-1], p[:-1, 1:], p[1:, 1:]
    xyz = torch.stack([torch.stack([a, b, c], 2), torch.stack([b, d, c], 2)], 2).reshape(-1, 9).contiguous()
    n = len(xyz)
    nodes = torch.zeros(80 * (n - 1), dtype=torch.uint8, device="cuda")
    tris = torch.zeros(48 * n, dtype=torch.uint8, device="cuda")
    ctx = abi.Context(0)
    ctx.build_bvh(xyz, n, nodes, tris)
    return ctx, nodes, tris


@pytest.fixture(scope="module")
def ground(torch):
    return _field(torch, GRID)


def _segments(torch, n=50000):
    g = torch.Generator(device="cuda").manual_seed(3)
    p1, p2 = torch.ones(n, 4, device="cuda"), torch.ones(n, 4, device="cuda")
    for p in (p1, p2):
        p[:, 0:3:2] = torch.rand(n, 2, device="cuda", generator=g) * 2 - 1
        p[:, 1] = torch.rand(n, device="cuda", generator=g) * 4e-3
    p2[: n // 2, 0:3:2] = p1[: n // 2, 0:3:2] + 1e-2 * (p2[: n // 2, 0:3:2] - p1[: n // 2, 0:3:2])
    return p1, p2


def _trace(torch, ctx, **kw):
    p1, p2 = _segments(torch)
    out = torch.full((len(p1),), 7, dtype=torch.int32, device="cuda")
    ctx.profile_read()
    ctx.profile_enable(True)
    ctx.trace_shadow(p1, p2, len(p1), out, **kw)
    rows = ctx.profile_read()
    ctx.profile_enable(False)
    torch.cuda.synchronize()
    # a batch that fits the 8-entry tracer's grid needs no counters
    return out, "k_zero_counters" not in rows


def test_the_nodes_found_decide(torch, ground):
    ctx = ground[0]
    ref, _ = _trace(torch, ctx, reference_loop=True)
    got, covered = _trace(torch, ctx)
    assert 0.05 < ref.float().mean() < 0.95
    assert torch.equal(got, ref)
    assert covered


def test_bound_without_room_for_8_entry_nodes(torch, ground):
    first, nodes, tris = ground
    ref, _ = _trace(torch, first, reference_loop=True)
    ctx = abi.Context(0)
    torch.cuda.empty_cache()
    # the 4-entry nodes take 2.05 GB, all of it 4.0
    leave, fill = 3 << 30, []
    while (free := torch.cuda.mem_get_info()[0] - leave) > (64 << 20):
        fill.append(torch.empty(min(free, 16 << 30) >> 21 << 21, dtype=torch.uint8, device="cuda"))
    assert abs(torch.cuda.mem_get_info()[0] - leave) < (512 << 20)
    ctx.set_bvh(nodes, N - 1, tris, N)
    got, covered = _trace(torch, ctx)
    assert torch.equal(got, ref) and not covered
    del fill
    torch.cuda.empty_cache()
    ctx.set_bvh(nodes, N - 1, tris, N)  # now there is
    got, covered = _trace(torch, ctx)
    assert torch.equal(got, ref) and covered


def test_walks_of_a_tree_beyond_32_bit_offsets(torch):
    """More than 2^25 nodes of 128 bytes: the 4-entry walk's quick form has 32 bits for their offsets."""
    assert 2 * (HUGE_GRID - 1) ** 2 - 1 > 1 << 25
    ctx, nodes, tris = _field(torch, HUGE_GRID)
    ref, _ = _trace(torch, ctx, reference_loop=True)
    visits = torch.zeros(len(ref), dtype=torch.int32, device="cuda")
    for name, kw in (("first hit", {}), ("with counts", {"visits": visits}), ("a ray per lane", {"one_ray_per_lane": True})):
        got, _ = _trace(torch, ctx, **kw)
        assert torch.equal(got, ref), name
