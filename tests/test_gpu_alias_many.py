"""The device alias-table build above 4,096 lights (power sum by increment maps, first rounds of the
pairing over the device) against the host build, byte for byte: sizes around the switch, the steps
and the segments; powers whose sum ties in its last bit (multiples of a half, small integers), stays
zero for long, spans many binades, or leaves few larges to many smalls."""
import numpy as np
import pytest

from restir_amd import abi

pytestmark = pytest.mark.gpu


def _powers(kind, n, rng):
    if kind == "log_uniform":
        p = np.exp(rng.uniform(np.log(0.01), np.log(10.0), n))
    elif kind == "halves":
        p = rng.integers(1, 2048, n) * 0.5
    elif kind == "integers":
        p = rng.integers(0, 5, n)
    elif kind == "zeros_first":
        p = np.where(np.arange(n) < n // 2, 0.0, rng.random(n))
    elif kind == "binades":
        p = np.exp(rng.uniform(-60.0, 20.0, n))
    elif kind == "few_larges":
        p = np.ones(n)
        p[rng.choice(n, 5, replace=False)] = n / 8.0
    else:  # one light with almost all the power: the smalls run out in its round
        p = np.full(n, 1e-3)
        p[n // 3] = 1e3
    return p.astype(np.float32)


def _build(torch, ctx, pts, cols):
    ctx.build_alias_table(pts, len(cols) // 16, None, 0, cols)


@pytest.mark.parametrize("kind", ["log_uniform", "halves", "integers", "zeros_first", "binades", "few_larges", "one"])
@pytest.mark.parametrize("n", [4096, 4097, 8193, 16385, 65793])
def test_large_tables_equal_the_host_build(kind, n):
    import torch
    if kind in ("few_larges", "one") and n > 10000:
        n = 10001  # thousands of rounds
    pts = np.zeros(n, dtype=abi.POINT_LIGHT_DTYPE)
    pts["color_lum"][:, 3] = _powers(kind, n, np.random.default_rng(n))
    host = abi.build_alias_table(pts, None)
    ctx = abi.Context(0)
    d = torch.from_numpy(pts.view(np.uint8).reshape(-1).copy()).cuda()
    cols = torch.full((16 * n,), 0xCD, dtype=torch.uint8, device="cuda")
    for _ in range(2):  # the second build finds the first one's scratch
        _build(torch, ctx, d, cols)
        got = cols.cpu().numpy().view(abi.ALIAS_DTYPE)
        bad = np.flatnonzero(got.view(np.uint32).reshape(n, 4).view("V16") != host.view(np.uint32).reshape(n, 4).view("V16"))
        assert len(bad) == 0, f"{kind} {n}: {len(bad)} columns differ, first {bad[0]}: {got[bad[0]]} {host[bad[0]]}"
        cols.fill_(0xCD)


def test_captured_with_and_without_the_large_scratch():
    import torch
    n = 6000
    pts = np.zeros(n, dtype=abi.POINT_LIGHT_DTYPE)
    pts["color_lum"][:, 3] = _powers("log_uniform", n, np.random.default_rng(1))
    host = abi.build_alias_table(pts, None).view(np.uint8)
    d = torch.from_numpy(pts.view(np.uint8).reshape(-1).copy()).cuda()
    for first in (7000, 4096):  # 7,000 lights' scratch holds the device-wide build's; 4,096 lights' does not
        ctx = abi.Context(0)
        warm = np.zeros(first, dtype=abi.POINT_LIGHT_DTYPE)
        warm["color_lum"][:, 3] = 1.0
        big = torch.zeros(16 * first, dtype=torch.uint8, device="cuda")
        _build(torch, ctx, torch.from_numpy(warm.view(np.uint8).reshape(-1).copy()).cuda(), big)
        torch.cuda.synchronize()
        m = n if first == 7000 else 4000  # what the scratch allowed before stays allowed
        cols = torch.zeros(16 * m, dtype=torch.uint8, device="cuda")
        s = torch.cuda.Stream()
        s.wait_stream(torch.cuda.current_stream())
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            ctx.build_alias_table(d, m, None, 0, cols, stream=s)
        want = host if m == n else abi.build_alias_table(pts[:m].copy(), None).view(np.uint8)
        for _ in range(3):
            cols.zero_()
            g.replay()
            torch.cuda.synchronize()
            assert np.array_equal(cols.cpu().numpy(), want)


def test_graph_of_the_small_scratch_survives_its_growth():
    """Above 4,096 lights with scratch for one workgroup only, a capture records that route; an eager
    build of the same size then needs the larger scratch, and the graph keeps the one it has."""
    import torch
    n = 6000
    ctx = abi.Context(0)
    want = {}
    for m in (5000, n, 20000):
        pts = np.zeros(m, dtype=abi.POINT_LIGHT_DTYPE)
        pts["color_lum"][:, 3] = _powers("log_uniform", m, np.random.default_rng(m))
        want[m] = (abi.build_alias_table(pts, None).view(np.uint8),
                   torch.from_numpy(pts.view(np.uint8).reshape(-1).copy()).cuda(),
                   torch.zeros(16 * m, dtype=torch.uint8, device="cuda"))

    def check(m):
        torch.cuda.synchronize()
        assert np.array_equal(want[m][2].cpu().numpy(), want[m][0]), m
        want[m][2].zero_()

    _build(torch, ctx, *want[5000][1:])  # device-wide: more than 6,000 lights take in one workgroup
    check(5000)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        ctx.build_alias_table(want[n][1], n, None, 0, want[n][2], stream=s)
    for m in (n, 20000):
        for _ in range(3):
            _build(torch, ctx, *want[m][1:])
            check(m)
            g.replay()
            check(n)
