"""The wide learned proposal over its workgroup slots: images of fewer and of more tiles than there
are slots (two per compute unit), odd sizes, a count of clusters that is no power of two, few
candidates, two streams at a time in one context, and a captured graph that outlives the slots it
was recorded with.

Exact: a K = 256 network embedded in a wider one (every other cluster masked to a numerator of zero)
draws the lights and q of the K = 256 network bit for bit, from its own kernel.
"""
import numpy as np
import pytest

from restir_amd.learned import LearnedProposal
from restir_amd.pipeline import Renderer
from test_gpu_propose_wide import Embedded, many_light_terrain

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch as t
    assert t.cuda.is_available(), "GPU tests need a HIP device"
    return t


class Frame:
    def __init__(self, torch, W, H, M):
        self.torch, self.n = torch, M * W * H
        self.r = Renderer(many_light_terrain(5000), W, H)
        self.lp = LearnedProposal(self.r.ctx, self.r.scene, k=256, seed=9)
        self.r.begin_frame(self.r.scene.camera)
        self.u, _ = self.r.uniforms(self.r.scene.camera)
        self.g = self.r.gstruct(self.r.cur)
        self.M = M

    def outputs(self):
        return (self.torch.full((self.n,), -7, dtype=self.torch.int32, device="cuda"),
                self.torch.full((self.n,), -7.0, dtype=self.torch.float32, device="cuda"))

    def propose(self, mlp, out, stream=None):
        self.r.ctx.learned_candidates(self.u, self.g, mlp, self.lp.lo, self.lp.hi, self.M, self.lp.mix, *out,
                                      stream=stream)

    def narrow(self):
        out = self.outputs()
        self.propose(self.lp.mlp, out)
        return [o.cpu().numpy().copy() for o in out]

    def check(self, got, want):
        assert (want[0] >= 0).sum() > 100
        np.testing.assert_array_equal(got[0].cpu().numpy(), want[0])
        np.testing.assert_array_equal(got[1].cpu().numpy().view(np.uint32), want[1].view(np.uint32))


@pytest.mark.parametrize("W,H,M,K,offset", [(1, 1, 1, 384, 0), (65, 47, 5, 384, 128), (1031, 517, 3, 384, 0),
                                            (257, 129, 8, 2176, 1920)])
def test_equals_the_narrow_kernel(torch, W, H, M, K, offset):
    f = Frame(torch, W, H, M)
    want = f.narrow()
    e = Embedded(torch, f.lp, K, offset)
    f.r.ctx.set_light_clusters(K, *e.tables)
    got = f.outputs()
    f.propose(e.mlp, got)
    if W == 1:  # one pixel, which may be background
        np.testing.assert_array_equal(got[0].cpu().numpy(), want[0])
    else:
        f.check(got, want)


def test_two_streams(torch):
    f = Frame(torch, 1031, 517, 3)
    want = f.narrow()
    e = Embedded(torch, f.lp, 512, 256)
    f.r.ctx.set_light_clusters(512, *e.tables)
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    outs = [[f.outputs() for _ in range(4)] for _ in streams]
    torch.cuda.synchronize()
    for i in range(4):
        for s, o in zip(streams, outs):
            f.propose(e.mlp, o[i], s)
    torch.cuda.synchronize()
    for o in outs:
        for got in o:
            f.check(got, want)


def test_graph_outlives_its_slots(torch):
    f = Frame(torch, 64, 48, 8)
    want = f.narrow()
    e = Embedded(torch, f.lp, 512, 0)
    f.r.ctx.set_light_clusters(512, *e.tables)
    got = f.outputs()
    f.propose(e.mlp, got)  # eagerly first
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    s = torch.cuda.Stream()
    with torch.cuda.graph(graph, stream=s):
        f.propose(e.mlp, got, s)
    wide = Embedded(torch, f.lp, 4096, 1024)
    f.r.ctx.set_light_clusters(4096, *wide.tables)  # larger slots
    for _ in range(3):
        for o in got:
            o.fill_(-7)
        graph.replay()
        f.check(got, want)
        eager = f.outputs()
        f.propose(wide.mlp, eager)
        f.check(eager, want)


def test_slots_are_ready_on_return(torch):
    """set_light_clusters leaves nothing of the slots' set-up under way: a launch on a stream that does
    not wait for the default one may follow at once."""
    f = Frame(torch, 257, 129, 8)
    want = f.narrow()
    for k in (512, 1024, 2048, 4096):  # larger slots each time
        e = Embedded(torch, f.lp, k, k // 2)
        out, s = f.outputs(), torch.cuda.Stream()
        torch.cuda.synchronize()
        f.r.ctx.set_light_clusters(k, *e.tables)
        assert torch.cuda.default_stream().query()
        f.propose(e.mlp, out, s)
        torch.cuda.synchronize()
        f.check(out, want)


def test_two_networks_share_the_slots(torch):
    """Launches of 4,096 and 512 clusters in flight at a time, over the slots made for 4,096."""
    f = Frame(torch, 1031, 517, 3)
    want = f.narrow()
    big, small = Embedded(torch, f.lp, 4096, 1024), Embedded(torch, f.lp, 512, 256)
    f.r.ctx.set_light_clusters(4096, *big.tables)
    out, got = f.outputs(), [f.outputs() for _ in range(6)]
    f.propose(big.mlp, out)
    torch.cuda.synchronize()
    graph, streams = torch.cuda.CUDAGraph(), [torch.cuda.Stream(), torch.cuda.Stream()]
    with torch.cuda.graph(graph, stream=streams[0]):
        f.propose(big.mlp, out, streams[0])
    f.r.ctx.set_light_clusters(512, *small.tables)
    for o in out:
        o.fill_(-7)
    torch.cuda.synchronize()
    for o in got:
        with torch.cuda.stream(streams[0]):
            graph.replay()
        f.propose(small.mlp, o, streams[1])
    torch.cuda.synchronize()
    for o in [out, *got]:
        f.check(o, want)
