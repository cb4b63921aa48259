"""Forward pass, loss and gradients of the proposal's network over tiles of 32 samples, at the sizes
where the tiles change shape: the smallest batch, batches that are no power of two (one and several
ranges of samples per weight gradient), 64 clusters (half a staged block of output weights), and
counts of clusters split over 128 and over 256 per workgroup. Against the oracle, with the tolerances
of the tests at K = 256 and 4,096."""
import numpy as np
import pytest

import oracle
from restir_amd import abi
from restir_amd.abi import MlpStruct, mlp_sizes
from test_gpu_mlp import bf16_to_f32, rand_features

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K,n", [(64, 64), (64, 4096), (128, 192), (384, 128), (512, 1088), (256, 320)])
def test_matches_oracle(K, n):
    import torch
    ctx = abi.Context(0)
    nW, nB = mlp_sizes(K)
    z = lambda m, t=torch.float32: torch.zeros(m, dtype=t, device="cuda")  # noqa: E731
    w_bf16, w, b, m, v = z(nW, torch.int16), z(nW), z(nB), z(nW + nB), z(nW + nB)
    mlp = MlpStruct(K, 0, w_bf16.data_ptr(), w.data_ptr(), b.data_ptr(), m.data_ptr(), v.data_ptr())
    rng = np.random.default_rng(K + n)
    ctx.mlp_init(mlp, 5, torch.from_numpy(rng.normal(0, 1, K).astype(np.float32)).cuda())
    b[:384] = torch.from_numpy(rng.normal(0, 0.1, 384).astype(np.float32)).cuda()
    X16, Xf = rand_features(torch, n, 1)
    Wf, Bf = bf16_to_f32(w_bf16), b.cpu().numpy()
    logits = torch.full((n, K), 7e30, dtype=torch.float32, device="cuda")
    ctx.mlp_forward(mlp, X16, n, logits)
    ref = oracle.mlp_forward(Wf, Bf, K, Xf, emulate_bf16=True)
    assert np.linalg.norm(logits.cpu().numpy().astype(np.float64) - ref) / np.linalg.norm(ref) < 2e-3
    tgt = rng.integers(0, K, n).astype(np.int32)
    mask = (rng.uniform(size=n) < 0.8).astype(np.uint32)
    gw, gb, loss = z(nW), z(nB), z(1)
    ctx.mlp_loss_grad(mlp, X16, torch.from_numpy(tgt).cuda(), torch.from_numpy(mask).cuda(), n, gw, gb, loss)
    ref_loss, rgW, rgB = oracle.mlp_loss_grad(Wf, Bf, K, Xf, tgt, mask.astype(np.uint8), emulate_bf16=True)
    assert abs(loss.item() - ref_loss) < 1e-3 * abs(ref_loss)
    gW, gB = gw.cpu().numpy().astype(np.float64), gb.cpu().numpy().astype(np.float64)
    for layer in range(4):
        rows = 128 if layer < 3 else K
        sl, bl = slice(layer * 128 * 128, (layer * 128 + rows) * 128), slice(layer * 128, layer * 128 + rows)
        assert np.linalg.norm(gW[sl] - rgW[sl]) / np.linalg.norm(rgW[sl]) < 2e-2, layer
        assert np.linalg.norm(gB[bl] - rgB[bl]) / np.linalg.norm(rgB[bl]) < 2e-2, layer


def test_graph_keeps_its_scratch():
    """A captured step's activations and partial sums stay its own when a larger batch needs more."""
    import torch
    K, n, larger = 256, 256, 4096
    ctx = abi.Context(0)
    nW, nB = mlp_sizes(K)
    z = lambda m, t=torch.float32: torch.zeros(m, dtype=t, device="cuda")  # noqa: E731
    w_bf16, w, b, m, v = z(nW, torch.int16), z(nW), z(nB), z(nW + nB), z(nW + nB)
    mlp = MlpStruct(K, 0, w_bf16.data_ptr(), w.data_ptr(), b.data_ptr(), m.data_ptr(), v.data_ptr())
    ctx.mlp_init(mlp, 5, z(K))
    X, tgt, mask = rand_features(torch, larger, 1)[0], z(larger, torch.int32), z(larger, torch.int32) + 1
    out = z(nW), z(nB), z(1)

    def step(count, stream=None):
        ctx.mlp_loss_grad(mlp, X, tgt, mask, count, *out, stream=stream)

    def results():
        torch.cuda.synchronize()
        got = [t.clone() for t in out]
        for t in out:
            t.zero_()
        return got

    step(n)
    ref = results()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        step(n, s)
    for _ in range(3):
        step(larger)
        assert results()[2].item() > 0
        graph.replay()
        assert all(torch.equal(a, c) for a, c in zip(results(), ref))


@pytest.mark.parametrize("K,n", [(128, 8192), (384, 4096), (384, 8192), (640, 4096), (640, 16384), (1024, 320), (3968, 1088)])
def test_groups_of_clusters_give_the_same_logits(K, n):
    """A workgroup's share of the clusters depends on the batch: groups of one to all blocks of 128, the
    last of them shorter. A sample's logits don't."""
    import torch
    ctx = abi.Context(0)
    nW, nB = mlp_sizes(K)
    z = lambda m, t=torch.float32: torch.zeros(m, dtype=t, device="cuda")  # noqa: E731
    w_bf16, w, b, m, v = z(nW, torch.int16), z(nW), z(nB), z(nW + nB), z(nW + nB)
    mlp = MlpStruct(K, 0, w_bf16.data_ptr(), w.data_ptr(), b.data_ptr(), m.data_ptr(), v.data_ptr())
    ctx.mlp_init(mlp, 5, z(K) + torch.arange(K, device="cuda") * 0.25)
    X = rand_features(torch, n, 1)[0]
    got, piece = z(n * K).view(n, K) - 1, z(64 * K).view(64, K)
    ctx.mlp_forward(mlp, X, n, got)
    for i in range(0, n, 64 * (1 + n // 1024)):
        ctx.mlp_forward(mlp, X[i:i + 64], 64, piece)
        assert torch.equal(got[i:i + 64], piece), i
    assert got.std() > 0.1 and not (got == -1).any()
