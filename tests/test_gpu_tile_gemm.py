"""Products of ordinary size (tile_gemm.hip): tile edges, row tails, K that is not whole steps, one and several K ranges,
against the oracle; results must not depend on which workgroup of a split product came last."""
import numpy as np
import pytest

import oracle as orc
from conftest import max_abs_rel

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def g():
    import gpu_util

    return gpu_util


# rows one below, at and one above tiles of 32 / 64 / 128; N odd, below and above a tile; K of half a step, odd halves of a
# step, long enough for several ranges
SHAPES = [(3, 33, 96), (15, 500, 2048), (16, 1, 16), (31, 64, 544), (33, 65, 4112), (64, 129, 2080), (97, 700, 5632), (129, 127, 1056), (260, 2050, 4096),
          (300, 20, 14336)]


@pytest.mark.parametrize("dt", [orc.F16, orc.BF16])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_dequant_matmul_tiles(g, dt, M, N, K):
    rng = np.random.default_rng(M + N + K)
    act = orc.to_storage(rng.standard_normal((M, K)), dt)
    W = rng.integers(-127, 128, (N, K)).astype(np.int8)
    sc = orc.to_storage(rng.uniform(1e-3, 1e-2, N), dt)
    want = orc.dequant_matmul(act, W, sc, dt, dt, mode=2 if M >= 16 else 0)
    da, dw, ds = g.to_dev(act, dt), g.to_dev(W), g.to_dev(sc, dt)
    first = g.to_host(g.mynn.dequant_matmul(da, dw, ds))
    assert max_abs_rel(g.f32(first, dt), g.f32(want, dt)) <= 1e-2
    assert np.mean(first == want) > 0.97
    for _ in range(5):
        assert np.array_equal(g.to_host(g.mynn.dequant_matmul(da, dw, ds)), first)


@pytest.mark.parametrize("dt", [orc.F16, orc.BF16, orc.F32])
@pytest.mark.parametrize("M,N,K", [(3, 33, 96), (31, 65, 544), (33, 700, 8192), (97, 129, 2080), (129, 2050, 4096), (300, 20, 14336)])
def test_quantized_matmul_tiles(g, dt, M, N, K):
    rng = np.random.default_rng(M + N + K)
    lhs, rhs = rng.integers(-128, 128, (M, K)).astype(np.int8), rng.integers(-128, 128, (N, K)).astype(np.int8)
    ls, rs = orc.to_storage(rng.uniform(1e-3, 1e-2, M), dt), orc.to_storage(rng.uniform(1e-3, 1e-2, N), dt)
    want, want_acc = orc.quantized_matmul(lhs, ls, rhs, rs, dt)
    args = [g.to_dev(lhs), g.to_dev(ls, dt), g.to_dev(rhs), g.to_dev(rs, dt)]
    for acc in (True, False):
        out, got_acc = g.mynn.quantized_matmul(*args, want_acc=acc)
        assert np.array_equal(g.to_host(out), want)
        if acc:
            assert np.array_equal(got_acc.cpu().numpy(), want_acc)


def test_split_products_replay_from_a_captured_graph(g):
    """The arrival counters of the K ranges are zero again after every launch: replays between eager calls on the same
    stream's workspace all give the eager result."""
    import torch

    dt, M, N, K = orc.F16, 100, 256, 8192
    rng = np.random.default_rng(3)
    W, sc = g.to_dev(rng.integers(-127, 128, (N, K)).astype(np.int8)), g.to_dev(orc.to_storage(rng.uniform(1e-3, 1e-2, N), dt), dt)
    act = g.to_dev(orc.to_storage(rng.standard_normal((M, K)), dt), dt)
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        g.mynn.dequant_matmul(act, W, sc)  # the stream's workspace exists
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            out = g.mynn.dequant_matmul(act, W, sc)
    for rep in range(3):
        act.copy_(g.to_dev(orc.to_storage(rng.standard_normal((M, K)), dt), dt))
        with torch.cuda.stream(side):
            want = g.mynn.dequant_matmul(act, W, sc)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want), rep
