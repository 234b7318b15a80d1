"""DequantMatMul of 16 and more rows has one order of sums for a shape and type, also where a long K is summed up in several
ranges: the plain call, the same captured into a graph, the caller-workspace form, every forced tile, a prepared weight and
weights that are not aligned for the tiles give the same bits."""
import numpy as np
import pytest

import oracle as orc
from conftest import max_abs_rel

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def g():
    import gpu_util

    return gpu_util


def captured(torch, call):
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        out = call()
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
    return out


# one and two row tiles of 16 .. 300 rows x few and many columns; K of two steps, of half a step more, of 4 .. 8 ranges; the
# last two: 256-row tiles that do not fill the device once, whole and ragged (captured on a new stream: the int8 tiles)
@pytest.mark.parametrize("dt", [orc.F16, orc.BF16])
@pytest.mark.parametrize("M,N,K", [(16, 2048, 2048), (64, 2048, 2048), (33, 65, 4112), (100, 256, 8192), (128, 4096, 4096), (300, 4096, 14336),
                                   (300, 1000, 4096), (17, 31, 128), (40, 72, 2200), (1500, 5632, 2048), (1300, 7177, 1088)])
@pytest.mark.parametrize("size", [1.0, 1e-5])  # (1e-5: fp16 weights that are subnormal once scaled)
def test_same_bits_from_every_form(g, dt, M, N, K, size):
    import torch

    rng = np.random.default_rng(M + N + K)
    act, sc = orc.to_storage(rng.standard_normal((M, K)), dt), orc.to_storage(rng.uniform(1e-3, 1e-2, N) * size, dt)
    W = rng.integers(-127, 128, (N, K)).astype(np.int8)
    da, dw, ds = g.to_dev(act, dt), g.to_dev(W), g.to_dev(sc, dt)
    want = g.mynn.dequant_matmul(da, dw, ds)
    if N * K * M < 1 << 28:
        assert max_abs_rel(g.f32(g.to_host(want), dt), g.f32(orc.dequant_matmul(act, W, sc, dt, dt, mode=2), dt)) <= 1e-2
    wt = g.mynn.dequant_weight_prepare(dw, ds)
    for tile in (0, 1, 2, 3, 4):
        assert torch.equal(g.mynn.dequant_matmul_prepared(da, wt, N, gemm_tile=tile), want), tile
        assert torch.equal(g.mynn.dequant_matmul_ws(da, dw, ds, gemm_tile=tile), want), tile
    odd = torch.empty(N * K + 8, dtype=torch.int8, device="cuda")[8:].view(N, K)  # (8-byte aligned)
    odd.copy_(dw)
    assert torch.equal(g.mynn.dequant_matmul(da, odd, ds), want)
    if K % 16 == 0:  # (else the call dequantises into the stream's block, and there is none yet on a new stream)
        assert torch.equal(captured(torch, lambda: g.mynn.dequant_matmul(da, dw, ds)), want)


@pytest.mark.parametrize("dt", [orc.F16, orc.BF16])
@pytest.mark.parametrize("M,N,K", [(3, 33, 96), (6, 4096, 14336), (15, 500, 2064)])
def test_few_rows_captured(g, dt, M, N, K):
    """the same below 16 rows (scale after the sum)"""
    import torch

    rng = np.random.default_rng(M + N + K)
    act = g.to_dev(orc.to_storage(rng.standard_normal((M, K)), dt), dt)
    W = g.to_dev(rng.integers(-127, 128, (N, K)).astype(np.int8))
    sc = g.to_dev(orc.to_storage(rng.uniform(1e-3, 1e-2, N), dt), dt)
    want = g.mynn.dequant_matmul(act, W, sc)
    assert torch.equal(captured(torch, lambda: g.mynn.dequant_matmul(act, W, sc)), want)
