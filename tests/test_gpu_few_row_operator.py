"""DequantMatMul of 2 .. 15 rows over whole 128-byte lines of row-major weights (rowblock.hip): one to eight and nine to fifteen rows, fewer
weight rows than a block, ragged blocks of every workgroup form, K of fewer steps than waves and of one more than they share evenly;
outputs and operands at odd places; against the sums in 64 bits, the same bits from the workspace form and from a captured call."""
import numpy as np
import pytest

import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def g():
    import gpu_util

    return gpu_util


@pytest.mark.parametrize("dt", [orc.F16, orc.BF16])
@pytest.mark.parametrize("M", [2, 8, 9, 15])
@pytest.mark.parametrize("N,K", [(1, 128), (15, 256), (33, 1152), (4096, 2048), (4099, 384), (8193, 1024), (12290, 640), (16400, 1152), (700, 14336)])
def test_few_rows_row_major(g, dt, M, N, K):
    import torch

    rng = np.random.default_rng(M + N + K)
    act, sc = orc.to_storage(rng.standard_normal((M, K)), dt), orc.to_storage(rng.uniform(1e-3, 1e-2, N), dt)
    W = rng.integers(-128, 128, (N, K)).astype(np.int8)
    da, dw, ds = g.to_dev(act, dt), g.to_dev(W), g.to_dev(sc, dt)
    got = g.mynn.dequant_matmul(da, dw, ds)
    a, s = g.f32(act, dt).astype(np.float64).reshape(M, K), g.f32(sc, dt).astype(np.float64)
    w = W.astype(np.float64)
    exact = (a @ w.T) * s
    # f32 sums of K exact products in any order, one rounding of the stored value
    bound = (np.abs(a) @ np.abs(w).T) * s * K * 2.0 ** -24 + np.abs(exact) * (2.0 ** -8 if dt == orc.BF16 else 2.0 ** -11) * 1.01 + 1e-30
    assert np.all(np.abs(g.f32(g.to_host(got), dt).reshape(M, N) - exact) <= bound)
    assert torch.equal(g.mynn.dequant_matmul_ws(da, dw, ds), got)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        out = g.mynn.dequant_matmul(da, dw, ds)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, got)
