"""QuantizedMatMul of 2 .. 128 rows (qrows.hip): one to four groups of 8 rows and several of 32, fewer weight rows than a block and ragged blocks of every
workgroup form, K of fewer steps than waves, of one more than they share evenly and of twice the stages of the rings and more for each wave;
integer sums and outputs, bit for bit."""
import numpy as np
import pytest

import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def g():
    import gpu_util

    return gpu_util


@pytest.mark.parametrize("dt", [orc.F32, orc.F16, orc.BF16])
@pytest.mark.parametrize("M", [2, 8, 9, 17, 32, 33, 65, 128])
@pytest.mark.parametrize("N,K", [(1, 128), (15, 256), (33, 1152), (4096, 1024), (4099, 384), (8193, 640), (12290, 1152), (16385, 512), (700, 14336), (2050, 1152)])
def test_few_rows_int8(g, dt, M, N, K):
    import torch

    rng = np.random.default_rng(M + N + K)
    a, w = rng.integers(-128, 128, (M, K)).astype(np.int8), rng.integers(-128, 128, (N, K)).astype(np.int8)
    sa, sw = orc.to_storage(rng.uniform(1e-3, 1e-2, M), dt), orc.to_storage(rng.uniform(1e-3, 1e-2, N), dt)
    da, dw, dsa, dsw = g.to_dev(a), g.to_dev(w), g.to_dev(sa, dt), g.to_dev(sw, dt)
    out, acc = g.mynn.quantized_matmul(da, dsa, dw, dsw)
    want = (a.astype(np.float64) @ w.astype(np.float64).T).astype(np.int64)  # (below 2^53: exact)
    assert np.array_equal(acc.cpu().numpy().astype(np.int64), want)
    y = (want.astype(np.float32) * g.f32(sa, dt).reshape(M, 1)) * g.f32(sw, dt).reshape(1, N)
    assert np.array_equal(g.to_host(out).reshape(M, N), orc.to_storage(y, dt).reshape(M, N))
    alone, none = g.mynn.quantized_matmul(da, dsa, dw, dsw, want_acc=False)
    assert none is None and torch.equal(alone, out)


# (row blocks, groups of 8 lhs rows, waves: 20 / (2 blocks + groups) stages of 128 k, 8 at most)
@pytest.mark.parametrize("M,N,K,blocks,groups,waves", [
    (8, 700, 12288, 1, 1, 8), (16, 700, 10240, 1, 2, 8), (32, 700, 6272, 1, 4, 8), (65, 300, 6144, 1, 4, 8), (8, 5700, 8320, 2, 1, 8), (9, 5700, 8320, 2, 2, 8),
    (31, 5700, 8320, 2, 4, 8), (64, 2560, 4096, 2, 4, 8), (3, 8200, 4224, 3, 1, 8), (15, 8200, 4224, 3, 2, 8), (32, 8200, 4224, 3, 4, 8), (8, 12290, 4224, 4, 1, 8),
    (16, 12290, 4224, 4, 2, 8), (5, 16400, 2176, 4, 1, 4), (12, 16400, 2176, 4, 2, 4), (24, 12290, 2176, 2, 4, 4), (32, 16400, 3200, 2, 4, 4)])
def test_rings_in_turn(g, M, N, K, blocks, groups, waves):
    assert K // 128 // waves >= 2 * min(8, 20 // (2 * blocks + groups)) and g.mynn.lib().mynn_few_rows_first(1, M, N, K)
    test_few_rows_int8(g, orc.F16, M, N, K)


# (where K ranges are the faster form a captured call, whose tiles would take them as one, takes the streams)
@pytest.mark.parametrize("M,N,K", [(3, 500, 32768), (32, 1024, 32768), (33, 160, 16384), (128, 1024, 16384)])
def test_captured(g, M, N, K):
    import torch

    assert not g.mynn.lib().mynn_few_rows_first(1, M, N, K)
    rng = np.random.default_rng(M)
    a, w = (g.to_dev(rng.integers(-127, 128, sh).astype(np.int8)) for sh in ((M, K), (N, K)))
    sa, sw = (g.to_dev(orc.to_storage(rng.uniform(1e-3, 1e-2, n), orc.F16), orc.F16) for n in (M, N))
    side, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        got, acc = g.mynn.quantized_matmul(a, sa, w, sw)
    for _ in range(3):
        got.zero_(), acc.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        want, sums = g.mynn.quantized_matmul(a, sa, w, sw)
        assert torch.equal(got, want) and torch.equal(acc, sums)
        a.copy_(torch.roll(a, 1, 0))
