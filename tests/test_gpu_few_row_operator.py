"""DequantMatMul of 2 .. 15 rows over whole 128-byte lines of row-major weights (rowblock.hip): one to eight and nine to fifteen rows, fewer
weight rows than a block, ragged blocks of every workgroup form, K of fewer steps than waves, of one more than they share evenly and of
twice the stages of the rings and more for each wave; outputs and operands at odd places; against the sums in 64 bits, the same bits from
the workspace form and from a captured call."""
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


def operands(g, M, N, K, dt):
    """activations, weights, scales, the sums in 64 bits, and what f32 sums of K exact products in any order and one rounding of the stored
    value may be off"""
    rng = np.random.default_rng(M + N + K)
    act, sc = orc.to_storage(rng.standard_normal((M, K)), dt), orc.to_storage(rng.uniform(1e-3, 1e-2, N), dt)
    W = rng.integers(-128, 128, (N, K)).astype(np.int8)
    a, s, w = g.f32(act, dt).astype(np.float64).reshape(M, K), g.f32(sc, dt).astype(np.float64), W.astype(np.float64)
    exact = (a @ w.T) * s
    return act, W, sc, exact, (np.abs(a) @ np.abs(w).T) * s * K * 2.0 ** -24 + np.abs(exact) * (2.0 ** -8 if dt == orc.BF16 else 2.0 ** -11) * 1.01 + 1e-30


# (1, 2 and 3 row blocks and eight waves, 2 and 4 and four waves: a ring has up to 5, 3, 2, 3 and 2 stages of 128 k)
@pytest.mark.parametrize("dt", [orc.F16, orc.BF16])
@pytest.mark.parametrize("M", [5, 15])
@pytest.mark.parametrize("N,K,waves,stages", [(75, 10368, 8, 5), (4099, 6400, 8, 3), (8193, 4224, 8, 2), (12290, 3200, 4, 3), (16400, 2176, 4, 2)])
def test_rings_in_turn(g, dt, M, N, K, waves, stages):
    assert K // 128 // waves >= 2 * stages and g.mynn.lib().mynn_few_rows_first(0, M, N, K)
    act, W, sc, exact, bound = operands(g, M, N, K, dt)
    got = g.mynn.dequant_matmul(g.to_dev(act, dt), g.to_dev(W), g.to_dev(sc, dt))
    assert np.all(np.abs(g.f32(g.to_host(got), dt).reshape(M, N) - exact) <= bound)


# (an output or scales at any element take the same kernel: the same bits; activations or weights that are not 16-byte aligned another one)
@pytest.mark.parametrize("dt", [orc.F16, orc.BF16])
@pytest.mark.parametrize("M,N,K", [(2, 33, 1152), (9, 4099, 384)])
def test_odd_places(g, dt, M, N, K):
    import torch

    act, W, sc, exact, bound = operands(g, M, N, K, dt)
    ops = [g.to_dev(act, dt), g.to_dev(W), g.to_dev(sc, dt)]
    want = g.mynn.dequant_matmul(*ops)

    def run(shifts):  # elements of activations, weights, scales, output
        placed = []
        for t, n in zip(ops, shifts):
            flat = torch.empty(t.numel() + 16, dtype=t.dtype, device="cuda")
            placed.append(flat[n:n + t.numel()])
            placed[-1].copy_(t.reshape(-1))
        flat = torch.full((M * N + 16,), 7.0, dtype=want.dtype, device="cuda")
        out = flat[shifts[3]:shifts[3] + M * N]
        a, w, s = (t.data_ptr() for t in placed)
        g.mynn.check(g.mynn.lib().mynn_dequant_matmul(out.data_ptr(), a, w, s, M, N, K, dt, dt, torch.cuda.current_stream().cuda_stream))
        torch.cuda.synchronize()
        assert (flat[:shifts[3]] == 7).all() and (flat[shifts[3] + M * N:] == 7).all()
        return out.view(M, N)

    for shifts in ((0, 0, 0, 1), (0, 0, 1, 0), (0, 0, 3, 5)):
        assert torch.equal(run(shifts), want), shifts
    for shifts in ((4, 0, 0, 0), (0, 8, 0, 0), (4, 8, 1, 1)):
        assert np.all(np.abs(g.f32(g.to_host(run(shifts).contiguous()), dt).reshape(M, N) - exact) <= bound), shifts


# Few weight rows with long rows, which K ranges do faster: with a caller's workspace (there is none for fewer than 16 rows) and for an output that the
# tiles refuse it is the streams all the same, whose sums do not depend on how many weight rows there are
@pytest.mark.parametrize("dt", [orc.F16, orc.BF16])
@pytest.mark.parametrize("M", [2, 15])
def test_streams_where_k_ranges_cannot_be(g, dt, M):
    import torch

    N, wide, K = 500, 3100, 49152
    first = g.mynn.lib().mynn_few_rows_first
    assert first(0, M, wide, K) and not first(0, M, N, K)
    gen = torch.Generator(device="cuda").manual_seed(M)
    tdt = torch.float16 if dt == orc.F16 else torch.bfloat16
    act = torch.randn((M, K), generator=gen, device="cuda").to(tdt)
    w = torch.randint(-128, 128, (wide, K), generator=gen, device="cuda").to(torch.int8)
    sc = (torch.rand((wide,), generator=gen, device="cuda") * 1e-3 + 1e-3).to(tdt)
    want = g.mynn.dequant_matmul(act, w, sc)[:, :N]
    assert torch.equal(g.mynn.dequant_matmul_ws(act, w[:N], sc[:N]), want)
    flat = torch.full((M * N + 16,), 7.0, dtype=tdt, device="cuda")
    g.mynn.check(g.mynn.lib().mynn_dequant_matmul(flat.data_ptr() + 2, act.data_ptr(), w.data_ptr(), sc.data_ptr(), M, N, K, dt, dt,
                                                  torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    assert flat[0] == 7 and (flat[1 + M * N:] == 7).all()
    assert torch.equal(flat[1:1 + M * N].view(M, N), want)
