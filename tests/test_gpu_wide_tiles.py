"""int8-weight products of 97 and more rows by the tiles and ranges that their sizes choose: rows and columns that do not fill a tile, few K
steps, rows that are not whole steps; captured, where a smaller tile may take the ranges one after the other, the same bits.  (Every tile by
name: test_gpu_tile_forms.py.)"""
import pytest

import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def g():
    import gpu_util

    return gpu_util


@pytest.mark.parametrize("dt", [orc.F16, orc.BF16])
@pytest.mark.parametrize("M,N,K", [
    (97, 11264, 2048), (129, 11250, 1040), (168, 6469, 5792), (200, 5000, 8208), (1000, 4096, 4096), (127, 28672, 4096), (300, 11264, 2048),
    (319, 11001, 1040), (300, 4096, 14336), (481, 11250, 528), (500, 11264, 2048), (321, 15000, 272), (640, 15000, 144), (639, 15001, 80),
    (700, 11264, 2048), (640, 15000, 16), (257, 9001, 272), (160, 4090, 14352),
])
def test_wide_tiles(g, dt, M, N, K):
    import torch

    T = g.torch_dtype(dt)
    gen = torch.Generator(device="cuda").manual_seed(M + N + K)
    act = torch.randn((M, K), generator=gen, device="cuda").to(T)
    W = torch.randint(-127, 128, (N, K), generator=gen, dtype=torch.int8, device="cuda")
    sc = (torch.rand((N,), generator=gen, device="cuda") * 9e-3 + 1e-3).to(T)
    got = g.mynn.dequant_matmul(act, W, sc)
    wt = (W.float() * sc.float()[:, None]).to(T).double()  # (one rounding: the product of an int8 and a 16-bit number is exact in f32)
    want = act.double() @ wt.T.contiguous()
    # the sum of K products in f32 (any order: K * 2^-24 of the sum of their magnitudes, K / 16 of it where 16 are added at once), rounded to T
    size = act.double().abs() @ wt.T.abs().contiguous()
    u = 2.0 ** -8 if dt == orc.BF16 else 2.0 ** -11
    assert ((got.double() - want).abs() <= u * want.abs() + (K / 16 + 16) * 2.0 ** -24 * size).all()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            out = g.mynn.dequant_matmul(act, W, sc)
    for _ in range(2):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, got)
