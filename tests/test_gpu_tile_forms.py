"""Every tile of tile_gemm_kernel with every store it is built for, chosen by name: rows and columns that do not fill it, from one K step to
more than it has stages, rows of whole steps and not, in one K range, in several side by side and one after the other."""
import ctypes as C

import pytest

import oracle as orc

pytestmark = pytest.mark.gpu

W8, W8S, I8 = 0, 1, 2  # (kernels.h)
PLAIN, RESIDUAL, PAIRS, PAIRS_EXP = 0, 1, 3, 4
TILES = {W8: [(32, 64), (32, 128), (64, 64), (64, 128), (96, 128), (128, 128), (160, 128), (128, 256), (160, 256)], W8S: [(32, 32), (32, 64), (32, 128)],
         I8: [(32, 64), (64, 64), (64, 128), (64, 128), (128, 128), (128, 256)]}
STEP = {W8: 64, W8S: 64, I8: 128}  # values of K in a step
GRAIN = {W8: 16, W8S: 16, I8: 32}  # K is a multiple of it


@pytest.fixture(scope="module")
def g():
    import gpu_util

    return gpu_util


def product(g, kind, tile, ks, seq, act, W, a_scale, w_scale, T, epi, res=None, want_acc=False):
    import torch

    M, (N, K) = act.shape[0], W.shape
    bm, bn = TILES[kind][tile]
    part = torch.empty((ks * -(-M // bm) * -(-N // bn) * bm * bn,), dtype=torch.float32, device="cuda")
    counters = torch.zeros((4096,), dtype=torch.int32, device="cuda")
    out = torch.full((M, N // 2 if epi in (PAIRS, PAIRS_EXP) else N), float("nan"), dtype=T, device="cuda")
    acc = torch.empty((M, N), dtype=torch.int32, device="cuda") if want_acc else None
    p = lambda t: C.c_void_p(t.data_ptr() if t is not None else None)
    dt = {torch.float16: g.mynn.F16, torch.bfloat16: g.mynn.BF16, torch.float32: g.mynn.F32}[T]
    g.mynn.check(g.mynn.lib().mynn_tile_gemm(kind, tile, ks, seq, p(out), p(acc), p(act), p(W), p(a_scale), p(w_scale), p(res), M, N, K, dt, epi, p(part),
                                             C.c_size_t(part.numel() * 4), p(counters), C.c_void_p(torch.cuda.current_stream().cuda_stream)))
    assert not counters.any()
    return out, acc


def sizes(kind, tile):
    """(M, N, K, K ranges)"""
    (bm, bn), step, grain = TILES[kind][tile], STEP[kind], GRAIN[kind]
    for M, N in ((bm + 1, 2 * bn - 6), (bm - 1, bn + 2), (2 * bm + 7, bn)):
        for steps in (1, 2, 3, 4, 6, 9, 14):
            for K in (step * steps, step * (steps - 1) + grain, step * steps - grain):
                for ks in (1, 2, 3):
                    if ks == 1 or (steps >= 3 * ks and M == bm + 1):
                        yield M, N, K, ks


@pytest.mark.parametrize("T", ["float16", "bfloat16"])
@pytest.mark.parametrize("kind,tile", [(W8, t) for t in range(9)] + [(W8S, t) for t in range(3)])
def test_tiles_of_int8_weights(g, T, kind, tile):
    import torch

    T = getattr(torch, T)
    u = 2.0 ** -8 if T == torch.bfloat16 else 2.0 ** -11
    gen = torch.Generator(device="cuda").manual_seed(tile)
    for M, N, K, ks in sizes(kind, tile):
        act = torch.randn((M, K), generator=gen, device="cuda").to(T)
        W = torch.randint(-127, 128, (N, K), generator=gen, dtype=torch.int8, device="cuda")
        sc = (torch.rand((N,), generator=gen, device="cuda") * 9e-3 + 1e-3).to(T)
        wt = (W.float() * sc.float()[:, None]).to(T).double() if kind == W8 else W.double() * sc.double()[:, None]
        wt = wt.T.contiguous()
        sums = act.double() @ wt
        # a sum of K products in f32, in any order
        off = (K / 16 + 16 + 16 * ks) * 2.0 ** -24 * (act.double().abs() @ wt.abs())
        case = (M, N, K, ks)
        out, _ = product(g, kind, tile, ks, 0, act, W, None, sc, T, PLAIN)
        assert ((out.double() - sums).abs() <= u * sums.abs() + off).all(), case
        if ks > 1 and TILES[kind][tile][0] * TILES[kind][tile][1] <= 128 * 128:
            assert torch.equal(product(g, kind, tile, ks, 1, act, W, None, sc, T, PLAIN)[0], out), case
        if kind == W8S:
            continue
        res = torch.randn((M, N), generator=gen, device="cuda").to(T)
        out, _ = product(g, kind, tile, ks, 0, act, W, None, sc, T, RESIDUAL, res)
        want = res.double() + sums
        assert ((out.double() - want).abs() <= u * want.abs() * (1 + u) + (1 + u) * (u * sums.abs() + off)).all(), case
        gate, up, goff, uoff = sums[:, ::2], sums[:, 1::2], (u * sums.abs() + off)[:, ::2], (u * sums.abs() + off)[:, 1::2]
        swish = gate * torch.sigmoid(gate)
        want = swish * up
        # (the derivative of swish is at most 1.1; exponential, reciprocal and products in f32: 2^-20 of the result)
        bound = 1.1 * (up.abs() + uoff) * goff + swish.abs() * uoff + (u + 2.0 ** -20) * (want.abs() + 1.1 * (up.abs() + uoff) * goff + swish.abs() * uoff)
        bound = bound + 2.0 ** -24  # (values below the normal numbers of fp16)
        for epi in (PAIRS, PAIRS_EXP):
            out, _ = product(g, kind, tile, ks, 0, act, W, None, sc, T, epi)
            assert ((out.double() - want).abs() <= bound).all(), (case, epi)


@pytest.mark.parametrize("T", ["float16", "bfloat16", "float32"])
@pytest.mark.parametrize("tile", range(6))
def test_tiles_of_int8_products(g, T, tile):
    import torch

    T = getattr(torch, T)
    u = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -24}[T]
    gen = torch.Generator(device="cuda").manual_seed(tile)
    for M, N, K, ks in sizes(I8, tile):
        lhs = torch.randint(-128, 128, (M, K), generator=gen, dtype=torch.int8, device="cuda")
        rhs = torch.randint(-128, 128, (N, K), generator=gen, dtype=torch.int8, device="cuda")
        ls, rs = [(torch.rand((n,), generator=gen, device="cuda") * 9e-4 + 1e-4).to(T) for n in (M, N)]
        sums = (lhs.double() @ rhs.double().T.contiguous())  # (whole numbers below 2^53)
        plain = ((sums.float() * ls.float()[:, None]) * rs.float()).to(T)
        case = (M, N, K, ks)
        for want_acc in (False, True):
            out, acc = product(g, I8, tile, ks, 0, lhs, rhs, ls, rs, T, PLAIN, want_acc=want_acc)
            assert torch.equal(out, plain), case
            if want_acc:
                assert torch.equal(acc.double(), sums), case
        if T == torch.float32:
            continue
        res = torch.randn((M, N), generator=gen, device="cuda").to(T)
        out, _ = product(g, I8, tile, ks, 0, lhs, rhs, ls, rs, T, RESIDUAL, res)
        assert torch.equal(out, (res.float() + plain.float()).to(T)), case
        out, _ = product(g, I8, tile, ks, 0, lhs, rhs, ls, rs, T, PAIRS_EXP)
        gate, up = plain[:, ::2].double(), plain[:, 1::2].double()
        want = gate * torch.sigmoid(gate) * up
        assert ((out.double() - want).abs() <= (u + 2.0 ** -20) * want.abs() + 2.0 ** -24).all(), case
