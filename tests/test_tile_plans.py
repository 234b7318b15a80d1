"""What the choice of a product's tile promises, without a GPU: the plan of a call that is being captured."""
import ctypes as C
import importlib

import pytest

mynn = importlib.import_module("my-nn-engine_amd")

W8, W8S, I8 = 0, 1, 2  # (kernels.h)


def plan(kind, dtype, M, N, K, scratch=32 << 20, seq_ks=0):
    """(tile, rows, columns, K ranges, one after the other, bytes of partial sums)"""
    out = (C.c_long * 6)()
    mynn.check(mynn.lib().mynn_tile_gemm_plan(kind, dtype, M, N, K, C.c_size_t(scratch), seq_ks, out, None))
    return tuple(out)


@pytest.mark.parametrize("N,K", [(28672, 4096), (11264, 2048), (4096, 14336), (5476, 7456)])
@pytest.mark.parametrize("M", [97, 300, 500, 1000, 2000])
def test_captured_int8_product_takes_the_best_tile_for_one_range(M, N, K):
    """(one range needs one set of sums in the registers whatever the tile)"""
    assert plan(I8, mynn.F16, M, N, K, seq_ks=4) == plan(I8, mynn.F16, M, N, K, scratch=0)


@pytest.mark.parametrize("dtype", [mynn.F16, mynn.BF16])
@pytest.mark.parametrize("M,N,K", [(97, 4096, 4096), (300, 4096, 14336), (1000, 4096, 14336)])
def test_captured_product_of_several_ranges_fits_the_registers(dtype, M, N, K):
    tile, rows, columns, ks, seq, part = plan(W8, dtype, M, N, K, seq_ks=3)
    assert ks == 3 and seq == 1 and rows * columns <= 128 * 128
