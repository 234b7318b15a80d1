"""K ranges of fewer than 16 rows: K is no multiple of 128, or the streams per wave would take the call, which use no scratch memory.  The tests of
scratch memory, of captured calls and of the tiles at such shapes."""
import ctypes

import numpy as np
import pytest

import oracle as orc
import test_gpu_product_identity
import test_gpu_stream_block
import test_gpu_tile_gemm

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def g():
    import gpu_util

    return gpu_util


def k_ranges(m, M, N, K, kind=1):
    """of the plan of a product of fewer than 16 rows"""
    out = (ctypes.c_long * 6)()
    m.check(m.lib().mynn_tile_gemm_plan(kind, m.F16, M, N, K, ctypes.c_size_t(32 << 20), 0, out, None))
    return out[3]


def calls(g, rng):
    small, large = (test_gpu_stream_block.linear(g, rng, *s) for s in ((6, 256, 8208), (12, 4096, 14352)))
    assert k_ranges(g.mynn, 6, 256, 8208) >= 4 and k_ranges(g.mynn, 12, 4096, 14352) >= 4
    for _ in range(2):  # (the first is passed over by the test of two streams)
        yield "K ranges of few rows", lambda: g.mynn.dequant_matmul(*small), lambda: g.mynn.dequant_matmul(*large)


def test_growth_between_capture_and_replay(g, monkeypatch):
    monkeypatch.setattr(test_gpu_stream_block, "calls", calls)
    test_gpu_stream_block.test_growth_between_capture_and_replay(g)


def test_graphs_on_two_streams(g, monkeypatch):
    monkeypatch.setattr(test_gpu_stream_block, "calls", calls)
    test_gpu_stream_block.test_graphs_of_split_products_on_two_streams(g)


# ... and few weight rows with long rows of whole lines
@pytest.mark.parametrize("dt", [orc.F16, orc.BF16])
@pytest.mark.parametrize("M,N,K", [(6, 4096, 14352), (15, 500, 32768), (2, 500, 49152)])
def test_captured(g, dt, M, N, K):
    assert k_ranges(g.mynn, M, N, K) > 1
    test_gpu_product_identity.test_few_rows_captured(g, dt, M, N, K)


@pytest.mark.parametrize("dt", [orc.F16, orc.BF16])
@pytest.mark.parametrize("M,N,K", [(15, 500, 4112), (15, 33, 20480)])
def test_tiles(g, dt, M, N, K):
    assert k_ranges(g.mynn, M, N, K) > 1
    test_gpu_tile_gemm.test_dequant_matmul_tiles(g, dt, M, N, K)
