"""What the choice of a product's tile promises, without a GPU: the plan of a call that is being captured, the choice against measured times."""
import ctypes as C
import importlib
import os

import pytest

from conftest import ROOT

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


def measured():
    """(kind, dtype, M, N, K, {(tile, ranges): microseconds of those within 15 % of the best}) of profiles/tile_gemm_plans.csv"""
    for line in open(os.path.join(ROOT, "profiles", "tile_gemm_plans.csv")):
        if not line.startswith("#"):
            kind, dtype, M, N, K, _, times = line.strip().split(",")
            yield (dict(W8=W8, W8S=W8S, I8=I8)[kind.split()[0]], dict(f16=mynn.F16, bf16=mynn.BF16)[dtype], int(M), int(N), int(K),
                   {tuple(map(int, t.split("=")[0].split("/"))): float(t.split("=")[1]) for t in times.split()}, kind.endswith("LONG"))


@pytest.mark.parametrize("kind,dtype,mean,late", [(W8, mynn.F16, 1.01, 0.005), (W8, mynn.BF16, 1.01, 0.005), (W8S, mynn.F16, 1.035, 0.03),
                                                  (W8S, mynn.BF16, 1.035, 0.03), (I8, mynn.F16, 1.03, 0.05)])
def test_choice_against_measured_times(kind, dtype, mean, late):
    """The tile and the ranges that the cost model chooses, over matrices of the benchmark's models and others, are on average within `mean` of the best
    (times of one run: they differ by 1 - 2 % from run to run) and 15 % and more behind it in no more than a share `late` of the shapes."""
    over = []
    for k, d, M, N, K, times, long in measured():
        if (k, d) == (kind, dtype):
            scratch = min(32 << 20, max(0, 2 * N * K - 16384)) if kind == W8 else 32 << 20
            tile, _, _, ks, _, _ = plan(k, d, M, N, K, 0 if long else scratch)
            over.append(times.get((tile, ks), 1.15 * min(times.values())) / min(times.values()))
    assert len(over) >= 200
    behind = sum(o >= 1.15 for o in over)
    assert sum(over) / len(over) <= mean and behind <= late * len(over), (sum(over) / len(over), behind, len(over))
