"""GEMV over rows of more than 4096 values, whose 1024-value chunks go through a ring of places: rows that end at, just past and just
before a chunk and a change of form, odd numbers of rows, and more rows than the waves take at once; against the sums in 64 bits."""
import numpy as np
import pytest

import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def g():
    import gpu_util

    return gpu_util


@pytest.mark.parametrize("dt", [orc.F16, orc.BF16])
@pytest.mark.parametrize("N", [1, 37, 8195])
@pytest.mark.parametrize("K", [4096, 4112, 5136, 6144, 6160, 8176, 8192, 8208, 9600, 14320, 14336, 14352])
def test_long_rows(g, dt, N, K):
    rng = np.random.default_rng(N + K)
    act = orc.to_storage(rng.standard_normal((1, K)), dt)
    W = rng.integers(-127, 128, (N, K)).astype(np.int8)
    sc = orc.to_storage(rng.uniform(1e-3, 1e-2, N), dt)
    got = g.f32(g.to_host(g.mynn.dequant_gemv(g.to_dev(act, dt), g.to_dev(W), g.to_dev(sc, dt))), dt)
    a, s = g.f32(act, dt)[0], g.f32(sc, dt)
    exact = (W.astype(np.float32) @ a.astype(np.float64)) * s
    # the bound of test_gpu_ops.py: K * 2^-24 of the sum of magnitudes, and one rounding of the stored value
    bound = (np.abs(W).astype(np.float32) @ np.abs(a).astype(np.float64)) * s * K * 2.0 ** -24
    assert np.all(np.abs(got.reshape(-1) - exact) <= bound + np.abs(exact) * (2.0 ** -8 if dt == orc.BF16 else 2.0 ** -10))
