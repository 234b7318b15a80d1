"""RMSNorm and row quantisation with a row's 16-byte pieces in registers (elementwise.hip): rows that end inside a thread's
pieces, at the edges of the forms, one wave and one workgroup per row, against the oracle."""
import numpy as np
import pytest

import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def g():
    import gpu_util

    return gpu_util


@pytest.mark.parametrize("dt", [orc.F16, orc.BF16])
@pytest.mark.parametrize("rows,dim", [(1, 8), (3, 24), (5, 2040), (2, 2048), (3, 2056), (2, 4096), (3, 4104), (2, 8184), (2, 8192), (2, 8200), (3, 14336),
                                      (2, 16384), (2048, 24), (2049, 512), (2050, 520), (2048, 4104), (2048, 6152), (2048, 8192)])
def test_rows_in_registers(g, dt, rows, dim):
    rng = np.random.default_rng(rows + dim)
    x = rng.standard_normal((rows, dim)).astype(np.float32) * 2
    x[0, -1] = 19.0  # the largest of its row is the very last value
    if rows > 1:
        x[-1] = 0.0
    x = orc.to_storage(x, dt)
    w = orc.to_storage(1 + 0.1 * rng.standard_normal(dim), dt)
    got = g.f32(g.to_host(g.mynn.rms_norm(g.to_dev(x, dt), g.to_dev(w, dt), 1e-5)), dt).astype(np.float64)
    xd, wd = g.f32(x, dt).astype(np.float64), g.f32(w, dt).astype(np.float64)
    want = xd / np.sqrt((xd * xd).mean(1, keepdims=True) + 1e-5) * wd
    # one rounding to the type behind f32 arithmetic: a sum of squares in at most 32 + 8 steps, a root, a division, two products
    u = 2.0 ** -8 if dt == orc.BF16 else 2.0 ** -11
    assert (np.abs(got - want) <= (u + 48 * 2.0 ** -24) * np.abs(want) + 2.0 ** -24).all()
    gy, gs, _ = g.mynn.dynamic_quantize_linear(g.to_dev(x, dt), symmetric=True)
    wy, ws = orc.dynquant_i8(x, dt)
    assert np.array_equal(g.to_host(gy), wy) and np.array_equal(g.to_host(gs), ws)
