"""QuantizedMatMul into an output that is not 16-byte aligned: the tiles of every size store it element by element, and
nothing around it."""
import numpy as np
import pytest

import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def g():
    import gpu_util

    return gpu_util


@pytest.mark.parametrize("dt", [orc.F16, orc.BF16, orc.F32])
@pytest.mark.parametrize("M,N,K", [(2, 40, 64), (3, 40, 64), (33, 64, 128), (97, 200, 8192), (130, 257, 2048), (2048, 4096, 128)])
@pytest.mark.parametrize("shift", [1, 3, 4])
def test_shifted_output(g, dt, M, N, K, shift):
    import torch

    rng = np.random.default_rng(M + N + K)
    lhs, rhs = rng.integers(-128, 128, (M, K)).astype(np.int8), rng.integers(-128, 128, (N, K)).astype(np.int8)
    ls, rs = orc.to_storage(rng.uniform(1e-3, 1e-2, M), dt), orc.to_storage(rng.uniform(1e-3, 1e-2, N), dt)
    args = [g.to_dev(lhs), g.to_dev(ls, dt), g.to_dev(rhs), g.to_dev(rs, dt)]
    want = g.mynn.quantized_matmul(*args, want_acc=False)[0]
    if M * N * K < 1 << 26:
        assert np.array_equal(g.to_host(want), orc.quantized_matmul(lhs, ls, rhs, rs, dt)[0])
    flat = torch.full((M * N + 16,), 7.0, dtype=want.dtype, device="cuda")
    out = flat[shift:shift + M * N]
    p = [t.data_ptr() for t in args]
    g.mynn.check(g.mynn.lib().mynn_quantized_matmul(out.data_ptr(), None, p[0], p[1], p[2], p[3], M, N, K, dt, torch.cuda.current_stream().cuda_stream))
    assert torch.equal(out.view(M, N), want)
    assert (flat[:shift] == 7).all() and (flat[shift + M * N:] == 7).all()
