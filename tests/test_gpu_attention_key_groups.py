"""Prefill attention whose key tiles are dealt to groups of waves, and over an int8 cache: rows at the edges of key tiles,
query blocks and of the rule that picks the split, against the oracle."""
import numpy as np
import pytest

import oracle as orc
from conftest import max_err_rel_to_max

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def g():
    import gpu_util

    return gpu_util


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("B,Hq,Hkv,S,past,causal", [(1, 2, 1, 64, 0, True), (1, 2, 1, 65, 0, True), (2, 3, 3, 129, 0, True), (1, 8, 2, 128, 70, True),
                                                    (1, 40, 4, 513, 0, True), (1, 41, 41, 513, 0, True), (1, 4, 1, 100, 1, False), (1, 32, 8, 2000, 0, True)])
def test_key_groups(g, D, B, Hq, Hkv, S, past, causal):
    dt = orc.F16 if (S + D) % 2 else orc.BF16
    rng = np.random.default_rng(S * 7 + D)
    L, active = past + S + 3, past + S
    q = orc.to_storage(rng.standard_normal((B, Hq, S, D)), dt)
    k = orc.to_storage(rng.standard_normal((B, Hkv, L, D)), dt)
    v = orc.to_storage(rng.standard_normal((B, Hkv, L, D)), dt)
    k[:, :, active:] = v[:, :, active:] = orc.to_storage(np.full(1, np.nan), dt)  # (never to be read into a result)
    want = orc.attention(q, k, v, dt, D ** -0.5, causal, active)
    got = g.to_host(g.mynn.attention(g.to_dev(q, dt), g.to_dev(k, dt), g.to_dev(v, dt), D ** -0.5, causal, active))
    assert max_err_rel_to_max(g.f32(got, dt), g.f32(want, dt)) <= 1e-2


@pytest.mark.parametrize("dt", [orc.F16, orc.BF16])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("S,past,causal,v_size", [(16, 300, True, 1.0), (64, 64, True, 1.0), (65, 63, True, 6e4), (130, 200, True, 1e-4), (97, 0, False, 1.0)])
def test_int8_cache(g, dt, D, S, past, causal, v_size):
    """v_size: values at both ends of the type (their scales enter the weights of the second product)."""
    rng = np.random.default_rng(S * 11 + D)  # (16 rows take this kernel behind a past of 256 rows or more)
    B, Hq, Hkv, active = 3, 32, 8, past + S
    q = orc.to_storage(rng.standard_normal((B, Hq, S, D)), dt)
    k = orc.to_storage(rng.standard_normal((B, Hkv, active, D)), dt)
    size = v_size * np.exp2(-rng.integers(0, 10, (B, Hkv, active, 1)) * (v_size > 1))  # (rows of very different scales)
    v = orc.to_storage(rng.uniform(-1, 1, (B, Hkv, active, D)) * size, dt)
    kq, vq = np.zeros(k.shape, np.int8), np.zeros(v.shape, np.int8)
    ks, vs = orc.to_storage(np.zeros(k.shape[:3]), dt), orc.to_storage(np.zeros(v.shape[:3]), dt)
    orc.quantizing_kv_cache_update(kq, ks, k, 0, dt)
    orc.quantizing_kv_cache_update(vq, vs, v, 0, dt)
    want = orc.attention(q, kq, vq, dt, D ** -0.5, causal, active, ks, vs)
    got = g.to_host(g.mynn.attention(g.to_dev(q, dt), g.to_dev(kq), g.to_dev(vq), D ** -0.5, causal, active,
                                     k_scale=g.to_dev(ks, dt), v_scale=g.to_dev(vs, dt)))
    assert np.isfinite(g.f32(want, dt)).all()
    assert max_err_rel_to_max(g.f32(got, dt), g.f32(want, dt)) <= 1e-2
