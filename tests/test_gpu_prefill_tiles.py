"""Prefill executors of 65 and more rows, whose linears multiply by tiles of the int8 weights with the residual and SwiGLU stores, against the
oracle: row counts that fill no tile, K ranges in the executor's own memory, two chunks behind each other."""
import ctypes as C

import numpy as np
import pytest

import llm_weights
import oracle as orc
from conftest import max_err_rel_to_max
from test_gpu_decoder import SMALL, dev_weights

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def g():
    import gpu_util

    return gpu_util


def rows_of_tile(g, dt, M, N, K):
    plan = (C.c_long * 6)()
    g.mynn.check(g.mynn.lib().mynn_tile_gemm_plan(0, dt, M, N, K, C.c_size_t(32 << 20), 0, plan, None))
    return plan[1]


@pytest.mark.parametrize("dt", [orc.F16, orc.BF16])
@pytest.mark.parametrize("S,hidden,ffn", [(128, 768, 1600), (129, 256, 9040), (300, 768, 4096), (97, 512, 11264)])
def test_prefill_by_tiles_of_int8_weights(g, dt, S, hidden, ffn):
    cfg, w = llm_weights.synthetic_int8(dict(SMALL, n_layers=1, hidden=hidden, ffn=ffn, n_heads=hidden // 64, n_kv_heads=2, head_dim=64, vocab=1000, max_seq=2 * S), dt, seed=S)
    if ffn in (4096, 11264):
        assert rows_of_tile(g, dt, S, 2 * ffn, hidden) >= 96  # (the loop of the wide tiles, with the SwiGLU store)
    ref = orc.Model(cfg, w)
    ref.set_gemm_mode(2)
    dec = g.mynn.Decoder(cfg, dev_weights(g, w, dt), seq_q=S)
    names = [k[0] for k in dec.profile(np.zeros(S, np.int64), np.arange(S), 0, S)]
    assert "linear_gateup_swiglu" in names and "swiglu" not in names, names
    rng = np.random.default_rng(S)
    for past in (0, S):
        ids, pos = rng.integers(0, cfg["vocab"], S), np.arange(past, past + S)
        want = ref.forward(ids, pos, past, past + S, True)
        _, got = dec.step(ids, pos, past, past + S, want_logits=True)
        assert max_err_rel_to_max(g.f32(got, dt), g.f32(want, dt)) <= 1e-2, past
    k_ref, v_ref = ref.kv_cache(0)
    k_gpu, v_gpu = g.to_host(dec.kv[0][0])[0], g.to_host(dec.kv[0][1])[0]
    assert max_err_rel_to_max(g.f32(k_gpu[:, : 2 * S], dt), g.f32(k_ref[:, : 2 * S], dt)) <= 1e-2
    assert max_err_rel_to_max(g.f32(v_gpu[:, : 2 * S], dt), g.f32(v_ref[:, : 2 * S], dt)) <= 1e-2
    dec.close()
