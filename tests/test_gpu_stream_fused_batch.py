"""Batched decode steps whose attention rotates, appends and attends in one launch, across borders of the key ranges that
several workgroups share (128 rows here), every sequence against its own oracle."""
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


@pytest.mark.parametrize("dt", [orc.F16, orc.BF16])
@pytest.mark.parametrize("kv8", [False, True], ids=["kv16", "kv_int8"])
@pytest.mark.parametrize("B,D,steps", [(2, 64, 260), (5, 128, 132)])
def test_steps_across_key_ranges(g, dt, kv8, B, D, steps):
    cfg, w = llm_weights.synthetic_int8(dict(SMALL, n_layers=1, hidden=256, ffn=384, n_heads=256 // D, n_kv_heads=128 // D if D == 64 else 1, head_dim=D,
                                             max_seq=384), dt, seed=B)
    dec = g.mynn.Decoder(cfg, dev_weights(g, w, dt), batch=B, quant_kv_cache=kv8)
    names = [k[0] for k in dec.profile(np.zeros(B, np.int64), [0], 0, 1)]
    assert any(n.startswith("attention_rope") for n in names)
    refs = [orc.Model(cfg, w) for _ in range(B)]
    for ref in refs:
        ref.set_options(quant_kv_cache=kv8, quantize_activations=False)
    rng = np.random.default_rng(B)
    for i in range(steps):
        toks = rng.integers(0, cfg["vocab"], B)
        wants = [ref.forward([t], [i], i, i + 1, False) for ref, t in zip(refs, toks)]
        _, got = dec.step(toks, [i], i, i + 1, want_logits=True)
        got = got.reshape(B, -1)
        for b in range(B):
            assert max_err_rel_to_max(g.f32(got[b], dt), g.f32(wants[b][0], dt)) <= (2e-2 if kv8 else 1e-2), (i, b)
    dec.close()
