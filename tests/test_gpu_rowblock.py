"""Decode batches whose linears are one launch each (rowblock.hip): K ranges that do not divide evenly over the waves, half a
row block to two per workgroup, with the norm inside (up to 16 rows) and in front, two to four tiles of rows, against the oracle."""
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
@pytest.mark.parametrize("B", [2, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("hidden,ffn", [(256, 384), (1152, 5120), (2176, 768), (2176, 5120), (256, 8320)])
def test_decode_batches_one_launch_per_linear(g, dt, B, hidden, ffn):
    # (ffn 5120: the gate/up rows are 320 row blocks, one and a half or two per workgroup; hidden 2176: 17 K steps; 8320:
    # one slab of activations per panel)
    cfg, w = llm_weights.synthetic_int8(dict(SMALL, n_layers=1, hidden=hidden, ffn=ffn, n_heads=hidden // 64, n_kv_heads=hidden // 128, head_dim=64), dt, seed=B)
    dec = g.mynn.Decoder(cfg, dev_weights(g, w, dt), batch=B)
    names = [k[0] for k in dec.profile(np.zeros(B, np.int64), [0], 0, 1)]
    if B <= 32:  # (more rows: the final norm may ride in the down projection's second launch)
        assert names.count("rms_norm") == (0 if B <= 16 else 3) and "attention_rope_append" in names
    rng = np.random.default_rng(B)
    refs = {b: orc.Model(cfg, w) for b in (0, B // 2, B - 1)}
    for step in range(3):
        toks = rng.integers(0, cfg["vocab"], B)
        _, got = dec.step(toks, [step], step, step + 1, want_logits=True)
        got = got.reshape(B, -1)
        for b, ref in refs.items():
            want = ref.forward([toks[b]], [step], step, step + 1, False)
            assert max_err_rel_to_max(g.f32(got[b], dt), g.f32(want[0], dt)) <= 1e-2, (step, b)
    dec.close()
