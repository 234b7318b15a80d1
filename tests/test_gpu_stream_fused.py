"""Decode executors over a cache too long for the short attention form: RoPE, both appends, the attention and the merge of
its key ranges are one launch.  Steps across a border of key ranges against the oracle, and bit for bit against the same
executor over pages."""
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
@pytest.mark.parametrize("D", [64, 128])
def test_long_cache_decode_is_one_attention_launch(g, dt, kv8, D):
    import torch

    cfg, w = llm_weights.synthetic_int8(dict(SMALL, n_layers=1, n_heads=256 // D, n_kv_heads=128 // D if D == 64 else 1, head_dim=D,
                                             max_seq=8192), dt, seed=D)
    dw = dev_weights(g, w, dt)
    dec = g.mynn.Decoder(cfg, dw, quant_kv_cache=kv8)
    pool = g.mynn.KvPool(32, 256)
    kv = pool.buffers(1, cfg["n_kv_heads"], D, {orc.F16: torch.float16, orc.BF16: torch.bfloat16}[dt], kv_int8=kv8)
    paged = g.mynn.Decoder(cfg, dw, quant_kv_cache=kv8, kv=kv, kv_pages=g.mynn.KvPages(pool, 1, 8192))
    names = [k[0] for k in dec.profile([1], [0], 0, 1)]
    assert any(n.startswith("attention_rope") for n in names) and not any("kv_append" in n for n in names)
    ref = orc.Model(cfg, w)
    ref.set_options(quant_kv_cache=kv8, quantize_activations=False)
    rng = np.random.default_rng(D)
    for i in range(133):  # (key ranges are 128 rows: rows 127, 128 and 129 end, begin and continue one)
        t = int(rng.integers(0, cfg["vocab"]))
        want = ref.forward([t], [i], i, i + 1, False)
        nxt, got = dec.step([t], [i], i, i + 1, want_logits=True)
        pnxt, pgot = paged.step([t], [i], i, i + 1, want_logits=True)
        assert max_err_rel_to_max(g.f32(got, dt), g.f32(want, dt)) <= (2e-2 if kv8 else 1e-2), i
        assert np.array_equal(got, pgot) and list(nxt) == list(pnxt), i
    dec.close(), paged.close()
