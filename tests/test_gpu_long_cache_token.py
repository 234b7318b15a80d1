"""Batch-1 decode over a cache too long for the single-launch layer, contiguous or in pages, with and without projection biases: the lm_head launch finds the greedy token and moves the loop state on.
Its give-up (forced by a spin limit of none; every kernel ends normally) leaves the executor with launches of their own and the same results."""
import numpy as np
import pytest

import llm_weights
import oracle as orc
from conftest import max_err_rel_to_max
from test_gpu_decoder import SMALL_D64, dev_weights

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def g():
    import gpu_util

    return gpu_util


@pytest.mark.parametrize("kv8", [False, True], ids=["kv16", "kv_int8"])
@pytest.mark.parametrize("dt", [orc.F16, orc.BF16])
def test_token_inside_the_lm_head_launch(g, dt, kv8):
    cfg, w = llm_weights.synthetic_int8(dict(SMALL_D64, max_seq=8192), dt, seed=17)
    dw, L = dev_weights(g, w, dt), cfg["n_layers"]
    dec, quick = (g.mynn.Decoder(cfg, dw, quant_kv_cache=kv8, **kw) for kw in ({}, dict(handover_spin_limit=-1)))
    assert dec.stats()["launches_per_step"] == quick.stats()["launches_per_step"] == 5 * L + 2 and dec.stats()["graph"]
    toks = np.random.default_rng(3).integers(0, cfg["vocab"], 6)
    for i, t in enumerate(toks):
        a, la = dec.step([t], [i], i, i + 1, want_logits=True)
        b, lb = quick.step([t], [i], i, i + 1, want_logits=True)
        assert a[0] == orc.argmax_last(la[0], dt) and a == b and np.array_equal(la, lb), i
    assert dec.handover_failures == 0 and quick.handover_failures == 1 and quick.stats()["launches_per_step"] > 5 * L + 2
    # the device loop, more steps than one of its graphs holds, against single steps
    n, t = 40, int(toks[0])
    got = list(dec.decode_loop(t, 0, n))
    want = []
    for i in range(n):
        a, _ = quick.step([t], [i], i, i + 1)
        t = int(a[0])
        want.append(t)
    assert got == want
    dec.close(), quick.close()


# (the same launch behind pages and behind a biased projection)
@pytest.mark.parametrize("dt", [orc.F16, orc.BF16])
@pytest.mark.parametrize("paged,bias", [(True, False), (False, True), (True, True)], ids=["paged", "bias", "bias_paged"])
def test_token_of_paged_and_biased_executors(g, dt, paged, bias):
    import torch

    cfg, w = llm_weights.synthetic_int8(dict(SMALL_D64, max_seq=8192), dt, seed=19)
    if bias:
        w = llm_weights.add_qkv_bias(cfg, w, dt, seed=20, std=0.05)
    dw = dev_weights(g, w, dt)

    def make(**kw):
        if paged:
            pool = g.mynn.KvPool(32, 256)
            kw.update(kv=pool.buffers(cfg["n_layers"], cfg["n_kv_heads"], 64, {orc.F16: torch.float16, orc.BF16: torch.bfloat16}[dt]),
                      kv_pages=g.mynn.KvPages(pool, 1, 8192))
        return g.mynn.Decoder(cfg, dw, **kw)

    dec, quick, ref = make(), make(handover_spin_limit=-1), orc.Model(cfg, w)
    names = [k[0] for k in dec.profile([1], [0], 0, 1)]
    assert any(n.startswith("attention_rope") for n in names) and not any("argmax_p" in n for n in names), names
    toks = np.random.default_rng(4).integers(0, cfg["vocab"], 6)
    for i, t in enumerate(toks):
        want = ref.forward([t], [i], i, i + 1, False)
        a, la = dec.step([t], [i], i, i + 1, want_logits=True)
        b, lb = quick.step([t], [i], i, i + 1, want_logits=True)
        assert max_err_rel_to_max(g.f32(la, dt), g.f32(want, dt)) <= (1e-2 if dt == orc.F16 else 13 * 2.0 ** -9), i
        assert a[0] == orc.argmax_last(la[0], dt) and a == b and np.array_equal(la, lb), i
    assert dec.handover_failures == 0 and quick.handover_failures == 1
    n, t = 40, int(toks[0])
    got, want = list(dec.decode_loop(t, 0, n)), []
    for i in range(n):
        a, _ = quick.step([t], [i], i, i + 1)
        t = int(a[0])
        want.append(t)
    assert got == want
    dec.close(), quick.close()
