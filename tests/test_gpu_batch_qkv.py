"""Decode steps of 17 to 64 sequences whose o or down product goes over K ranges: q|k|v are one launch, RoPE and the cache appends (with the
quantiser of an int8 cache) ride on the attention.  16-bit and int8 caches, contiguous and in pages, with and without projection biases,
across the border of a key range; against the oracle."""
import numpy as np
import pytest

import llm_weights
import oracle as orc
from conftest import max_err_rel_to_max
from test_gpu_decoder import SMALL, dev_weights

pytestmark = pytest.mark.gpu

# 12416 x 1024 weights of the down projection: more than 12 million, so that more than 16 rows take K ranges for it
SHAPE = dict(SMALL, n_layers=1, hidden=1024, ffn=12416, vocab=300, n_heads=16, n_kv_heads=4, head_dim=64, max_seq=384)


@pytest.fixture(scope="module")
def g():
    import gpu_util

    return gpu_util


@pytest.fixture(scope="module")
def model():
    made = {}

    def get(dt, bias):
        if dt not in made:
            made[dt] = llm_weights.synthetic_int8(SHAPE, dt, seed=5)
        cfg, w = made[dt]
        return cfg, llm_weights.add_qkv_bias(cfg, w, dt, seed=6, std=0.05) if bias else w

    return get


# (17 sequences: three key ranges of 128 rows; rows 127, 128 and 129 end, begin and continue one)
@pytest.mark.parametrize("dt", [orc.F16, orc.BF16])
@pytest.mark.parametrize("kv8,paged,bias", [(0, 0, 0), (1, 0, 0), (0, 1, 0), (1, 1, 0), (0, 0, 1), (1, 1, 1)],
                         ids=["kv16", "kv_int8", "paged", "paged_int8", "bias", "bias_paged_int8"])
@pytest.mark.parametrize("B,steps", [(17, 130), (48, 3), (64, 3)])
def test_batched_steps(g, model, dt, kv8, paged, bias, B, steps):
    import torch

    cfg, w = model(dt, bias)
    kw = {}
    if paged:
        pool = g.mynn.KvPool(B * 3, 128)
        kw = dict(kv=pool.buffers(1, cfg["n_kv_heads"], 64, {orc.F16: torch.float16, orc.BF16: torch.bfloat16}[dt], kv_int8=bool(kv8)),
                  kv_pages=g.mynn.KvPages(pool, B, 384))
    dec = g.mynn.Decoder(cfg, dev_weights(g, w, dt), batch=B, quant_kv_cache=bool(kv8), **kw)
    names = [k[0] for k in dec.profile(np.zeros(B, np.int64), [0], 0, 1)]
    assert "linear_qkv" in names and any(n.startswith("attention_rope") for n in names), names
    assert not any(n.startswith("kv_append") or n == "linear_qkv_reduce" for n in names), names
    follow = sorted({B - 1} if steps > 3 else {0, B // 2, B - 1})
    refs = {b: orc.Model(cfg, w) for b in follow}
    for ref in refs.values():
        ref.set_options(quant_kv_cache=bool(kv8), quantize_activations=False)
    rng = np.random.default_rng(B)
    for i in range(steps):
        toks = rng.integers(0, cfg["vocab"], B)
        _, got = dec.step(toks, [i], i, i + 1, want_logits=True)
        got = got.reshape(B, -1)
        for b, ref in refs.items():
            want = ref.forward([toks[b]], [i], i, i + 1, False)
            # 13 stored values lie between a token and its logits, each up to half a unit of its type off; a cached row's int8 code may be one off
            bound = (1e-2 if dt == orc.F16 else 13 * 2.0 ** -9) + (1 / 127 if kv8 else 0)
            assert max_err_rel_to_max(g.f32(got[b], dt), g.f32(want[0], dt)) <= bound, (i, b)
    dec.close()


# prompts and chunks of fewer than 16 rows: one launch per linear, the norm inside up to 4096 values
@pytest.mark.parametrize("dt", [orc.F16, orc.BF16])
@pytest.mark.parametrize("bias", [False, True], ids=["plain", "bias"])
@pytest.mark.parametrize("batch,rows", [(1, 2), (1, 7), (1, 15), (3, 4)])
@pytest.mark.parametrize("hidden,ffn", [(256, 384), (2176, 768)])
def test_prefill_of_few_rows(g, dt, bias, batch, rows, hidden, ffn):
    cfg, w = llm_weights.synthetic_int8(dict(SMALL, n_layers=2, hidden=hidden, ffn=ffn, n_heads=hidden // 64, n_kv_heads=hidden // 128, head_dim=64), dt, seed=rows)
    if bias:
        w = llm_weights.add_qkv_bias(cfg, w, dt, seed=9, std=0.05)
    dec = g.mynn.Decoder(cfg, dev_weights(g, w, dt), seq_q=rows, batch=batch)
    names = [k[0] for k in dec.profile(np.zeros(batch * rows, np.int64), np.arange(rows), 0, rows)]
    assert names.count("rms_norm") == 0, names
    refs = [orc.Model(cfg, w) for _ in range(batch)]
    rng = np.random.default_rng(rows + batch)
    for past in (0, rows, 2 * rows):
        ids, pos = rng.integers(0, cfg["vocab"], (batch, rows)), np.arange(past, past + rows)
        _, got = dec.step(ids.reshape(-1), pos, past, past + rows, want_logits=True)
        got = got.reshape(batch, rows, -1)
        for b, ref in enumerate(refs):
            want = ref.forward(ids[b], pos, past, past + rows, True)
            # 25 stored values lie between a token and its logits through two layers
            assert max_err_rel_to_max(g.f32(got[b], dt), g.f32(want, dt)) <= (1e-2 if dt == orc.F16 else 25 * 2.0 ** -9), (past, b)
    dec.close()
