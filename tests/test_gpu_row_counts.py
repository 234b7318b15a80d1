"""Executors at row counts between the ones their kernels are tiled for: each against the oracle."""
import numpy as np
import pytest

import llm_weights
import oracle as orc
from conftest import max_err_rel_to_max
from test_gpu_decoder import FEWROWS, dev_weights

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def g():
    import gpu_util

    return gpu_util


@pytest.mark.parametrize("dt", [orc.F16, orc.BF16])
@pytest.mark.parametrize("B", [2, 15])
def test_small_batch_decode_vs_per_sequence_oracles(g, dt, B):
    """2 .. 15 sequences take the few-row matrix-core kernel too (most of an MFMA's columns empty)."""
    cfg, w = llm_weights.synthetic_int8(FEWROWS, dt, seed=13)
    dec = g.mynn.Decoder(cfg, dev_weights(g, w, dt), batch=B)
    assert "linear_gateup_swiglu" in [k[0] for k in dec.profile(np.zeros(B, np.int64), [0], 0, 1)]
    refs = [orc.Model(cfg, w) for _ in range(B)]
    rng = np.random.default_rng(B)
    for step in range(4):
        toks = rng.integers(0, cfg["vocab"], B)
        nxt, got = dec.step(toks, [step], step, step + 1, want_logits=True)
        for b in range(B):
            want = refs[b].forward([toks[b]], [step], step, step + 1, False)
            assert max_err_rel_to_max(g.f32(got[b:b + 1], dt), g.f32(want, dt)) <= 1e-2, (step, b)
            assert nxt[b] == orc.argmax_last(got[b], dt)
    dec.close()


@pytest.mark.parametrize("vocab", [65537, 73728, 81923])
def test_greedy_tokens_of_a_prefill_batch_with_a_long_vocabulary(g, vocab):
    """Rows long enough to be shared by several workgroups (parts of 8192 entries, the last one ragged; odd lengths, whose
    rows are not 16-byte aligned), the last rows of two prompts in one launch, replayed from the captured step."""
    dt = orc.F16
    cfg, w = llm_weights.synthetic_int8(dict(FEWROWS, n_layers=1, vocab=vocab), dt, seed=3)
    B, S = 2, 3
    dec = g.mynn.Decoder(cfg, dev_weights(g, w, dt), seq_q=S, batch=B)
    assert dec.stats()["graph"]
    rng = np.random.default_rng(vocab)
    for _ in range(3):
        ids = rng.integers(0, vocab, B * S)
        nxt, got = dec.step(ids, np.arange(S), 0, S, want_logits=True)
        got = got.reshape(B, S, vocab)
        assert list(nxt) == [orc.argmax_last(got[b, S - 1], dt) for b in range(B)]
    dec.close()
