"""Batch-1 decode over a long cache with rows of one to fourteen chunks of 1024 values: the RMSNorm inside the GEMV, in the projection of q, k
and v, in gate/up with its SwiGLU and in the lm_head, whose launch finds the greedy token; against the oracle."""
import numpy as np
import pytest

import oracle as orc
from conftest import max_err_rel_to_max
from test_gpu_decoder import SMALL, dev_weights

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def g():
    import gpu_util

    return gpu_util


def check(g, dt, hidden, kv_heads, vocab):
    cfg = dict(SMALL, n_layers=1, hidden=hidden, n_heads=hidden // 64, n_kv_heads=kv_heads, head_dim=64, ffn=128, vocab=vocab, max_seq=8192, dtype=dt)
    rng = np.random.default_rng(hidden)
    H, KD, F, V = hidden, kv_heads * 64, cfg["ffn"], cfg["vocab"]

    def lin(n, k, std):
        return rng.integers(-127, 128, (n, k), dtype=np.int8), orc.to_storage(rng.uniform(0.9, 1.1, n) * std / 73.0, dt)

    def norm():
        return orc.to_storage(rng.uniform(0.5, 1.5, H), dt)

    w = {"embed": lin(V, H, 1.0), "lm_head": lin(V, H, H**-0.5), "final_norm": norm(), "layers.0.norm1": norm(), "layers.0.norm2": norm()}
    for name, n, k in (("q", H, H), ("k", KD, H), ("v", KD, H), ("o", H, H), ("gate", F, H), ("up", F, H), ("down", H, F)):
        w["layers.0." + name] = lin(n, k, k**-0.5)
    dec, ref = g.mynn.Decoder(cfg, dev_weights(g, w, dt)), orc.Model(cfg, w)
    assert dec.stats()["launches_per_step"] == 5 + 2
    for i, t in enumerate(rng.integers(0, V, 3)):
        want = ref.forward([t], [i], i, i + 1, False)
        tok, got = dec.step([t], [i], i, i + 1, want_logits=True)
        # 13 stored values lie between a token and its logits, each up to half a unit of its type off
        assert max_err_rel_to_max(g.f32(got, dt), g.f32(want, dt)) <= (1e-2 if dt == orc.F16 else 13 * 2.0**-9), i
        assert tok[0] == orc.argmax_last(got[0], dt), i
    dec.close()


@pytest.mark.parametrize("dt", [orc.F16, orc.BF16])
@pytest.mark.parametrize("hidden,kv_heads", [(8448, 33), (14336, 28)])
def test_norm_over_long_rows(g, dt, hidden, kv_heads):
    check(g, dt, hidden, kv_heads, 301)


# (four rows per wave and more rows than the waves take at once; rings of three and of four chunks)
@pytest.mark.parametrize("dt", [orc.F16, orc.BF16])
@pytest.mark.parametrize("hidden,kv_heads,vocab", [(512, 2, 16391), (1024, 4, 30), (4608, 9, 8195), (6144, 12, 301), (7168, 14, 8195), (8192, 16, 301)])
def test_token_of_row_lengths(g, dt, hidden, kv_heads, vocab):
    check(g, dt, hidden, kv_heads, vocab)
