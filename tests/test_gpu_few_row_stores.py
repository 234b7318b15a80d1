"""Few-row products (skinny.hip) that store whole runs turned through LDS, and the launches that add up their K ranges: columns that
end inside a run, a wave's tile and a workgroup's, numbers of columns that no run fits (odd, not a multiple of 16), one and two
tiles of rows, four to twelve ranges, against the oracle."""
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


# q|k|v of 6912 rows and 18 K steps: five ranges; down of 2304 rows and 46 steps: twelve; vocabularies of 6001 and 6004 rows: five;
# from 24545 rows on (vocabulary, or gate|up of 12416) a workgroup has the whole K range and stores the finished output
@pytest.mark.parametrize("dt", [orc.F16, orc.BF16])
@pytest.mark.parametrize("B", [17, 32, 33, 64])
@pytest.mark.parametrize("hidden,ffn,vocab,kv8", [(2304, 5888, 6001, False), (2304, 5888, 6004, True), (256, 12416, 24560, False), (256, 384, 24592, False),
                                                  (256, 384, 24561, False), (256, 384, 24568, False)])
def test_few_row_products(g, dt, B, hidden, ffn, vocab, kv8):
    heads = (18, 18, 128) if kv8 else (hidden // 64, hidden // 64, 64)
    cfg, w = llm_weights.synthetic_int8(dict(SMALL, n_layers=1, hidden=hidden, ffn=ffn, vocab=vocab, n_heads=heads[0], n_kv_heads=heads[1],
                                             head_dim=heads[2]), dt, seed=B)
    dec = g.mynn.Decoder(cfg, dev_weights(g, w, dt), batch=B, quant_kv_cache=kv8)
    rng = np.random.default_rng(B)
    refs = {b: orc.Model(cfg, w) for b in (0, 16, B - 1)}
    for ref in refs.values():
        ref.set_options(quant_kv_cache=kv8)
    for step in range(2):
        toks = rng.integers(0, cfg["vocab"], B)
        ids, got = dec.step(toks, [step], step, step + 1, want_logits=True)
        got = got.reshape(B, -1)
        for b, ref in refs.items():
            want = ref.forward([toks[b]], [step], step, step + 1, False)
            assert max_err_rel_to_max(g.f32(got[b], dt), g.f32(want[0], dt)) <= (2e-2 if kv8 else 1e-2), (step, b)
    dec.close()
