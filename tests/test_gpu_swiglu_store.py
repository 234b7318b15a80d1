"""SwiGLU in the store of a W8A8 executor's gate/up product (tile_gemm.hip; 500 x 11264: gate/up, and no other linear, in
the 256-row tiles of gemm.hip) against the operators one by one: int32 sums are exact, so one-token sequences, whose
attention returns their value row, have to agree in every bit of every row."""
import numpy as np
import pytest

import llm_weights
import oracle as orc
from test_gpu_decoder import SMALL, dev_weights

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def g():
    import gpu_util

    return gpu_util


@pytest.mark.parametrize("dt", [orc.F16, orc.BF16])
@pytest.mark.parametrize("B,ffn,gates", [(2, 320, "both"), (97, 5632, "both"), (300, 5632, "both"), (300, 5632, "negative"), (500, 11264, "negative")])
def test_layer_equals_the_operators(g, dt, B, ffn, gates):
    import torch

    m = g.mynn
    cfg, w = llm_weights.synthetic_int8(dict(SMALL, n_layers=1, hidden=256, ffn=ffn, n_heads=4, n_kv_heads=2, head_dim=64, max_seq=4), dt, seed=B)
    dw = dev_weights(g, w, dt)
    # gates of every size up to some ten: wide enough for both ends of the sigmoid
    dw["layers.0.gate"] = (dw["layers.0.gate"][0], dw["layers.0.gate"][1] * 4)
    if gates == "negative":
        # (all around -5: there the largest of a row, which sets the codes of the others, comes from the sigmoid's tail)
        dw["layers.0.gate"] = (-dw["layers.0.gate"][0].abs().clamp(max=127), dw["layers.0.gate"][1] * 0.375)
        dw["embed"] = (dw["embed"][0].abs().clamp(max=127), dw["embed"][1])
        dw["layers.0.up"] = (dw["layers.0.up"][0], dw["layers.0.up"][1] * 64)
    dec = m.Decoder(cfg, dw, batch=B, quantize_activations=True)
    ids = np.random.default_rng(B).integers(0, cfg["vocab"], B)
    names = [k[0] for k in dec.profile(ids, [0], 0, 1)]
    assert "qlinear_gateup_swiglu" in names and "swiglu" not in names
    _, got = dec.step(ids, [0], 0, 1, want_logits=True)

    def linear(x, name):
        q, s, _ = m.dynamic_quantize_linear(x)
        return m.quantized_matmul(q, s, *dw[name], want_acc=False)[0]

    codes, scale = dw["embed"]
    rows = torch.from_numpy(ids).cuda()
    x = m.dequantize_linear(codes[rows].contiguous(), scale[rows].contiguous())
    v = linear(m.rms_norm(x, dw["layers.0.norm1"], cfg["eps"]), "layers.0.v").view(B, 2, 1, 64)
    x2 = m.add(linear(v.expand(B, 2, 2, 64).reshape(B, 256).contiguous(), "layers.0.o"), x)
    n = m.rms_norm(x2, dw["layers.0.norm2"], cfg["eps"])
    h = m.swiglu(linear(n, "layers.0.gate"), linear(n, "layers.0.up"))
    x3 = m.add(linear(h, "layers.0.down"), x2)
    want = linear(m.rms_norm(x3, dw["final_norm"], cfg["eps"]), "lm_head")
    assert np.array_equal(np.asarray(got).reshape(B, -1), g.to_host(want))
    dec.close()


@pytest.mark.parametrize("dt", [orc.F16, orc.BF16])
@pytest.mark.parametrize("B", [2, 3, 97])
def test_a_forced_tile_runs_the_operators_with_the_same_bits(g, dt, B):
    """an executor with a forced GEMM tile keeps one operator per launch (and no scratch memory for K ranges)"""
    cfg, w = llm_weights.synthetic_int8(dict(SMALL, n_layers=1, hidden=256, ffn=5632, n_heads=4, n_kv_heads=2, head_dim=64, max_seq=4), dt, seed=B)
    dw = dev_weights(g, w, dt)
    ids = np.random.default_rng(B).integers(0, cfg["vocab"], B)
    rows = []
    for tile in (0, 1):
        dec = g.mynn.Decoder(cfg, dw, batch=B, quantize_activations=True, gemm_tile=tile)
        assert ("swiglu" in [k[0] for k in dec.profile(ids, [0], 0, 1)]) == (tile == 1)
        rows.append(dec.step(ids, [0], 0, 1, want_logits=True)[1])
        dec.close()
    assert np.array_equal(*rows)
