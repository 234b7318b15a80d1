"""How exactly the softmax weights enter the second product of the matrix-core attention kernels.  The outputs are 16-bit
values; an error e of the f32 arithmetic (relative, against 64 bits) makes 2 e / ulp of them round to a neighbour of the
nearest value, an ulp being 2^-7.5 (bf16) or 2^-10.5 (fp16) of the value on average.  Scores, exponentials and sums in f32
come to e of some 2^-21; 2^-19 is allowed.  Weights cut to 16 bits (two bf16 values) come to 2^-18, to one value of the type
to 2^-9 and more."""
import numpy as np
import pytest

import oracle as orc


def share_allowed(dt):
    return 2 * 2.0 ** -19 / 2.0 ** (-7.5 if dt == orc.BF16 else -10.5)


def exact(q, k, v, causal, cut=None):
    """[B,Hq,S,D] x [B,Hkv,L,D] in 64 bits; cut: what becomes of the weights"""
    B, Hq, S, D = q.shape
    L, G = k.shape[2], Hq // k.shape[1]
    out = np.empty(q.shape)
    for b in range(B):
        for h in range(Hq):
            s = q[b, h] @ k[b, h // G].T * D ** -0.5
            if causal:
                s[np.arange(L)[None] > np.arange(S)[:, None] + L - S] = -np.inf
            p = np.exp(s - s.max(1, keepdims=True))
            out[b, h] = (p if cut is None else cut(p)) @ v[b, h // G] / p.sum(1, keepdims=True)
    return out


def share_off(got, want, dt):
    return np.mean(got != orc.to_storage(want.astype(np.float32), dt))


def quantised(rng, shape, dt, size=1.0):
    """codes, row scales and values; size: of the largest rows (others are up to 2^6 smaller where it is not 1)"""
    codes = np.clip(np.round(rng.standard_normal(shape) * 45), -127, 127).astype(np.int8)
    scale = rng.uniform(0.018, 0.026, shape[:-1]) * size * np.exp2(-rng.integers(0, 7, shape[:-1]) * (size != 1.0))
    scale = orc.to_storage(scale, dt)
    return codes, scale, codes * orc.to_f32(scale, dt).astype(np.float64)[..., None]


def test_the_bound_tells_two_bf16_values_from_three():
    rng = np.random.default_rng(0)
    dt = orc.BF16
    q = orc.to_f32(orc.to_storage(rng.standard_normal((2, 8, 128, 64)), dt), dt).astype(np.float64)
    k, v = (quantised(rng, (2, 2, 300, 64), dt)[2] for _ in range(2))
    want = exact(q, k, v, True)

    def parts(n):
        def cut(p):
            total, rest = np.zeros_like(p), p
            for _ in range(n):
                total = total + orc.to_f32(orc.to_storage(rest.astype(np.float32), dt), dt)
                rest = p - total
            return total
        return share_off(orc.to_storage(exact(q, k, v, True, cut).astype(np.float32), dt), want, dt)

    assert parts(2) > share_allowed(dt) > parts(3) and parts(1) > 20 * share_allowed(dt)


@pytest.fixture(scope="module")
def g():
    import gpu_util

    return gpu_util


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [orc.F16, orc.BF16])
@pytest.mark.parametrize("D", [64, 128])
def test_prefill_over_an_int8_cache(g, dt, D):
    rng = np.random.default_rng(D)
    B, Hq, Hkv, S, L = 2, 16, 2, 200, 500
    q = orc.to_storage(rng.standard_normal((B, Hq, S, D)), dt)
    (kq, ks, k), (vq, vs, v) = quantised(rng, (B, Hkv, L, D), dt), quantised(rng, (B, Hkv, L, D), dt)
    got = g.to_host(g.mynn.attention(g.to_dev(q, dt), g.to_dev(kq), g.to_dev(vq), D ** -0.5, True, L, q_pos_offset=L - S,
                                     k_scale=g.to_dev(ks, dt), v_scale=g.to_dev(vs, dt)))
    assert share_off(got, exact(orc.to_f32(q, dt).astype(np.float64), k, v, True), dt) <= share_allowed(dt)


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [orc.F16, orc.BF16])
@pytest.mark.parametrize("kv8,size", [(False, 1.0), (True, 1.0), (True, 1.5e4), (True, 1e-3)], ids=["kv16", "kv_int8", "kv_int8_large", "kv_int8_small"])
@pytest.mark.parametrize("D,Hkv", [(64, 4), (128, 8)])
def test_streaming_decode(g, dt, kv8, size, D, Hkv):
    """the kernel of batched decode steps, through its paged form (which takes it at every size); values at both ends of
    fp16 (a value's scale multiplies its key's weight)"""
    import torch

    rng = np.random.default_rng(D + kv8)
    B, Hq, L, P = 8, 32, 300, 64
    n = (L + P - 1) // P
    off = []
    for _ in range(3):
        q = orc.to_storage(rng.standard_normal((B, Hq, 1, D)), dt)
        sc = [None, None]
        if kv8:
            (kq, sc[0], k), (vq, sc[1], v) = quantised(rng, (B, Hkv, n * P, D), dt), quantised(rng, (B, Hkv, n * P, D), dt, size)
        else:
            kq, vq = (orc.to_storage(rng.standard_normal((B, Hkv, n * P, D)), dt) for _ in range(2))
            k, v = (orc.to_f32(x, dt).astype(np.float64) for x in (kq, vq))

        def pool(x):  # pages of a sequence in a row
            x = x.reshape(B, Hkv, n, P, *x.shape[3:])
            return g.to_dev(np.ascontiguousarray(x.swapaxes(1, 2)).reshape(B * n, Hkv, P, *x.shape[4:]), dt)

        table = torch.arange(B * n, dtype=torch.int32, device="cuda").view(B, n)
        got = g.mynn.attention_paged(g.to_dev(q, dt), pool(kq), pool(vq), table, P, D ** -0.5, False, L, q_pos_offset=L - 1,
                                     k_scale_pool=pool(sc[0]) if kv8 else None, v_scale_pool=pool(sc[1]) if kv8 else None)
        off.append(share_off(g.to_host(got), exact(orc.to_f32(q, dt).astype(np.float64), k[:, :, :L], v[:, :, :L], False), dt))
    assert np.mean(off) <= share_allowed(dt), off
