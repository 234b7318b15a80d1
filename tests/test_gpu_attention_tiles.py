"""Prefill attention over a 16-bit cache, every split of the key tiles over waves at the edges of its tiles (32 or 64 keys, 32 rows a
wave), behind a past, paged and with values that are far apart, against the result in 64 bits."""
import numpy as np
import pytest

import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def g():
    import gpu_util

    return gpu_util


def reference(q, k, v, scale, causal, active):
    import torch

    B, Hq, S, D = q.shape
    G = Hq // k.shape[1]
    k, v = k[:, :, :active].double(), v[:, :, :active].double()
    rows = torch.arange(S, device=q.device)[:, None] + (active - S)
    hidden = (torch.arange(active, device=q.device)[None, :] > rows) if causal else None
    out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    for b in range(B):
        for h in range(Hq):
            s = q[b, h].double() @ k[b, h // G].T.contiguous() * scale
            if causal:
                s.masked_fill_(hidden, -np.inf)
            out[b, h] = torch.softmax(s, -1) @ v[b, h // G]
    return out


@pytest.mark.parametrize("dt", [orc.F16, orc.BF16])
@pytest.mark.parametrize("B,Hq,Hkv,D,S,past,causal", [
    (11, 32, 8, 64, 97, 0, True),     # 4 x 1 waves, 64 keys: more than 320 blocks
    (11, 32, 8, 128, 65, 31, True),
    (1, 3, 1, 64, 33, 95, True),      # ... and up to 64 rows
    (1, 3, 1, 128, 17, 0, True),
    (1, 4, 2, 64, 66, 62, True),      # 2 x 2, 64 keys
    (1, 4, 2, 64, 191, 1, False),
    (1, 4, 2, 128, 95, 33, True),
    (1, 4, 4, 128, 65, 0, True),
    (5, 32, 8, 128, 161, 30, True),   # 2 x 2, 32 keys: 320 blocks
    (5, 32, 8, 128, 129, 0, False),
    (1, 32, 8, 128, 2001, 30, True),  # 4 x 2: many rows of few heads
    (1, 32, 8, 128, 1281, 3, True),
    (1, 32, 8, 64, 1345, 0, True),    # ... and 2 x 2 at D = 64
])
@pytest.mark.parametrize("paged", [False, True])
def test_tiles(g, dt, B, Hq, Hkv, D, S, past, causal, paged):
    import torch

    T = g.torch_dtype(dt)
    gen = torch.Generator(device="cuda").manual_seed(S * 7 + D + past)
    active = past + S
    P = 64
    pps = (active + P - 1) // P
    if paged and (pps > 64 or not causal):
        pytest.skip("at most 64 pages of a sequence; the paged operator is causal for a block of rows")
    rows = pps * P if paged else active + 3

    def normal(*shape):
        return torch.randn(shape, generator=gen, device="cuda")

    q, k, v = normal(B, Hq, S, D).to(T), normal(B, Hkv, rows, D).to(T), normal(B, Hkv, rows, D).to(T)
    q[:, :, ::5] *= 30  # (rows whose weights are all at a few keys)
    k[:, :, active:] = v[:, :, active:] = float("nan")  # (never to be read into a result)
    if paged:
        table = torch.randperm(B * pps, generator=gen, device="cuda").to(torch.int32).view(B, pps)
        kp, vp = (torch.empty((B * pps, Hkv, P, D), dtype=T, device="cuda") for _ in range(2))
        for pool, rows_of in ((kp, k), (vp, v)):
            pool[table.flatten().long()] = rows_of.view(B, Hkv, pps, P, D).transpose(1, 2).reshape(B * pps, Hkv, P, D)
        got = g.mynn.attention_paged(q, kp, vp, table, P, D ** -0.5, causal, active, q_pos_offset=past)
    else:
        got = g.mynn.attention(q, k, v, D ** -0.5, causal, active)
    want = reference(q, k, v, D ** -0.5, causal, active)
    # weights and output are rounded to T once, the sums are f32: each weight is off by a factor of 1 +- u, and their weighted
    # mean of the values by at most u * max |v|
    u = 2.0 ** -8 if dt == orc.BF16 else 2.0 ** -11
    bound = u * v[:, :, :active].abs().max().item() * (1 + 1e-2) + u * want.abs()
    assert ((got.double() - want).abs() <= bound).all()
