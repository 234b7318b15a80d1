"""Streaming decode attention: workgroups of four and of eight waves, one key range, as many as are merged with one wait for memory
(8, 16) and more, at lengths that leave a range or a wave without keys, against the result in 64 bits and against the separate
merge (the entry that allocates nothing)."""
import pytest

import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def g():
    import gpu_util

    return gpu_util


@pytest.mark.parametrize("dt", [orc.F16, orc.BF16])
@pytest.mark.parametrize("kv8", [False, True])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("B,Hq,Hkv,active", [
    (16, 32, 4, 129), (16, 32, 4, 256), (20, 8, 4, 250),   # eight waves, one range
    (16, 32, 4, 257), (8, 4, 4, 500), (4, 32, 4, 1000),    # four waves, a few ranges
    (2, 16, 4, 2048), (8, 8, 1, 2041),                     # four waves, sixteen ranges
    (4, 8, 4, 2048), (16, 2, 1, 1993), (1, 32, 4, 4090),   # eight waves, eight and more ranges
    (4, 32, 4, 1153), (3, 8, 4, 1790), (9, 8, 4, 1500),    # ... and five to seven
    (1, 8, 4, 8192), (1, 4, 1, 16300),                     # more than sixteen
    (17, 16, 8, 1056), (64, 8, 8, 1300),                   # a wave walks several tiles; caches beyond 320 MB (D = 128)
])
def test_ranges(g, dt, kv8, D, B, Hq, Hkv, active):
    import torch

    T, G = g.torch_dtype(dt), Hq // Hkv
    gen = torch.Generator(device="cuda").manual_seed(active + D + B)
    rows = (active + 32) // 32 * 32
    q = torch.randn((B, Hq, 1, D), generator=gen, device="cuda").to(T)
    if kv8:
        k, v = (torch.randint(-127, 128, (B, Hkv, rows, D), generator=gen, dtype=torch.int8, device="cuda") for _ in range(2))
        ks, vs = ((torch.rand((B, Hkv, rows), generator=gen, device="cuda") * 0.02 + 0.01).to(T) for _ in range(2))
        kd, vd = k.double() * ks.double()[..., None], v.double() * vs.double()[..., None]
        k[:, :, active:] = v[:, :, active:] = -128
        ks[:, :, active:] = vs[:, :, active:] = float("nan")
    else:
        k, v = (torch.randn((B, Hkv, rows, D), generator=gen, device="cuda").to(T) for _ in range(2))
        ks = vs = None
        kd, vd = k.double(), v.double()
        k[:, :, active:] = v[:, :, active:] = float("nan")
    got = g.mynn.attention(q, k, v, D ** -0.5, active=active, k_scale=ks, v_scale=vs)
    want = torch.empty(q.shape, dtype=torch.float64, device="cuda")
    for b in range(B):
        for h in range(Hq):
            s = kd[b, h // G, :active] @ q[b, h, 0].double() * D ** -0.5
            want[b, h, 0] = torch.softmax(s, -1) @ vd[b, h // G, :active]
    # the output is rounded once; scores, weights and sums are f32 (a score of size s moves its weight by 2^-24 s, with scores up
    # to some 10 and sums of `active` terms well below 2^-16 of the largest value)
    u = 2.0 ** -8 if dt == orc.BF16 else 2.0 ** -11
    assert ((got.double() - want).abs() <= u * want.abs() + 2.0 ** -16 * vd[:, :, :active].abs().max()).all()
    out = torch.empty_like(q)
    try:
        g.mynn.attention_noalloc(q, k, v, D ** -0.5, out, active=active, k_scale=ks, v_scale=vs)
    except g.mynn.MynnError:
        return  # (more partial results than its memory holds)
    assert torch.equal(out, got)
