"""The softmax denominator of prefill attention over a 16-bit cache: the weights of a tile are summed before they join the row's
running sum, so weights that are too small to move it one at a time still count."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D, Hkv", [(64, 4), (128, 8)])
@pytest.mark.parametrize("Sq", [40, 130, 300, 1300])  # (the splits of a workgroup: 4 x 1, 2 x 2, 2 x 2 with 32-key tiles at D = 128, 4 x 1)
def test_small_weights_count(D, Hkv, Sq):
    import torch

    import gpu_util as g

    T, Hq, keys = torch.float16, 32, 8192
    gen = torch.Generator(device="cuda").manual_seed(Sq + D)
    # key 0 has the weight 1 and the only value, key 1 a weight of no particular size (so that the outputs round as often up as down),
    # each of the others one between 2^-25.8 and 2^-24.2 (half a unit in the last place of 1 is 2^-24): out = value / denominator
    a = torch.linspace(24.2, 25.8, Hq * Sq, dtype=torch.float64, device="cuda").reshape(1, Hq, Sq) * 0.6931471805599453
    q = torch.zeros((1, Hq, Sq, D), dtype=T, device="cuda")
    k = torch.zeros((1, Hkv, keys, D), dtype=T, device="cuda")
    v = torch.zeros_like(k)
    q[..., 0] = a.to(T)
    q[..., 1] = (a - 0.1 - 2 * torch.rand(a.shape, generator=gen, device="cuda")).to(T)
    k[:, :, 0, 0] = 1.0
    k[:, :, 1, 1] = 1.0
    v[:, :, 0] = (1.0 + torch.rand((1, Hkv, D), generator=gen, device="cuda")).to(T)
    out = g.mynn.attention(q, k, v, 1.0)
    s0, s1 = q[..., 0].double(), q[..., 1].double()
    denominator = 1.0 + torch.exp(s1 - s0) + (keys - 2) * torch.exp(-s0)
    want = v[:, :, 0].double().repeat_interleave(Hq // Hkv, 1)[:, :, None] / denominator[..., None]
    off = (out.double() / want - 1.0).mean().item()
    # The running sum of a lane is rounded once per tile, 2^-24 of it at most; a weight's exponential is 2^-22 off at most.  The outputs'
    # own rounding spreads them by 2^-11 / sqrt(3) at most.  (One weight at a time, all those are lost that share a lane with key 0: half
    # of 2^-12, a quarter with two key groups, of a denominator of 1.1 .. 1.9.)
    bound = keys / 32 * 2.0 ** -24 / 2 + 2.0 ** -22 + 5 * 2.0 ** -11 / 3 ** 0.5 / out.numel() ** 0.5
    assert abs(off) <= bound, (off, bound)
