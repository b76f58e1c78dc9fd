"""fp32 exact mode on split bf16 products: against 64-bit attention, at the edges of its tiles and at the limits of
what a split can represent."""

import math

import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

SCALE = 1.0 / math.sqrt(128.0)


def _attention64(q, k, v, causal):
    q, k, v = (t.double().permute(0, 2, 1, 3) for t in (q, k, v))
    s = q @ k.transpose(-1, -2).contiguous() * SCALE
    if causal:
        T = s.shape[-1]
        s = s.masked_fill(torch.ones(T, T, dtype=torch.bool, device=s.device).triu(1), float("-inf"))
    m = s.amax(-1)
    p = torch.exp(s - m[..., None])
    l = p.sum(-1)
    o = p @ v / l[..., None]
    return o.permute(0, 2, 1, 3), m.permute(0, 2, 1), l.permute(0, 2, 1)


def _qkv(B, T, H, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return [torch.randn((B, T, H, 128), generator=g, device="cuda") for _ in range(3)]


def _rel(a, b):
    return float((a.double() - b).norm() / b.norm())


# A split operand is exact and the partial products left out come to at most 2^-24 of a product (2^-28 on average), no more
# than one fp32 rounding. The rest is fp32 accumulation, at most 2^-24 per addition of a chain of 48 for S and of 12 per 32
# keys for O, and exp2's argument rounded at 2^-24 of a score's size (a few tens): 1e-6 in the 2-norm is several times what
# these give on random data, where the roundings are independent.
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("B,T,H", [(1, 1, 1), (1, 31, 2), (2, 32, 1), (1, 33, 3), (1, 64, 16), (1, 65, 2), (1, 127, 1),
                                   (2, 129, 2), (1, 191, 1), (1, 256, 8), (1, 385, 2), (1, 1000, 2)])
def test_against_64_bits(B, T, H, causal):
    from dirktensor_amd import flash_attention_forward

    q, k, v = _qkv(B, T, H, seed=T)
    r = flash_attention_forward(q, k, v, SCALE, causal)
    o, m, l = _attention64(q, k, v, causal)
    assert _rel(r.output, o) < 1e-6
    assert _rel(r.softmax_m, m) < 1e-6
    assert _rel(r.softmax_l, l) < 2e-6


@pytest.mark.parametrize("vs", [1e-35, 1e-30, 1e30, 1e36])
def test_scaled_values(vs):
    """V far from 1, down to where the last part of its split would be denormal without a factor and up to where the unnormalised sum of 150 rows
    (l is at most a few tens) nears fp32's range; Q and K scaled against each other."""
    from dirktensor_amd import flash_attention_forward

    q, k, v = _qkv(1, 150, 2, seed=3)
    v = (v.clamp(-5, 5) * vs).float()
    qs, ks = (q * 1e25).float(), (k * 1e-25).float()
    r = flash_attention_forward(qs, ks, v, SCALE, True)
    o, m, l = _attention64(qs, ks, v, True)
    assert _rel(r.output / vs, o / vs) < 1e-6
    assert _rel(r.softmax_m, m) < 1e-6


def test_what_does_not_split():
    """Infinities and values past the largest bf16: the rows that see them come out as fp32 arithmetic gives them,
    the others are untouched."""
    from dirktensor_amd import flash_attention_forward

    q, k, v = _qkv(1, 200, 2, seed=5)
    big = float(np.finfo(np.float32).max)
    v[0, 70, 0, 3] = big          # rounds to infinity in bf16
    v[0, 130, 1, 5] = float("inf")
    k[0, 100, 1, 7] = float("-inf")
    r = flash_attention_forward(q, k, v, SCALE, True)
    o, m, l = _attention64(q, k, v, True)
    out = r.output.double()
    # head 0: finite everywhere
    rest = [d for d in range(128) if d != 3]
    assert torch.isfinite(out[0, :, 0]).all()
    assert _rel(out[0, :, 0, rest], o[0, :, 0, rest]) < 1e-6
    assert _rel(out[0, :, 0, 3] / big, o[0, :, 0, 3] / big) < 1e-6
    # head 1: rows before key 100's tile are untouched; from key 100 on a query of positive dim 7 does not see it
    # (-inf), one of negative dim 7 has no finite softmax and reads as an empty row
    rest = [d for d in range(128) if d != 5]  # (dim 5 of the reference is 0 * inf there)
    assert _rel(out[0, :96, 1][:, rest], o[0, :96, 1][:, rest]) < 1e-6
    assert torch.isfinite(out[0, :96, 1, 5]).all()
    for t in range(100, 200):
        if q[0, t, 1, 7] > 0:
            assert _rel(out[0, t, 1, :5], o[0, t, 1, :5]) < 1e-5, t
            if t >= 160:
                assert out[0, t, 1, 5] == float("inf"), t
        else:
            assert (out[0, t, 1] == 0).all() and r.softmax_l[0, t, 1] == 0, t
