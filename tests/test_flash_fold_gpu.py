"""Folded launches of sequences that are no multiple of 128 (an even number of 64-query tiles, the last one partial):
against 64-bit attention, and bit for bit against the unfolded schedule that the same heads take in a larger launch."""

import math

import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

SCALE = 1.0 / math.sqrt(128.0)


# tolerances as in the kernels' own tests: 1e-6 / 2e-6 for the split fp32 products, 1e-2 for bf16
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,T,H", [(1, 193, 3), (1, 255, 16), (2, 1985, 8), (1, 1999, 16), (1, 2047, 16)])
def test_folded_odd_lengths(B, T, H, dtype):
    from dirktensor_amd import flash_attention_forward

    g = torch.Generator(device="cuda").manual_seed(T)
    q, k, v = (torch.randn((B, T, H, 128), generator=g, device="cuda").to(dtype) for _ in range(3))
    r = flash_attention_forward(q, k, v, SCALE, True)
    Q, K, V = (t.double().permute(0, 2, 1, 3).contiguous() for t in (q, k, v))
    s = Q @ K.transpose(-1, -2).contiguous() * SCALE
    s.masked_fill_(torch.ones(T, T, dtype=torch.bool, device=s.device).triu(1), float("-inf"))
    m = s.amax(-1)
    p = torch.exp_(s.sub_(m[..., None]))
    l = p.sum(-1)
    o = (p @ V / l[..., None]).permute(0, 2, 1, 3)
    tol = 2e-6 if dtype == torch.float32 else 1e-2
    for got, want in zip((r.output, r.softmax_m, r.softmax_l), (o, m.permute(0, 2, 1), l.permute(0, 2, 1))):
        assert float((got.double() - want).norm() / want.norm()) < tol
    rep = 300 // (B * H * (T // 128 + 1)) + 1  # more than one round: unfolded
    big = flash_attention_forward(*[t.repeat(1, 1, rep, 1) for t in (q, k, v)], SCALE, True)
    for i in range(rep):
        assert torch.equal(big.output[:, :, i * H:(i + 1) * H], r.output)
        assert torch.equal(big.softmax_m[:, :, i * H:(i + 1) * H], r.softmax_m)
        assert torch.equal(big.softmax_l[:, :, i * H:(i + 1) * H], r.softmax_l)
