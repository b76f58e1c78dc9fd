"""bf16 forward of launches with few queries (fewer items than CUs, folded or not): edges of query and key tiles and
ragged batches, against attention in 64 bits."""

import math

import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

SCALE = 1.0 / math.sqrt(128.0)


def _reference(q, k, v, causal, lens):
    Q, K, V = (t.double().permute(0, 2, 1, 3).contiguous() for t in (q, k, v))
    B, H, T, _ = Q.shape
    s = Q @ K.transpose(-1, -2).contiguous() * SCALE
    pos = torch.arange(T, device=s.device)
    mask = torch.zeros((B, T, T), dtype=torch.bool, device=s.device)
    if causal:
        mask |= pos[None, None, :] > pos[None, :, None]
    if lens is not None:
        L = torch.as_tensor(np.asarray(lens), device=s.device)
        mask |= pos[None, None, :] >= L[:, None, None]
    s = s.masked_fill(mask[:, None], float("-inf"))
    m = s.amax(-1)
    p = torch.exp(s - m[..., None])
    l = p.sum(-1)
    o = p @ V / l[..., None]
    return o.permute(0, 2, 1, 3), m.permute(0, 2, 1), l.permute(0, 2, 1)


# bf16 Q (scaled), K, V and P: 2^-9 each, in sums of many terms; O lies at about 2.4e-3 from 64 bits, m and l
# (scores of a few units from bf16 operands) below that
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("B,T,H", [(1, 1, 1), (1, 31, 2), (2, 32, 1), (1, 33, 3), (1, 64, 16), (3, 65, 2), (1, 96, 1), (1, 127, 2),
                                   (1, 129, 3), (2, 161, 2), (1, 1000, 16), (1, 1025, 16), (1, 1536, 4), (1, 1537, 4)])
def test_against_64_bits(B, T, H, causal):
    from dirktensor_amd import flash_attention_forward

    g = torch.Generator(device="cuda").manual_seed(T)
    q, k, v = (torch.randn((B, T, H, 128), generator=g, device="cuda").bfloat16() for _ in range(3))
    r = flash_attention_forward(q, k, v, SCALE, causal)
    for got, want in zip((r.output, r.softmax_m, r.softmax_l), _reference(q, k, v, causal, None)):
        assert float((got.double() - want).norm() / want.norm()) < 1e-2


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("T,lens", [(300, [300, 1, 64, 65]), (130, [17, 130, 128]), (640, [640, 321])])
def test_ragged(T, lens, causal):
    from dirktensor_amd import flash_attention_forward

    g = torch.Generator(device="cuda").manual_seed(T)
    q, k, v = (torch.randn((len(lens), T, 3, 128), generator=g, device="cuda").bfloat16() for _ in range(3))
    r = flash_attention_forward(q, k, v, SCALE, causal, seq_lens=lens)
    o, m, l = _reference(q, k, v, causal, lens)
    for b, L in enumerate(lens):
        assert float((r.output[b, :L].double() - o[b, :L]).norm() / o[b, :L].norm()) < 1e-2
        assert float((r.softmax_m[b, :L].double() - m[b, :L]).norm() / m[b, :L].norm()) < 1e-2
        assert float((r.softmax_l[b, :L].double() - l[b, :L]).norm() / l[b, :L].norm()) < 1e-2
        assert (r.output[b, L:] == 0).all() and (r.softmax_l[b, L:] == 0).all()
        assert (r.softmax_m[b, L:] == float("-inf")).all()
