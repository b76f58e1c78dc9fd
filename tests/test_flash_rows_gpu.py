"""A row's results do not depend on what else is in the launch: heads alone and among others, a sequence alone and in a
(padded) batch, come out bit for bit the same, at lengths that are no multiple of any tile too. (Launches whose items
are split, long sequences of few heads, are merged in another order; none of these is.)"""

import math

import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

SCALE = 1.0 / math.sqrt(128.0)


def _qkv(B, T, H, dtype):
    g = torch.Generator(device="cuda").manual_seed(T)
    return [torch.randn((B, T, H, 128), generator=g, device="cuda").to(dtype) for _ in range(3)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("T,H", [(1, 16), (33, 2), (65, 3), (300, 2), (511, 16), (777, 4), (960, 8), (1000, 16)])
def test_heads_alone_and_among_others(T, H, causal, dtype):
    from dirktensor_amd import flash_attention_forward

    q, k, v = _qkv(1, T, H, dtype)
    r = flash_attention_forward(q, k, v, SCALE, causal)
    rep = 600 // (H * ((T + 127) // 128)) + 1  # more than two rounds of any device's CUs
    big = flash_attention_forward(*[t.repeat(1, 1, rep, 1) for t in (q, k, v)], SCALE, causal)
    for i in range(rep):
        for x, y in zip((r.output, r.softmax_m, r.softmax_l), (big.output, big.softmax_m, big.softmax_l)):
            assert torch.equal(y[:, :, i * H:(i + 1) * H], x)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("T,lens", [(300, [300, 1, 64, 65]), (1000, [1000, 511, 770])])
def test_sequences_alone_and_in_a_batch(T, lens, causal, dtype):
    from dirktensor_amd import flash_attention_forward

    q, k, v = _qkv(len(lens), T, 3, dtype)
    r = flash_attention_forward(q, k, v, SCALE, causal, seq_lens=lens)
    for b, L in enumerate(lens):
        one = flash_attention_forward(*[t[b:b + 1, :L].contiguous() for t in (q, k, v)], SCALE, causal)
        for x, y in zip((r.output, r.softmax_m, r.softmax_l), (one.output, one.softmax_m, one.softmax_l)):
            assert torch.equal(x[b:b + 1, :L], y)
