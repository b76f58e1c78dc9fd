"""bf16 backward on both sides of the rule that picks one or two groups per workgroup (flash_bwd_two_groups), at edges of the
64-row blocks and tiles, against gradients in 64 bits from the same inputs."""

import math

import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

SCALE = 1.0 / math.sqrt(128.0)


# bf16 operands of the second products and bf16 results: 2^-9 each, in sums of many terms of random sign; the gradients
# lie at about 3e-3 from 64 bits, as without the groups.
@pytest.mark.parametrize("path", ["recompute", "from_ds"])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("B,T,H", [(1, 63, 1), (1, 64, 2), (1, 65, 1), (1, 129, 2), (1, 193, 3), (1, 1000, 16), (1, 1025, 16)])
def test_groups(B, T, H, causal, path):
    from dirktensor_amd import Context, flash_attention_backward

    ctx = Context(0)
    ctx.set_bwd_dq_path(path)
    g = torch.Generator(device="cuda").manual_seed(T)
    q, k, v, do = (torch.randn((B, T, H, 128), generator=g, device="cuda").bfloat16() for _ in range(4))
    Q, K, V, G = (t.double().permute(0, 2, 1, 3).contiguous() for t in (q, k, v, do))
    tr = lambda t: t.transpose(-1, -2).contiguous()
    s = Q @ tr(K) * SCALE
    if causal:
        s = s.masked_fill(torch.ones(T, T, dtype=torch.bool, device=s.device).triu(1), float("-inf"))
    m = s.amax(-1)
    l = torch.exp(s - m[..., None]).sum(-1)
    p = torch.exp(s - m[..., None]) / l[..., None]
    o = (p @ V).permute(0, 2, 1, 3).contiguous().bfloat16()
    ds = p * (G @ tr(V) - (G * o.double().permute(0, 2, 1, 3)).sum(-1, keepdim=True)) * SCALE
    ref = [t.permute(0, 2, 1, 3) for t in (ds @ K, tr(ds) @ Q, tr(p) @ G)]
    stat = lambda t: t.float().permute(0, 2, 1).contiguous()
    r = flash_attention_backward(do, o, stat(m), stat(l), q, k, v, SCALE, causal, ctx=ctx)
    for got, want in zip((r.d_Q, r.d_K, r.d_V), ref):
        assert float((got.double() - want).norm() / want.norm()) < 8e-3
