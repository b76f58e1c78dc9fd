"""fp32 exact-mode backward on split bf16 products: against 64-bit gradients at the edges of its blocks and tiles, on
both sides of the rule that picks one or two groups per workgroup, and at the limits of what a split can represent."""

import math

import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

SCALE = 1.0 / math.sqrt(128.0)


def _inputs(B, T, H, causal, seed, vs=1.0, gs=1.0):
    """q, k, v, d_out in fp32, the forward's results and the gradients in 64 bits."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    q, k, v, do = (torch.randn((B, T, H, 128), generator=g, device="cuda") for _ in range(4))
    v, do = v * vs, do * gs
    Q, K, V, G = (t.double().permute(0, 2, 1, 3).contiguous() for t in (q, k, v, do))
    tr = lambda t: t.transpose(-1, -2).contiguous()
    s = Q @ tr(K) * SCALE
    if causal:
        s = s.masked_fill(torch.ones(T, T, dtype=torch.bool, device=s.device).triu(1), float("-inf"))
    m = s.amax(-1)
    l = torch.exp(s - m[..., None]).sum(-1)
    p = torch.exp(s - m[..., None]) / l[..., None]
    o = p @ V
    # the kernel takes o, m and l as fp32: the reference takes the same values
    o32, m32, l32 = (t.float() for t in (o, m, l))
    p = torch.exp(s - m32.double()[..., None]) / l32.double()[..., None]
    ds = p * (G @ tr(V) - (G * o32.double()).sum(-1, keepdim=True)) * SCALE
    ref = [t.permute(0, 2, 1, 3) for t in (ds @ K, tr(ds) @ Q, tr(p) @ G)]
    args = (do, o32.permute(0, 2, 1, 3).contiguous(), m32.permute(0, 2, 1).contiguous(), l32.permute(0, 2, 1).contiguous(), q, k, v)
    return args, ref


def _rel(a, b):
    return float((a.double() - b).norm() / b.norm())


def _ctx(path):
    from dirktensor_amd import Context

    ctx = Context(0)
    ctx.set_bwd_dq_path(path)
    return ctx


# What the split leaves is fp32 accumulation (2^-24 per addition), exp2's argument rounded at 2^-24 of a score's size
# and the row statistics as the caller rounded them to fp32 (delta: 2^-24 of |O| |dO|): 3e-6 in the 2-norm is several
# times their sum.
@pytest.mark.parametrize("path", ["recompute", "from_ds"])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("B,T,H", [(1, 1, 1), (1, 31, 2), (2, 33, 1), (1, 64, 16), (1, 65, 2), (1, 127, 1), (2, 161, 3),
                                   (1, 512, 2), (1, 700, 2), (2, 1000, 16)])
def test_against_64_bits(B, T, H, causal, path):
    from dirktensor_amd import flash_attention_backward

    args, ref = _inputs(B, T, H, causal, T)
    r = flash_attention_backward(*args, SCALE, causal, ctx=_ctx(path))
    for got, want in zip((r.d_Q, r.d_K, r.d_V), ref):
        if T > 1 or want is ref[2]:  # (T = 1: dQ and dK are 0 up to rounding)
            assert _rel(got, want) < 3e-6


@pytest.mark.parametrize("path", ["recompute", "from_ds"])
@pytest.mark.parametrize("gs,vs", [(1e-35, 1.0), (1e30, 1e-30), (1.0, 1e-33)])
def test_scaled_values(gs, vs, path):
    """Gradients and values far from 1, down to where a split's last part would be denormal without a factor."""
    from dirktensor_amd import flash_attention_backward

    args, ref = _inputs(1, 200, 2, True, 7, vs=vs, gs=gs)
    r = flash_attention_backward(*args, SCALE, True, ctx=_ctx(path))
    assert _rel(r.d_V / gs, ref[2] / gs) < 3e-6
    if gs * vs > 1e-37:  # (below, dP itself is denormal)
        for got, want in zip((r.d_Q, r.d_K), ref):
            assert _rel(got / (gs * vs), want / (gs * vs)) < 3e-6


@pytest.mark.parametrize("path", ["recompute", "from_ds"])
def test_infinite_gradient(path):
    """An infinite element of d_out: in fp32 arithmetic dV of its dim is infinite for the keys its query sees and 0
    times infinity, NaN, for the masked keys of the same tile; the other dims of dV are as without it."""
    from dirktensor_amd import flash_attention_backward

    args, ref = _inputs(1, 200, 1, True, 9)
    do = args[0].clone()
    do[0, 150, 0, 3] = float("inf")
    r = flash_attention_backward(do, *args[1:], SCALE, True, ctx=_ctx(path))
    rest = [d for d in range(128) if d != 3]
    assert (r.d_V[0, :128, 0, 3] == float("inf")).all()
    assert _rel(r.d_V[0, :, 0][:, rest], ref[2][0, :, 0][:, rest]) < 3e-6
