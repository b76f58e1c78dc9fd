"""fp32 exact mode over the range of fp32: numbers far smaller or larger than those beside them, in each operand and in the
probabilities and their gradients, keep their precision, forward and backward, whichever kernel forms them. Against 64 bits,
column by column or row by row where the magnitudes differ. Tolerances as in the kernels' own tests (1e-6 forward, 3e-6
backward) unless derived beside the test."""

import math

import pytest

from parity import attention64, attention_bwd64

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

SCALE = 1.0 / math.sqrt(128.0)


def _randn(shape, n, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return [torch.randn(shape, generator=g, device="cuda") for _ in range(n)]


def _bwd(do, q, k, v, scale, causal, path, q64=None, k64=None):
    """The kernel's gradients and the 64-bit ones, [B, H, T, D]. (q64, k64: rows of the same scores for the 64-bit side.)"""
    from dirktensor_amd import Context, flash_attention_backward

    q64, k64 = q if q64 is None else q64, k if k64 is None else k64
    o, m, l = attention64(q64, k64, v, scale, causal)
    stats = (o.permute(0, 2, 1, 3).float().contiguous(), m.permute(0, 2, 1).float().contiguous(),
             l.permute(0, 2, 1).float().contiguous())
    ctx = Context(0)
    ctx.set_bwd_dq_path(path)
    r = flash_attention_backward(do, *stats, q, k, v, scale, causal, ctx=ctx)
    got = [t.double().permute(0, 2, 1, 3) for t in (r.d_Q, r.d_K, r.d_V)]
    return got, attention_bwd64(do, *stats, q64, k64, v, scale, causal)


def _norm(x, dim):
    return torch.linalg.vector_norm(x, dim=dim)


def _rel(got, want, dim):
    """The largest relative error (2-norm) over the slices along the other dims."""
    return float((_norm(got - want, dim) / _norm(want, dim)).max())


ROWS = (0, 1, 2)  # norms over everything but the columns (head dims)


@pytest.mark.parametrize("causal", [True, False])
def test_forward_small_and_large_columns_of_v(causal):
    from dirktensor_amd import flash_attention_forward

    q, k, v = _randn((1, 200, 2, 128), 3, 1)
    for d, s in ((3, 1e-36), (40, 1e-33), (77, 1e-30), (101, 1e20)):
        v[..., d] *= s
    r = flash_attention_forward(q, k, v, SCALE, causal)
    o, _, _ = attention64(q, k, v, SCALE, causal)
    got = r.output.double().permute(0, 2, 1, 3)
    unit = _norm(o, ROWS)
    assert _rel(got / unit, o / unit, ROWS) < 1e-6


# scores of about 1e-7: m is their maximum, to the last bits of q, k and the scale. A few roundings of the products' sum.
@pytest.mark.parametrize("qs,ks,scale", [(1e28, 1e-36, SCALE), (1e-36, 1e28, SCALE), (1e-26, 1e29, 1e-10), (1e-12, 1e29, 1e-24),
                                         (1e10, 1e-6, 1e-38), (1e-20, 1e13, 1.0), (1e-36, 1e-2, 1e30)])
def test_forward_small_scores(qs, ks, scale):
    from dirktensor_amd import flash_attention_forward

    q, k, v = _randn((1, 150, 2, 128), 3, 2)
    q, k = q * qs, k * ks
    r = flash_attention_forward(q, k, v, scale, True)
    o, m, _ = attention64(q, k, v, scale, True)
    m = m.permute(0, 2, 1)
    unit = m.abs().max()
    if unit > 1e-37:  # (denormal results hold fewer bits)
        assert _rel(r.softmax_m.double() / unit, m / unit, (0, 1, 2)) < 1e-6
    assert _rel(r.output.double().permute(0, 2, 1, 3), o, (0, 1, 2, 3)) < 1e-6


def _one_key_far_below(T, H, gap):
    """q, k: key 5 scores `gap` nats below the others' log-sum-exp for every query (the others score about 0)."""
    q, k = _randn((1, T, H, 128), 2, 3)
    k *= 0.05
    q[..., 0], k[..., 0] = 8.0, 0.0
    k[:, 5] = 0.0
    k[:, 5, :, 0] = -(gap - math.log(T - 1)) / (8.0 * SCALE)
    return q, k


# exp2's argument is 123 here, rounded at 2^-24 of its size in a few places (q's factor, the product, the argument): 3e-5
# covers four of them
def test_forward_small_probability_of_a_large_value():
    from dirktensor_amd import flash_attention_forward

    T = 64
    q, k = _one_key_far_below(T, 2, 85.2)
    v = _randn((1, T, 2, 128), 1, 4)[0]
    v[..., 64:] = 0.0
    v[:, 5, :, 64:] = 2.0 ** 90
    r = flash_attention_forward(q, k, v, SCALE, False)
    o, _, _ = attention64(q, k, v, SCALE, False)
    got = r.output.double().permute(0, 2, 1, 3)
    assert _rel(got[..., 64:], o[..., 64:], (0, 1, 2, 3)) < 3e-5
    assert _rel(got[..., :64], o[..., :64], (0, 1, 2, 3)) < 1e-6


# heads: few blocks take the kernels with two groups per workgroup, many the ones with one
@pytest.mark.parametrize("path", ["recompute", "from_ds"])
@pytest.mark.parametrize("H", [2, 80])
@pytest.mark.parametrize("gs,vs", [(3e-18, 3e-18), (1e-18, 1e-18), (1e-30, 1e-6), (1e25, 1e-25)])
def test_backward_small_products(gs, vs, H, path):
    """d_out and V each within range, their product, and so dS, far below it."""
    q, k, v, do = _randn((1, 200, H, 128), 4, 5)
    got, want = _bwd(do * gs, q, k, v * vs, SCALE, True, path)
    for x, y, s in zip(got, want, (gs * vs, gs * vs, gs)):
        assert _rel(x / s, y / s, (0, 1, 2, 3)) < 3e-6


@pytest.mark.parametrize("path", ["recompute", "from_ds"])
@pytest.mark.parametrize("H", [2, 80])
def test_backward_small_columns(H, path):
    q, k, v, do = _randn((1, 200, H, 128), 4, 6)
    for t, d in ((q, 3), (k, 70), (v, 100), (do, 127)):
        t[..., d] *= 1e-36
    got, want = _bwd(do, q, k, v, SCALE, True, path)
    for x, y in zip(got, want):
        unit = _norm(y, ROWS)
        assert _rel(x / unit, y / unit, ROWS) < 3e-6


# as in the forward's test: P's exp2 argument is 123, and lse2 is rounded at the forward's log2 as well: 3e-5
@pytest.mark.parametrize("path", ["recompute", "from_ds"])
@pytest.mark.parametrize("H", [2, 200])
def test_backward_small_probabilities(H, path):
    T = 64
    q, k = _one_key_far_below(T, H, 85.2)
    v, do = _randn((1, T, H, 128), 2, 7)
    got, want = _bwd(do, q, k, v, SCALE, False, path)
    for x, y in zip(got[1:], want[1:]):
        x, y = x[:, :, 5], y[:, :, 5]  # (d_K and d_V of that key are all small)
        assert _rel(x / 1e-37, y / 1e-37, (0, 1, 2)) < 3e-5


@pytest.mark.parametrize("path", ["recompute", "from_ds"])
@pytest.mark.parametrize("H", [2, 80])
@pytest.mark.parametrize("which", ["q", "k", "v", "do", "one_row"])
def test_backward_large_values(which, H, path):
    """Values past what a split holds, in a whole operand or in one row of d_out: the fp32 instruction's results, which are
    the operation's."""
    q, k, v, do = _randn((1, 200, H, 128), 4, 8)
    big = 2.0 ** 106
    if which == "q":
        q, k = q * big, k / big
    elif which == "k":
        q, k = q / big, k * big
    elif which == "v":
        v, do = v * big, do / big
    elif which == "do":
        do = do * big
    else:
        do[:, 150] *= big
    got, want = _bwd(do, q, k, v, SCALE, True, path)
    for x, y in zip(got, want):
        # (one row: the gradients of that query, and of the keys up to it, are as large as it; the other rows are as without)
        for rows in ((slice(0, 150), slice(150, 151), slice(151, 200)) if which == "one_row" else (slice(0, 200),)):
            unit = y[:, :, rows].abs().max()
            assert _rel(x[:, :, rows] / unit, y[:, :, rows] / unit, (0, 1, 2, 3)) < 3e-6


@pytest.mark.parametrize("which", ["q", "k", "v"])
def test_forward_large_values(which):
    from dirktensor_amd import flash_attention_forward

    q, k, v = _randn((1, 200, 2, 128), 3, 9)
    big = 2.0 ** 110
    q, k, v = {"q": (q * big, k / big, v), "k": (q / big, k * big, v), "v": (q, k, v * big)}[which]
    r = flash_attention_forward(q, k, v, SCALE, True)
    o, m, l = attention64(q, k, v, SCALE, True)
    unit = o.abs().max()
    assert _rel(r.output.double().permute(0, 2, 1, 3) / unit, o / unit, (0, 1, 2, 3)) < 1e-6


@pytest.mark.parametrize("H", [2, 80])
def test_scores_that_overflow_on_the_way(H):
    """Terms of about -2^80 and +2^80 in a score's sum, which cancel before the others are added in fp32 (dims 0 and 2, then 16 and
    18, then the rest): a factor on the operands makes the first two overflow."""
    from dirktensor_amd import flash_attention_forward

    q, k, v, do = _randn((1, 200, H, 128), 4, 10)
    rest = torch.ones(128, device=q.device)
    rest[:24], rest[64:88] = 0.0, 0.0
    q0, k0 = q * rest, k * rest
    q, k = q0.clone(), k0.clone()
    for d, s in ((0, -1.0), (2, -1.0), (16, 1.0), (18, 1.0)):
        q[..., d], k[..., d] = 2.0 ** 39, s * 0.75 * 2.0 ** 41
    r = flash_attention_forward(q, k, v, SCALE, True)
    o, _, _ = attention64(q0, k0, v, SCALE, True)
    assert _rel(r.output.double().permute(0, 2, 1, 3), o, (0, 1, 2, 3)) < 1e-6
    got, want = _bwd(do, q, k, v, SCALE, True, "recompute", q0, k0)
    assert _rel(got[2], want[2], (0, 1, 2, 3)) < 3e-6
