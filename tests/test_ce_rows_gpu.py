"""The loss and its gradient at row lengths around every form of the row kernel, aligned and not, against 64 bits."""

import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

PAD = 0


# fp32 sums of V exponentials in a tree, expf at 1-2 ulp: 1e-6 covers the loss; the gradient's elements carry the
# exponentials' and the sum's errors
@pytest.mark.parametrize("V", [1, 2, 3, 4, 5, 7, 1023, 2047, 2048, 2051, 2052, 4099, 8193, 16387, 16388, 32771, 32773, 53251, 53252,
                               77827, 102403, 102404, 131075, 131076, 131079])
def test_row_lengths(V):
    from dirktensor_amd import ce_loss

    B, T = 2, 5
    g = torch.Generator(device="cuda").manual_seed(V)
    lg = 3.0 * torch.randn((B, T, V), generator=g, device="cuda")
    tok = np.random.default_rng(V).integers(0, V, size=(B, T)).astype(np.int32)
    tok[1, 3] = PAD
    tok[0, 2] = V - 1
    loss, grad = ce_loss(lg, tok, PAD, with_grad=True)
    z = lg[:, :-1].double().reshape(-1, V)
    tgt = torch.as_tensor(tok[:, 1:].astype(np.int64), device="cuda").reshape(-1)
    keep = tgt != PAD
    want = torch.zeros((B, T, V), dtype=torch.float64, device="cuda")
    if int(keep.sum()) == 0:  # (V = 1: every token is the ignored one)
        assert np.isnan(loss) and torch.isnan(grad).all()
        return
    lse = torch.logsumexp(z, -1)
    terms = (lse - z.gather(1, tgt[:, None])[:, 0])[keep]
    p = torch.exp(z - lse[:, None])
    p.scatter_add_(1, tgt[:, None], -torch.ones_like(p[:, :1]))
    p[~keep] = 0
    want[:, :-1] = p.reshape(B, T - 1, V) / int(keep.sum())
    assert abs(loss - float(terms.mean())) <= 1e-6 * abs(float(terms.mean())) + 1e-7
    assert float((grad.double() - want).norm() / want.norm()) < 1e-6


def test_rows_off_16_bytes():
    """Logits and gradient that start 4 bytes past a 16-byte boundary."""
    from dirktensor_amd import ce_loss

    T, V = 4, 5000
    buf = torch.randn(T * V + 1, generator=torch.Generator(device="cuda").manual_seed(1), device="cuda")
    lg = buf[1:].view(1, T, V)
    tok = np.array([[1, 7, 4999, 3]], np.int32)
    loss, grad = ce_loss(lg, tok, PAD, with_grad=True)
    loss2, grad2 = ce_loss(lg.clone(), tok, PAD, with_grad=True)
    assert loss == loss2 and torch.equal(grad, grad2)


@pytest.mark.parametrize("V,offset", [(102400, 0), (102404, 0), (110001, 0), (110004, 1), (131072, 0), (131076, 0)])
@pytest.mark.parametrize("rows", [40, 600])
def test_loss_without_gradient(rows, V, offset):
    """Few and many rows (the form for long rows depends on their number), aligned and not; tolerance as above."""
    from dirktensor_amd import ce_loss

    buf = 3.0 * torch.randn((rows + 1) * V + offset, generator=torch.Generator(device="cuda").manual_seed(V), device="cuda")
    lg = buf[offset:].view(1, rows + 1, V)
    tok = np.random.default_rng(V).integers(1, V, size=(1, rows + 1)).astype(np.int32)
    loss = ce_loss(lg, tok, PAD)
    z = lg[0, :-1]
    tgt = torch.as_tensor(tok[0, 1:].astype(np.int64), device="cuda")
    want = float(np.mean([float(torch.logsumexp(r.double(), -1) - r[t].double()) for r, t in zip(z, tgt)]))
    assert abs(loss - want) <= 1e-6 * abs(want) + 1e-7
