"""Parity metrics shared by the tests.

err = max|O_gpu - O_ref| / max|O_ref| over the compared rows (the tolerance
the reference path is held to: 1e-4 in fp32 exact mode, 2e-2 in bf16 mode).
"""

import numpy as np

TOL_FP32 = 1e-4
TOL_BF16 = 2e-2


def rel_err(got, ref) -> float:
    got = np.asarray(got, dtype=np.float64)
    ref = np.asarray(ref, dtype=np.float64)
    scale = np.max(np.abs(ref))
    return float(np.max(np.abs(got - ref)) / (scale if scale > 0 else 1.0))


def to_np(t):
    import torch

    if isinstance(t, torch.Tensor):
        return t.detach().float().cpu().numpy()
    return np.asarray(t)


def _scores64(q, k, scale, causal):
    """Scaled scores in 64 bits, [B, H, T, T], masked ones -inf. q, k: [B, T, H, D] tensors."""
    import torch

    Q, K = (t.double().permute(0, 2, 1, 3).contiguous() for t in (q, k))
    s = Q @ K.transpose(-1, -2).contiguous() * scale
    if causal:
        T = s.shape[-1]
        s = s.masked_fill(torch.ones(T, T, dtype=torch.bool, device=s.device).triu(1), float("-inf"))
    return s


def attention64(q, k, v, scale, causal):
    """Attention of [B, T, H, D] tensors in 64 bits: o [B, H, T, D], m and l [B, H, T]."""
    import torch

    s = _scores64(q, k, scale, causal)
    m = s.amax(-1)
    p = torch.exp(s - m[..., None])
    l = p.sum(-1)
    return p @ v.double().permute(0, 2, 1, 3).contiguous() / l[..., None], m, l


def attention_bwd64(d_o, o, m, l, q, k, v, scale, causal):
    """Its gradients (dq, dk, dv), [B, H, T, D], in 64 bits from the forward's results o [B, T, H, D] and m, l [B, T, H]."""
    import torch

    Q, K, V, G, O = (t.double().permute(0, 2, 1, 3).contiguous() for t in (q, k, v, d_o, o))
    M, L = (t.double().permute(0, 2, 1) for t in (m, l))
    tr = lambda t: t.transpose(-1, -2).contiguous()
    p = torch.exp(_scores64(q, k, scale, causal) - M[..., None]) / L[..., None]
    ds = p * (G @ tr(V) - (G * O).sum(-1, keepdim=True)) * scale
    return ds @ K, tr(ds) @ Q, tr(p) @ G
