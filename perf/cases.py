"""The work that performance is measured on: calls that a program built on this package makes, from one
latency-bound attention launch to a training step of the model.

    attn_fwd     flash_attention_forward, fp32 or bf16, causal or full, equal lengths or right-padded batches
    attn_bwd     flash_attention_backward from the forward's output and statistics
    layer_train  one attention layer's step: zero_grad, forward, backward, step
    ce_loss      the next-token loss with its gradient, over a batch's logits
    model_fwd    prefill: tokens to logits
    model_train  zero_grad, forward, loss, backward, step

``listed()`` names the measured cases, ``draw(rng)`` takes one more from the same ranges, ``prepare`` makes what
a program holds before the call, ``run`` is one call, ``work`` counts what it cannot do without, ``tolerance``
says how far two correct implementations may lie apart and ``exact`` computes the result in 64 bits.
"""

import ctypes
import math

import numpy as np
import torch

import dirktensor_amd as dt
from dirktensor_amd import _capi as capi
from dirktensor_amd import synth

D = 128          # head size
DM = 2048        # model width of the layer and model cases (16 heads)
HIDDEN = 8192    # MLP width
SCALE = 1.0 / math.sqrt(D)
PAD = 100277     # the tokenizer's pad id, ignored by the loss
EPS = 1e-6
THETA = 500000.0
DEV = "cuda:0"


# ---- the cases ------------------------------------------------------------------------------------------------


def listed():
    return [
        # the shortest prompt in exact mode: the launch and the call around it count, not the arithmetic
        dict(name="attn_fwd_fp32_t64", kind="attn_fwd", mode="fp32", B=1, T=64, H=16, causal=True, ragged=False),
        # a prompt of ordinary length, not a multiple of any tile
        dict(name="attn_fwd_bf16_t1000", kind="attn_fwd", mode="bf16", B=1, T=1000, H=16, causal=True, ragged=False),
        # the long prefill that the package is quoted on
        dict(name="attn_fwd_bf16_t4096", kind="attn_fwd", mode="bf16", B=1, T=4096, H=16, causal=True, ragged=False),
        # serving: eight prompts of different lengths, right-padded into one batch
        dict(name="attn_fwd_bf16_ragged_b8", kind="attn_fwd", mode="bf16", B=8, T=2048, H=16, causal=True,
             ragged=True),
        # exact mode over a small batch of odd length
        dict(name="attn_fwd_fp32_b2_t1500", kind="attn_fwd", mode="fp32", B=2, T=1500, H=16, causal=True,
             ragged=False),
        # training on a small batch of short sequences
        dict(name="attn_bwd_bf16_b2_t777", kind="attn_bwd", mode="bf16", B=2, T=777, H=16, causal=True),
        # training at the long context
        dict(name="attn_bwd_bf16_t4096", kind="attn_bwd", mode="bf16", B=1, T=4096, H=16, causal=True),
        # exact-mode gradients (checks of a training run) at an ordinary length
        dict(name="attn_bwd_fp32_t1000", kind="attn_bwd", mode="fp32", B=1, T=1000, H=16, causal=True),
        # one layer's training step: projections, norms, rotation, attention both ways, update
        dict(name="layer_train_bf16_t512", kind="layer_train", mode="bf16", B=1, T=512),
        # the loss over the full vocabulary with the gradient that training starts from
        dict(name="ce_loss_t2048", kind="ce_loss", B=1, T=2048, V=100352),
        # end-to-end prefill of the 16-layer model
        dict(name="model_fwd_bf16_t2048", kind="model_fwd", mode="bf16", B=1, T=2048, layers=16, V=100352),
        # a whole training step, embedding to update, of a shallow model with the full vocabulary
        dict(name="model_train_bf16_t2048", kind="model_train", mode="bf16", B=1, T=2048, layers=2, V=100352),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["attn_fwd", "attn_fwd", "attn_fwd", "attn_bwd", "attn_bwd", "layer_train", "ce_loss",
                       "model_fwd", "model_train"])
    if kind in ("attn_fwd", "attn_bwd"):
        T = _log_int(rng, 33, 4096)
        B = min(rng.randint(1, 8), max(1, 16384 // T if kind == "attn_fwd" else 8192 // T))
        c = dict(kind=kind, mode=rng.choice(["bf16", "bf16", "fp32"]), B=B, T=T, H=rng.choice([2, 4, 8, 16, 16]),
                 causal=rng.random() < 0.85)
        if kind == "attn_fwd":
            c["ragged"] = B > 1 and rng.random() < 0.5
        return c
    if kind == "layer_train":
        T = _log_int(rng, 64, 2048)
        return dict(kind=kind, mode="bf16", B=rng.randint(1, max(1, min(4, 2048 // T))), T=T)
    if kind == "ce_loss":
        T = _log_int(rng, 64, 2048)
        return dict(kind=kind, B=rng.randint(1, max(1, min(4, 2048 // T))), T=T, V=_log_int(rng, 1000, 120000))
    T = _log_int(rng, 64, 2048)
    B = rng.randint(1, max(1, min(2, 2048 // T)))
    if kind == "model_fwd":
        return dict(kind=kind, mode="bf16", B=B, T=T, layers=rng.randint(1, 16), V=_log_int(rng, 1000, 100352))
    return dict(kind=kind, mode="bf16", B=B, T=T, layers=rng.randint(1, 2), V=_log_int(rng, 1000, 100352))


# ---- inputs ---------------------------------------------------------------------------------------------------


def _gen(seed, device=DEV):
    g = torch.Generator(device=device)
    g.manual_seed(int(seed))
    return g


def _tdt(case):
    return torch.bfloat16 if case["mode"] == "bf16" else torch.float32


def _qkv(case, seed, n=3):
    """Rows as the q/k norm and the rotation leave them: unit variance. (n = 4: and the output's gradient.)"""
    g = _gen(seed)
    shape = (case["B"], case["T"], case["H"], D)
    return [torch.randn(shape, generator=g, device=DEV).to(_tdt(case)) for _ in range(n)]


def _lens(case, seed):
    """Prompt lengths uniform in [64, T] (the whole of a shorter T); the longest fills the batch."""
    if not case.get("ragged"):
        return None
    rng = np.random.default_rng(int(seed) + 7)
    lens = rng.integers(min(64, case["T"]), case["T"] + 1, size=case["B"]).astype(np.int32)
    lens[int(rng.integers(case["B"]))] = case["T"]
    return lens


def _tokens(case, seed, pad=True):
    """Token ids; for training, one sequence in a batch of several ends in padding."""
    rng = np.random.default_rng(int(seed) + 11)
    tok = rng.integers(0, case["V"], size=(case["B"], case["T"])).astype(np.int32)
    if pad and case["B"] > 1:
        tok[-1, case["T"] - case["T"] // 4:] = _pad(case)
    return tok


def _pad(case):
    return PAD if case["V"] > PAD else case["V"] - 1


def _layer_weights(seed):
    """Wq, Wk, Wv, Wo ~ N(0, 0.02) ([out][in]), q/k norm weights ~ 1 + N(0, 0.01); and the layer's input and the
    gradient of its output are drawn after them from the same generator."""
    g = _gen(seed)
    ws = [(0.02 * torch.randn((DM, DM), generator=g, device=DEV)).bfloat16().float() for _ in range(4)]
    ns = [1.0 + 0.01 * torch.randn((DM,), generator=g, device=DEV) for _ in range(2)]
    return ws + ns, g


def _layer_io(case, g):
    shape = (case["B"], case["T"], DM)
    return torch.randn(shape, generator=g, device=DEV), torch.randn(shape, generator=g, device=DEV)


def _model_weights(case, seed):
    return synth.device_model_params(DEV, case["layers"], case["V"], HIDDEN, DM, seed=int(seed))


def _logits(case, seed):
    return 2.0 * torch.randn((case["B"], case["T"], case["V"]), generator=_gen(seed), device=DEV)


def prepare(case, seed):
    kind = case["kind"]
    st = dict(case=case)
    if kind == "attn_fwd":
        st["qkv"] = _qkv(case, seed)
        st["lens"] = _lens(case, seed)
    elif kind == "attn_bwd":
        q, k, v, g = _qkv(case, seed, 4)
        # the forward's results as the caller kept them
        o, m, l = _attention64(q, k, v, case["causal"], None)
        st["args"] = (g, o.to(q.dtype), m.float(), l.float(), q, k, v)
    elif kind == "layer_train":
        w, g = _layer_weights(seed)
        st["layer"] = dt.OlmoAttention.from_weights(*w)
        st["x"], st["g"] = _layer_io(case, g)
        st["grads"] = [torch.empty_like(t) for t in w]
    elif kind == "ce_loss":
        st["logits"] = _logits(case, seed)
        st["tok"] = _tokens(case, seed)
    else:
        ctx = dt.default_context(0)
        h = ctypes.c_void_p()
        capi.call("dt_model_create", ctx.handle, case["layers"], DM, DM // D, HIDDEN, case["V"], ctypes.byref(h))
        model = dt.OlmoModel(ctx=ctx, _handle=h, _dims=(case["layers"], DM, HIDDEN, case["V"]))
        st["model"] = model
        st["grads"] = []
        for name, w in _model_weights(case, seed):
            torch.cuda.synchronize()
            capi.call("dt_model_set_param", model.handle, name.encode(), w.data_ptr(), w.numel(),
                      capi.DT_MEM_DEVICE)
            torch.cuda.synchronize()
            if kind == "model_train":
                st["grads"].append((name.encode(), torch.empty_like(w)))
        st["tok"] = _tokens(case, seed, pad=kind == "model_train")
        st["logits"] = torch.empty((case["B"], case["T"], case["V"]), dtype=torch.float32, device=DEV)
    torch.cuda.synchronize()
    return st


# ---- one pass -------------------------------------------------------------------------------------------------


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "attn_fwd":
        q, k, v = st["qkv"]
        r = dt.flash_attention_forward(q, k, v, SCALE, case["causal"], seq_lens=st["lens"])
        return r.output, r.softmax_m, r.softmax_l
    if kind == "attn_bwd":
        r = dt.flash_attention_backward(*st["args"], SCALE, case["causal"])
        return r.d_Q, r.d_K, r.d_V
    if kind == "layer_train":
        layer = st["layer"]
        layer.zero_grad()
        out = layer.forward(st["x"], mode=case["mode"])
        dx = layer.backward(st["g"])
        layer.step(0.0)  # a rate of 0, so that every pass sees the same weights
        capi.call("dt_attn_layer_get_grads", layer.handle, *[t.data_ptr() for t in st["grads"]], capi.DT_MEM_DEVICE,
                  torch.cuda.current_stream().cuda_stream)
        return [out, dx] + st["grads"]
    if kind == "ce_loss":
        return dt.ce_loss(st["logits"], st["tok"], _pad(case), with_grad=True)
    model, logits = st["model"], st["logits"]
    if kind == "model_fwd":
        model.forward(st["tok"], mode=case["mode"], save_for_backward=False, out=logits)
        return logits
    model.zero_grad()
    model.forward(st["tok"], mode=case["mode"], save_for_backward=True, out=logits)
    loss, g = dt.ce_loss(logits, st["tok"], _pad(case), with_grad=True)
    model.backward(g)
    model.step(0.0)
    stream = torch.cuda.current_stream().cuda_stream
    for name, buf in st["grads"]:
        capi.call("dt_model_get_param", model.handle, name, buf.data_ptr(), buf.numel(), 1, capi.DT_MEM_DEVICE,
                  stream)
    return [loss, logits] + [buf for _, buf in st["grads"]]


# ---- what one pass cannot do without ----------------------------------------------------------------------------


def _attn_pairs(case, lens=None):
    """Unmasked (query, key) pairs over the batch."""
    ls = [case["T"]] * case["B"] if lens is None else [int(x) for x in lens]
    return sum(n * (n + 1) // 2 if case.get("causal", True) else n * n for n in ls)


def work(case):
    B, T = case["B"], case["T"]
    kind = case["kind"]
    es = 2 if case.get("mode") == "bf16" else 4
    if kind in ("attn_fwd", "attn_bwd"):
        H = case["H"]
        row = B * T * H
        if case.get("ragged"):  # the mean over uniform lengths
            pairs = int(B * (T * T / 3 + T / 2) / 2) if case["causal"] else int(B * T * T / 3)
            tok = B * T // 2
        else:
            pairs, tok = _attn_pairs(case), B * T
        if kind == "attn_fwd":  # Q K^T and P V; q, k, v in, o, m and l out
            return {"flops": 4 * pairs * H * D, "bytes": 3 * tok * H * D * es + row * (D * es + 8)}
        # S, dP, dV, dQ, dK; d_o, o, q, k, v, m and l in, three gradients out
        return {"flops": 10 * pairs * H * D, "bytes": row * (8 * D * es + 8)}
    rows = B * T
    pairs = _attn_pairs(case)
    layer_w = 4 * DM * DM
    layer_flops = 2 * rows * layer_w + 4 * pairs * DM
    if kind == "layer_train":  # x, d_out in; out, d_x out; weights read and written, gradients written twice
        return {"flops": 3 * 2 * rows * layer_w + 14 * pairs * DM,
                "bytes": 4 * rows * DM * 4 + layer_w * 4 * 5}
    if kind == "ce_loss":
        return {"flops": 4 * rows * case["V"], "bytes": 2 * rows * case["V"] * 4}
    n, V = case["layers"], case["V"]
    flops = n * (layer_flops + 6 * rows * DM * HIDDEN) + 2 * rows * DM * V
    params = n * (layer_w + 3 * DM * HIDDEN) + V * DM
    if kind == "model_fwd":
        return {"flops": flops, "bytes": params * 2 + rows * V * 4}
    # weights read and written, their gradients written, read by the step and copied out; the logits and their
    # gradient written once and read once; the embedding's gradient as the others'
    params += V * DM
    flops = n * (3 * (2 * rows * layer_w + 6 * rows * DM * HIDDEN) + 14 * pairs * DM) + 6 * rows * DM * V
    return {"flops": flops, "bytes": params * 4 * 5 + 4 * rows * V * 4}


def tolerance(case):
    # about four times the distance to exact() (at most 1e-6 in fp32, 2.5e-3 for bf16 attention, 6e-3 for the
    # layer's gradients, 8e-3 for the logits; the model's q/k norm weights' gradients reach 1.5e-2)
    kind = case["kind"]
    if kind in ("attn_fwd", "attn_bwd"):
        return {"rel": 1e-5} if case["mode"] == "fp32" else {"rel": 1e-2}
    if kind == "ce_loss":
        return {"rel": 1e-5}
    if kind == "layer_train":
        return {"rel": 2e-2}
    if kind == "model_fwd":
        return {"rel": 3e-2}
    return {"rel": 4e-2}


# ---- the same results in 64 bits, in plain torch ------------------------------------------------------------------


def _scores64(q, k, causal, L):
    """Scaled scores of one sequence, [H, T, T]; masked pairs at -inf. q, k: [T, H, D] in 64 bits."""
    s = torch.matmul(q.transpose(0, 1).contiguous(), k.permute(1, 2, 0).contiguous()) * SCALE
    T = s.shape[-1]
    pos = torch.arange(T, device=s.device)
    mask = pos[None, :] >= L
    if causal:
        mask = mask | (pos[None, :] > pos[:, None])
    return s.masked_fill_(mask[None], float("-inf"))


def _attention64(q, k, v, causal, lens):
    """(o, m, l) of [B, T, H, D] inputs; rows past a sequence's length are empty (0, -inf, 0)."""
    B, T, H, _ = q.shape
    o = torch.zeros(q.shape, dtype=torch.float64, device=q.device)
    m = torch.full((B, T, H), float("-inf"), dtype=torch.float64, device=q.device)
    l = torch.zeros((B, T, H), dtype=torch.float64, device=q.device)
    for b in range(B):
        L = T if lens is None else int(lens[b])
        s = _scores64(q[b, :L].double(), k[b, :L].double(), causal, L)
        mb = s.amax(-1)
        p = torch.exp_(s.sub_(mb[..., None]))
        lb = p.sum(-1)
        ob = torch.matmul(p, v[b, :L].double().transpose(0, 1).contiguous()) / lb[..., None]
        o[b, :L], m[b, :L], l[b, :L] = ob.transpose(0, 1), mb.transpose(0, 1), lb.transpose(0, 1)
        del s, p
    return o, m, l


def _attention_bwd64(g, o, m, l, q, k, v, causal):
    """Gradients of q, k and v from the forward's output and statistics (all given)."""
    out = [torch.empty(q.shape, dtype=torch.float64, device=q.device) for _ in range(3)]
    for b in range(q.shape[0]):
        T = q.shape[1]
        hd = lambda t: t[b].double().transpose(0, 1).contiguous()  # [H, T, D]
        tr = lambda t: t.transpose(1, 2).contiguous()
        gb, ob, qb, kb, vb = hd(g), hd(o), hd(q), hd(k), hd(v)
        s = _scores64(q[b].double(), k[b].double(), causal, T)
        p = torch.exp_(s.sub_(m[b].double().T[..., None])).div_(l[b].double().T[..., None])
        dp = torch.matmul(gb, tr(vb))
        ds = dp.sub_((gb * ob).sum(-1)[..., None]).mul_(p).mul_(SCALE)
        out[2][b] = torch.matmul(tr(p), gb).transpose(0, 1)
        out[0][b] = torch.matmul(ds, kb).transpose(0, 1)
        out[1][b] = torch.matmul(tr(ds), qb).transpose(0, 1)
        del s, p, dp, ds
    return out


class _Attn64(torch.autograd.Function):
    """Causal attention with the gradient formulas above, one sequence's scores at a time."""

    @staticmethod
    def forward(ctx, q, k, v):
        o, m, l = _attention64(q, k, v, True, None)
        ctx.save_for_backward(q, k, v, o, m, l)
        return o

    @staticmethod
    def backward(ctx, g):
        q, k, v, o, m, l = ctx.saved_tensors
        return tuple(_attention_bwd64(g, o, m, l, q, k, v, True))


def _rms64(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w


def _rope64(x):
    T = x.shape[1]
    inv = THETA ** (-torch.arange(0, D, 2, dtype=torch.float64, device=x.device) / D)
    ang = torch.arange(T, dtype=torch.float64, device=x.device)[:, None] * inv[None]
    cos, sin = (f(ang).repeat(1, 2)[None, :, None, :] for f in (torch.cos, torch.sin))
    rot = torch.cat([-x[..., D // 2:], x[..., :D // 2]], -1)
    return x * cos + rot * sin


def _layer64(x, wq, wk, wv, wo, qn, kn):
    shape = x.shape[:2] + (DM // D, D)
    q = _rope64(_rms64(x @ wq.T, qn).reshape(shape))
    k = _rope64(_rms64(x @ wk.T, kn).reshape(shape))
    v = (x @ wv.T).reshape(shape)
    return _Attn64.apply(q, k, v).reshape(x.shape) @ wo.T


def _model64(tok, p, layers):
    h = p["model.embed_tokens.weight"][tok]
    for i in range(layers):
        w = lambda n: p[f"model.layers.{i}.{n}.weight"]
        a = _layer64(h, *[w(f"self_attn.{n}") for n in ("q_proj", "k_proj", "v_proj", "o_proj", "q_norm", "k_norm")])
        h = h + _rms64(a, w("post_attention_layernorm"))
        act = torch.nn.functional.silu(h @ w("mlp.gate_proj").T) * (h @ w("mlp.up_proj").T)
        h = h + _rms64(act @ w("mlp.down_proj").T, w("post_feedforward_layernorm"))
    return _rms64(h, p["model.norm.weight"]) @ p["lm_head.weight"].T


def _loss64(logits, tok, ignore):
    """The mean next-token cross entropy and its gradient with respect to the logits."""
    tgt = torch.as_tensor(tok[:, 1:].astype(np.int64), device=logits.device).reshape(-1)
    keep = torch.nonzero(tgt != ignore).reshape(-1)
    B, T, V = logits.shape
    rows = (keep // (T - 1)) * T + keep % (T - 1)
    lg = logits.detach().reshape(B * T, V)
    grad = torch.zeros((B * T, V), dtype=torch.float64, device=logits.device)
    total = 0.0
    for r, t in zip(rows.split(256), tgt[keep].split(256)):
        z = lg[r].double()
        lse = torch.logsumexp(z, -1)
        ix = torch.arange(len(r), device=z.device)
        total += float((lse - z[ix, t]).sum())
        pr = torch.exp(z - lse[:, None])
        pr[ix, t] -= 1.0
        grad[r] = pr / len(keep)
    return total / len(keep), grad.reshape(B, T, V)


def exact(case, seed):
    kind = case["kind"]
    if kind == "attn_fwd":
        return _attention64(*_qkv(case, seed), case["causal"], _lens(case, seed))
    if kind == "attn_bwd":
        return tuple(_attention_bwd64(*prepare(case, seed)["args"], case["causal"]))
    if kind == "layer_train":
        w, g = _layer_weights(seed)
        x, dout = (t.double() for t in _layer_io(case, g))
        ws = [t.double().requires_grad_() for t in w]
        x.requires_grad_()
        out = _layer64(x, *ws)
        return [out.detach()] + list(torch.autograd.grad(out, [x] + ws, dout))
    if kind == "ce_loss":
        return _loss64(_logits(case, seed), _tokens(case, seed), _pad(case))
    train = kind == "model_train"
    tok_h = _tokens(case, seed, pad=train)
    tok = torch.as_tensor(tok_h.astype(np.int64), device=DEV)
    p = {n: w.double().requires_grad_(train) for n, w in _model_weights(case, seed)}
    with torch.set_grad_enabled(train):
        logits = _model64(tok, p, case["layers"])
    if not train:
        return logits
    loss, g = _loss64(logits, tok_h, _pad(case))
    grads = torch.autograd.grad(logits, list(p.values()), g)
    return [loss, logits.detach()] + list(grads)
