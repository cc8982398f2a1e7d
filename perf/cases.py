"""The work this library does for its users, as timed cases: one dict of plain values per case.

Every case is one pass through the public Python API (``kernels``), as a training or serving loop calls it:

* ``decode``     FusedAddRMSNorm, RoPE and SwiGLU forward on a handful of tokens without gradients (one layer's
                 operators of a decode step): launches and host time count.
* ``norm``       RMSNorm or FusedAddRMSNorm, forward and backward.
* ``rope``       rotate-half RoPE of q and k, forward and backward, on (B, H, T, D) views of [B, T, H, D] storage.
* ``glu``        SwiGLU or GeGLU, forward and backward.
* ``ce``         cross entropy with ignored rows: the loss and dlogits.
* ``grpo``       the GRPO loss (PPO clip and KL) with prefix masks: loss, KL, clip ratio and dlogits.
* ``attn_res``   attention residuals over N depth blocks, forward and backward.
* ``flce``       lm_head + cross entropy (the chunked fused-linear loss): loss, dhidden, dweight.
* ``fljsd``      student and teacher lm_heads + JSD: loss, dhidden, dweight.
* ``flgrpo``     lm_head + GRPO loss: loss, KL, clip ratio, dhidden, dweight.

Sizes are those of the benchmark configurations and of the parity tests, and ragged ones between them.
"""
from __future__ import annotations

import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "hilda-kernel_amd"))
from kernels import (  # noqa: E402
    hilda_attn_res,
    hilda_cross_entropy,
    hilda_fused_add_rms_norm,
    hilda_fused_linear_cross_entropy,
    hilda_fused_linear_grpo_loss,
    hilda_fused_linear_jsd,
    hilda_geglu,
    hilda_grpo_loss,
    hilda_rms_norm,
    hilda_rope,
    hilda_swiglu,
)

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
SIZE = {"bf16": 2, "fp16": 2, "fp32": 4}
EPS = 1e-6


def listed():
    return [
        # one layer's operators of a decode step on eight sequences: the smallest calls
        dict(name="decode_layer", kind="decode", tokens=8, hidden=4096, inter=14336, dtype="bf16"),
        # a full-precision norm of a 4096-token batch
        dict(name="rms_norm_fp32", kind="norm", add=False, rows=4096, hidden=4096, dtype="fp32"),
        # the residual norm of an 8B-sized layer in training, twice a layer
        dict(name="fused_add_rms_norm", kind="norm", add=True, rows=8192, hidden=4096, dtype="bf16"),
        # RoPE on a batch of odd length, fp16
        dict(name="rope_ragged", kind="rope", batch=3, seq=1021, heads=32, kv_heads=8, head_dim=128, dtype="fp16"),
        # the activation of an 8B-sized MLP in training
        dict(name="swiglu", kind="glu", act="swiglu", rows=8192, inter=14336, dtype="bf16"),
        # cross entropy of a 32K vocabulary, a tenth of the tokens ignored
        dict(name="cross_entropy", kind="ce", rows=8192, vocab=32000, ignored=0.1, dtype="bf16"),
        # GRPO on eight completions of up to 512 tokens with an odd vocabulary
        dict(name="grpo_odd_vocab", kind="grpo", batch=8, seq=513, vocab=50257, beta=0.1, dtype="bf16"),
        # attention residuals over eight depth blocks of an 8B-sized layer
        dict(name="attn_res", kind="attn_res", blocks=8, rows=8192, hidden=4096, dtype="bf16"),
        # the training loss behind a 32K-vocabulary lm_head under the default memory budget
        dict(name="fused_linear_ce", kind="flce", rows=8192, hidden=4096, vocab=32000, ignored=0.05, budget="default",
             dtype="bf16"),
        # the same loss at the largest size, without a memory limit
        dict(name="fused_linear_ce_large", kind="flce", rows=16384, hidden=4096, vocab=128256, ignored=0.05,
             budget="fastest", dtype="bf16"),
        # distillation behind two lm_heads under the default memory budget
        dict(name="fused_linear_jsd", kind="fljsd", rows=4096, hidden=4096, vocab=32000, ignored=0.05,
             budget="default", dtype="bf16"),
        # GRPO behind an lm_head under the default memory budget, prefix masks
        dict(name="fused_linear_grpo", kind="flgrpo", batch=4, seq=1024, hidden=4096, vocab=50257, beta=0.1,
             budget="default", dtype="bf16"),
    ]


def _log_int(rng, lo, hi):
    """An integer spread over the logarithm of [lo, hi]."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "norm", "norm", "rope", "glu", "ce", "ce", "grpo", "attn_res", "flce", "flce",
                       "fljsd", "flgrpo"])
    half = rng.choice(["bf16", "bf16", "fp16"])
    if kind == "decode":  # a few sequences to a small prefill
        return dict(kind=kind, tokens=_log_int(rng, 1, 256), hidden=rng.choice([1024, 2048, 4096, 5120, 8192]),
                    inter=rng.choice([11008, 14336, 28672]), dtype=half)
    if kind == "norm":
        return dict(kind=kind, add=rng.random() < 0.5, rows=_log_int(rng, 64, 16384),
                    hidden=rng.choice([1000, 1024, 2048, 4096, 5120, 8192]),
                    dtype=rng.choice(["fp32", "bf16", "bf16", "fp16"]))
    if kind == "rope":
        heads = rng.choice([8, 32, 64])
        return dict(kind=kind, batch=rng.randint(1, 8), seq=_log_int(rng, 33, 2048), heads=heads,
                    kv_heads=rng.choice([4, 8, heads]), head_dim=rng.choice([64, 128]),
                    dtype=rng.choice(["fp32", half]))
    if kind == "glu":
        return dict(kind=kind, act=rng.choice(["swiglu", "geglu"]), rows=_log_int(rng, 33, 8192),
                    inter=rng.choice([1001, 11008, 14336, 28672]), dtype=half)
    if kind == "ce":
        return dict(kind=kind, rows=_log_int(rng, 64, 8192), vocab=rng.choice([4096, 32000, 50257, 128256]),
                    ignored=rng.choice([0.0, 0.1, 0.4]), dtype=rng.choice(["fp32", half]))
    if kind == "grpo":
        return dict(kind=kind, batch=rng.randint(1, 16), seq=_log_int(rng, 65, 1024),
                    vocab=rng.choice([32000, 50257, 128256, 151936]), beta=rng.choice([0.0, 0.1]), dtype=half)
    if kind == "attn_res":
        return dict(kind=kind, blocks=rng.choice([2, 4, 8, 9, 16]), rows=_log_int(rng, 64, 8192),
                    hidden=rng.choice([1024, 2048, 4096]), dtype=half)
    hidden = rng.choice([1024, 2048, 4096])
    vocab = rng.choice([32000, 50257, 128256])
    budget = rng.choice(["default", "fastest"])
    if kind == "flgrpo":
        return dict(kind=kind, batch=rng.randint(1, 8), seq=_log_int(rng, 129, 1024), hidden=hidden, vocab=vocab,
                    beta=rng.choice([0.0, 0.1]), budget=budget, dtype="bf16")
    return dict(kind=kind, rows=_log_int(rng, 256, 8192), hidden=hidden, vocab=vocab, ignored=rng.choice([0.0, 0.05]),
                budget=budget, dtype="bf16")


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _budget(case):
    return "fastest" if case["budget"] == "fastest" else None


def _rope_tables(seq, dim, device):
    """fp32 cos and sin (1, seq, dim / 2) at base 500000."""
    inv = 1.0 / (500000.0 ** (torch.arange(0, dim, 2, dtype=torch.float32, device=device) / dim))
    ang = torch.outer(torch.arange(seq, dtype=torch.float32, device=device), inv)
    return ang.cos()[None].contiguous(), ang.sin()[None].contiguous()


def _lengths_mask(g, batch, length, device):
    """Prefix masks of valid lengths uniform in [length / 4, length]."""
    n = torch.randint(max(1, length // 4), length + 1, (batch,), generator=g, device=device)
    return (torch.arange(length, device=device)[None, :] < n[:, None]).to(torch.int32)


def _targets(g, rows, vocab, ignored, device):
    t = torch.randint(0, vocab, (rows,), generator=g, device=device)
    t[torch.rand(rows, generator=g, device=device) < ignored] = -100
    return t


def _old_logp(logits_of, ids, rows):
    """fp32 log-probs of the ids, a few sequences at a time (the rollout's own)."""
    return torch.stack([torch.log_softmax(logits_of(b).float(), -1).gather(-1, ids[b, :, None])[:, 0]
                        for b in range(rows)])


def prepare(case, seed):
    dev = torch.device("cuda")
    g = torch.Generator(device=dev)
    g.manual_seed(int(seed))
    dt = DTYPES[case["dtype"]]
    kind = case["kind"]

    def randn(*shape, scale=1.0, dtype=dt):
        t = torch.randn(*shape, generator=g, device=dev, dtype=torch.float32)
        return (t.mul_(scale) if scale != 1.0 else t).to(dtype)

    def leaf(t):
        return t.requires_grad_(True)

    s = dict(case)
    if kind == "decode":
        n, h = case["tokens"], case["hidden"]
        cos, sin = _rope_tables(2048, 128, dev)
        pos = torch.randint(0, 2048, (n,), generator=g, device=dev)
        s.update(x=randn(n, h), r=randn(n, h), w=(1 + randn(h, scale=0.02, dtype=torch.float32)).to(dt),
                 q=randn(n, 1, h // 128, 128).transpose(1, 2), k=randn(n, 1, 8, 128).transpose(1, 2),
                 cos=cos[0, pos][:, None].contiguous(), sin=sin[0, pos][:, None].contiguous(),
                 gate=randn(n, case["inter"]), up=randn(n, case["inter"]))
    elif kind == "norm":
        shape = (case["rows"], case["hidden"])
        s.update(x=leaf(randn(*shape)), w=leaf((1 + randn(shape[1], scale=0.02, dtype=torch.float32)).to(dt)),
                 dy=randn(*shape))
        if case["add"]:
            s.update(r=leaf(randn(*shape)), ds=randn(*shape))
    elif kind == "rope":
        b, t, d = case["batch"], case["seq"], case["head_dim"]
        cos, sin = _rope_tables(t, d, dev)
        s.update(q=leaf(randn(b, t, case["heads"], d).transpose(1, 2)),
                 k=leaf(randn(b, t, case["kv_heads"], d).transpose(1, 2)), cos=cos, sin=sin,
                 dq=randn(b, t, case["heads"], d).transpose(1, 2),
                 dk=randn(b, t, case["kv_heads"], d).transpose(1, 2))
    elif kind == "glu":
        shape = (case["rows"], case["inter"])
        s.update(a=leaf(randn(*shape)), b=leaf(randn(*shape)), dc=randn(*shape))
    elif kind == "ce":
        s.update(logits=leaf(randn(case["rows"], case["vocab"], scale=2.0)),
                 targets=_targets(g, case["rows"], case["vocab"], case["ignored"], dev))
    elif kind in ("grpo", "flgrpo"):
        B, T, V = case["batch"], case["seq"], case["vocab"]
        L = T - 1
        ids = torch.randint(0, V, (B, L), generator=g, device=dev)
        if kind == "grpo":
            logits = randn(B, T, V, scale=2.0)
            s.update(logits=leaf(logits))
            own = _old_logp(lambda b: logits.detach()[b, :L], ids, B)
        else:
            h, w = randn(B, T, case["hidden"]), randn(V, case["hidden"], scale=0.02)
            s.update(hidden=leaf(h), weight=leaf(w))
            own = _old_logp(lambda b: h.detach()[b, :L] @ w.detach().T, ids, B)
        s.update(ids=ids, adv=randn(B, dtype=torch.float32),
                 old=own + 0.05 * randn(B, L, dtype=torch.float32),
                 ref=own + 0.1 * randn(B, L, dtype=torch.float32) if case["beta"] else None,
                 mask=_lengths_mask(g, B, L, dev))
    elif kind == "attn_res":
        n, rows, d = case["blocks"], case["rows"], case["hidden"]
        s.update(v=leaf(randn(n, 1, rows, d)), wq=leaf(randn(d, scale=0.02)),
                 wn=leaf((1 + randn(d, scale=0.02, dtype=torch.float32)).to(dt)), dh=randn(1, rows, d))
    else:
        rows, h, V = case["rows"], case["hidden"], case["vocab"]
        s.update(hidden=leaf(randn(rows, h)), weight=leaf(randn(V, h, scale=0.02)),
                 targets=_targets(g, rows, V, case["ignored"], dev))
        if kind == "fljsd":
            s.update(t_hidden=randn(rows, h), t_weight=randn(V, h, scale=0.02))
    return s


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(s):
    kind, grad = s["kind"], torch.autograd.grad
    if kind == "decode":
        with torch.no_grad():
            y, res = hilda_fused_add_rms_norm(s["x"], s["r"], s["w"], EPS)
            q, k = hilda_rope(s["q"], s["k"], s["cos"], s["sin"])
            return y, res, q, k, hilda_swiglu(s["gate"], s["up"])
    if kind == "norm":
        if s["add"]:
            y, res = hilda_fused_add_rms_norm(s["x"], s["r"], s["w"], EPS)
            return (y, res) + grad([y, res], [s["x"], s["r"], s["w"]], [s["dy"], s["ds"]])
        y = hilda_rms_norm(s["x"], s["w"], EPS)
        return (y,) + grad([y], [s["x"], s["w"]], [s["dy"]])
    if kind == "rope":
        q, k = hilda_rope(s["q"], s["k"], s["cos"], s["sin"])
        return (q, k) + grad([q, k], [s["q"], s["k"]], [s["dq"], s["dk"]])
    if kind == "glu":
        c = (hilda_swiglu if s["act"] == "swiglu" else hilda_geglu)(s["a"], s["b"])
        return (c,) + grad([c], [s["a"], s["b"]], [s["dc"]])
    if kind == "ce":
        loss = hilda_cross_entropy(s["logits"], s["targets"])
        return (loss,) + grad([loss], [s["logits"]])
    if kind == "grpo":
        loss, kl, clip = hilda_grpo_loss(s["logits"], s["ids"], s["adv"], s["old"], s["ref"], s["mask"],
                                         beta=s["beta"])
        return (loss, kl, clip) + grad([loss], [s["logits"]])
    if kind == "attn_res":
        h = hilda_attn_res(s["v"], s["wq"], s["wn"], EPS)
        return (h,) + grad([h], [s["v"], s["wq"], s["wn"]], [s["dh"]])
    if kind == "flce":
        loss = hilda_fused_linear_cross_entropy(s["hidden"], s["weight"], s["targets"], workspace_budget=_budget(s))
        return (loss,) + grad([loss], [s["hidden"], s["weight"]])
    if kind == "fljsd":
        loss = hilda_fused_linear_jsd(s["hidden"], s["weight"], s["t_hidden"], s["t_weight"], s["targets"],
                                      workspace_budget=_budget(s))
        return (loss,) + grad([loss], [s["hidden"], s["weight"]])
    loss, kl, clip = hilda_fused_linear_grpo_loss(s["hidden"], s["weight"], s["ids"], s["adv"], s["old"], s["ref"],
                                             s["mask"], beta=s["beta"], workspace_budget=_budget(s))
    return (loss, kl, clip) + grad([loss], [s["hidden"], s["weight"]])


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def work(case):
    kind, es = case["kind"], SIZE[case["dtype"]]
    if kind == "decode":
        n, h = case["tokens"], case["hidden"]
        heads = h // 128 + 8
        return {"bytes": n * es * (4 * h + 2 * heads * 128 + 3 * case["inter"]) + h * es + n * 128 * 4,
                "flops": n * (5 * h + 4 * heads * 128 + 5 * case["inter"])}
    if kind == "norm":
        n, h = case["rows"], case["hidden"]
        return {"bytes": n * h * es * (7 if case["add"] else 4), "flops": n * h * (16 if case["add"] else 14)}
    if kind == "rope":
        rows = case["batch"] * case["seq"] * (case["heads"] + case["kv_heads"])
        return {"bytes": 4 * rows * case["head_dim"] * es, "flops": 6 * rows * case["head_dim"]}
    if kind == "glu":
        n = case["rows"] * case["inter"]
        return {"bytes": 6 * n * es, "flops": 16 * n}
    if kind == "ce":  # ignored rows are written as zeros and need no read
        n = case["rows"] * case["vocab"]
        return {"bytes": (2 - case["ignored"]) * n * es, "flops": 6 * n}
    if kind == "grpo":  # the masks keep 5 of 8 tokens on average
        n = case["batch"] * case["seq"] * case["vocab"]
        return {"bytes": 1.625 * n * es, "flops": 4 * n}
    if kind == "attn_res":  # blocks and dh read, h and dblocks written
        n = case["rows"] * case["hidden"]
        return {"bytes": (2 * case["blocks"] + 2) * n * es, "flops": 14 * case["blocks"] * n}
    h, V = case["hidden"], case["vocab"]
    if kind == "flgrpo":
        rows, live = case["batch"] * case["seq"], 0.625 * case["batch"] * (case["seq"] - 1)
    else:
        rows, live = case["rows"], (1 - case["ignored"]) * case["rows"]
    if kind == "fljsd":
        return {"bytes": es * (3 * rows * h + 3 * V * h), "flops": 8 * live * h * V}
    return {"bytes": es * (2 * rows * h + 2 * V * h), "flops": 6 * live * h * V}


# ---------------------------------------------------------------------------
# precision
# ---------------------------------------------------------------------------
def tolerance(case):
    """About four times the error measured against 64 bits: 2.9e-3 (bf16), 2.1e-4 (fp16, one rounding; 5e-4 with
    two), 6.5e-3 (fused-linear losses, bf16), 2e-7 (fp32; sums in another order differ by more)."""
    kind, dt = case["kind"], case["dtype"]
    if dt == "fp32":
        return {"rel": 1e-5, "max": 1e-3}
    if kind in ("flce", "fljsd", "flgrpo"):  # 16-bit logits, dlogits and (in the tight plans) partial sums
        return {"rel": 2e-2, "max": 0.5}
    if kind == "attn_res":  # keys rounded to 16 bits before the softmax over depth
        return {"rel": 1e-2, "max": 0.2}
    return {"rel": 1e-2 if dt == "bf16" else 1.5e-3, "max": 0.1 if dt == "bf16" else 0.02}


def _rms_norm64(x, w, dy):
    """(y, d out / d x without the residual's gradient, dw) in 64 bits."""
    rstd = torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS)
    xh = x * rstd
    m = dy * w
    return xh * w, rstd * (m - xh * (m * xh).mean(-1, keepdim=True)), (dy * xh).sum(0)


def _rope64(x, cos, sin):
    half = x.shape[-1] // 2
    a, b = x[..., :half], x[..., half:]
    c, s = cos.double()[:, None], sin.double()[:, None]
    return torch.cat((a * c - b * s, b * c + a * s), -1)


def _ce64(z, t):
    """(sum of the rows' losses, d sum / d z) of 64-bit logits; ignored rows (t < 0) give zero."""
    live = t >= 0
    at = t.clamp(min=0)[:, None]
    lp = torch.log_softmax(z, -1)
    loss = -(lp.gather(-1, at)[:, 0] * live).sum()
    d = lp.exp_()
    d.scatter_add_(-1, at, torch.full_like(at, -1, dtype=d.dtype))
    d.mul_(live[:, None])
    return loss, d


def _grpo64(s):
    """A function of one sequence's 64-bit logits: (its loss share, kl sum, clip sum, d loss / d logits)."""
    B = s["batch"]
    mask = s["mask"].double()
    lens = mask.sum(-1).clamp(min=1)

    def one(z, b):
        lp_all = torch.log_softmax(z, -1)
        at = s["ids"][b, :, None]
        lp = lp_all.gather(-1, at)[:, 0]
        ratio = torch.exp(lp - s["old"][b].double())
        A = s["adv"][b].double()
        l1, l2 = ratio * A, ratio.clamp(0.8, 1.2) * A
        loss = -torch.minimum(l1, l2)
        d = torch.where(l1 <= l2, -l1, torch.zeros_like(l1))
        kl = torch.zeros_like(lp)
        if s["beta"]:
            x = s["ref"][b].double() - lp
            kl = torch.exp(x) - x - 1
            loss = loss + s["beta"] * kl
            d = d + s["beta"] * (1 - torch.exp(x))
        clip = (((ratio < 0.8) & (A < 0)) | ((ratio > 1.2) & (A > 0))).double()
        w = mask[b] / (lens[b] * B)
        dz = lp_all.exp_().mul_(-(d * w)[:, None])
        dz.scatter_add_(-1, at, (d * w)[:, None])
        return (loss * w).sum(), (kl * mask[b]).sum(), (clip * mask[b]).sum(), dz

    return one


def _jsd64(zs, zt, live):
    """(sum of the rows' JSD at beta 1/2, d sum / d zs) of 64-bit logits."""
    X, Y = torch.log_softmax(zs, -1), torch.log_softmax(zt, -1)
    Q, P = X.exp(), Y.exp()
    logm = torch.log(0.5 * (P + Q))
    per = 0.5 * (P * (Y - logm)).sum(-1) + 0.5 * (Q * (X - logm)).sum(-1)
    dX = 0.5 * Q * (X - logm)
    d = dX - Q * dX.sum(-1, keepdim=True)
    return (per * live).sum(), d * live[:, None]


@torch.no_grad()
def exact(case, seed):
    s = prepare(case, seed)
    kind = case["kind"]
    if kind == "decode":
        res = s["x"].double() + s["r"].double()
        y = res * torch.rsqrt(res.square().mean(-1, keepdim=True) + EPS) * s["w"].double()
        gate = s["gate"].double()
        return (y, res, _rope64(s["q"].double(), s["cos"], s["sin"]), _rope64(s["k"].double(), s["cos"], s["sin"]),
                gate * torch.sigmoid(gate) * s["up"].double())
    if kind == "norm":
        x, w, dy = s["x"].double(), s["w"].double(), s["dy"].double()
        if not case["add"]:
            return _rms_norm64(x, w, dy)
        res = x + s["r"].double()
        y, dx, dw = _rms_norm64(res, w, dy)
        dx = dx + s["ds"].double()
        return y, res, dx, dx, dw
    if kind == "rope":
        out = [_rope64(s[n].double(), s["cos"], s["sin"]) for n in ("q", "k")]
        return tuple(out) + tuple(_rope64(s[n].double(), s["cos"], -s["sin"]) for n in ("dq", "dk"))
    if kind == "glu":
        a, b, dc = s["a"].double(), s["b"].double(), s["dc"].double()
        if case["act"] == "swiglu":
            sig = torch.sigmoid(a)
            act, dact = a * sig, sig * (1 + a * (1 - sig))
        else:
            c = math.sqrt(2.0 / math.pi)
            t = torch.tanh(c * (a + 0.044715 * a ** 3))
            act = 0.5 * a * (1 + t)
            dact = 0.5 * (1 + t) + 0.5 * a * (1 - t * t) * c * (1 + 3 * 0.044715 * a * a)
        return act * b, dc * b * dact, dc * act
    if kind == "ce":
        z, t = s["logits"].detach(), s["targets"]
        n = (t >= 0).sum().clamp(min=1)
        loss, dz = 0.0, torch.empty(z.shape, dtype=torch.float64, device=z.device)
        for i in range(0, z.shape[0], 1024):
            part, d = _ce64(z[i:i + 1024].double(), t[i:i + 1024])
            loss, dz[i:i + 1024] = loss + part, d / n
        return loss / n, dz
    if kind == "grpo":
        one, L = _grpo64(s), case["seq"] - 1
        z = s["logits"].detach()
        dz = torch.zeros(z.shape, dtype=torch.float64, device=z.device)
        loss = kl = clip = 0.0
        for b in range(case["batch"]):
            x, y, c, d = one(z[b, :L].double(), b)
            loss, kl, clip, dz[b, :L] = loss + x, kl + y, clip + c, d
        n = s["mask"].sum().clamp(min=1)
        return loss, kl / n if case["beta"] else None, clip / n, dz
    if kind == "attn_res":
        v, wq, wn, dh = (s[n].double() for n in ("v", "wq", "wn", "dh"))
        rstd = torch.rsqrt(v.square().mean(-1, keepdim=True) + EPS)
        xh = v * rstd
        a = torch.softmax((xh * (wn * wq)).sum(-1), 0)
        h = (a[..., None] * v).sum(0)
        da = (dh * v).sum(-1)
        ds = (a * (da - (a * da).sum(0, keepdim=True)))[..., None]
        S = (ds * xh).sum((0, 1, 2))
        dx = ds * (wn * wq)
        dv = a[..., None] * dh + rstd * (dx - xh * (dx * xh).mean(-1, keepdim=True))
        return h, dv, S * wn, S * wq
    w = s["weight"].detach().double()
    dw = torch.zeros_like(w)
    if kind == "flgrpo":
        one, L = _grpo64(s), case["seq"] - 1
        hid = s["hidden"].detach().double()
        dh = torch.zeros_like(hid)
        loss = kl = clip = 0.0
        for b in range(case["batch"]):
            x, y, c, d = one(hid[b, :L] @ w.T, b)
            loss, kl, clip = loss + x, kl + y, clip + c
            dh[b, :L] = d @ w
            dw += d.T @ hid[b, :L]
        n = s["mask"].sum().clamp(min=1)
        return loss, kl / n if case["beta"] else None, clip / n, dh, dw
    hid, t = s["hidden"].detach().double(), s["targets"]
    n = (t >= 0).sum().clamp(min=1)
    dh = torch.zeros_like(hid)
    loss = 0.0
    tw = s["t_weight"].double() if kind == "fljsd" else None
    for i in range(0, hid.shape[0], 1024):
        x, at = hid[i:i + 1024], t[i:i + 1024]
        if kind == "flce":
            part, d = _ce64(x @ w.T, at)
        else:
            part, d = _jsd64(x @ w.T, s["t_hidden"][i:i + 1024].double() @ tw.T, (at >= 0).double())
        loss = loss + part
        d /= n
        dh[i:i + 1024] = d @ w
        dw += d.T @ x
    return loss / n, dh, dw
