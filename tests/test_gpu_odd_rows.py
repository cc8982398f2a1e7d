"""CrossEntropy and GRPO on logit rows that are not 16-byte aligned: odd vocabularies, and an odd base address.

The register-resident row forms take such rows with unaligned 16-byte vectors, the row's last vector moved left to end
with the row, so that some elements are held by two lanes: each has to count once, and the target's gradient has to
win in both. Lengths: one vector and one element either side of it, the forms' spans and capacities plus or minus one
element, real odd vocabularies, and one past the longest form; targets among the row's last elements and its first.

Tolerances are those of the aligned rows of the same kernels (the arithmetic is the same; only which lane sums which
element differs): fp64 oracle, one rounding of the gradient to its dtype; 1e-5 for fp32.
"""
import math

import pytest
import torch

import oracle
from _util import assert_close, gpu, rel_fro, tol

from kernels import hilda_cross_entropy, hilda_grpo_loss

pytestmark = pytest.mark.gpu

BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32

# (V, elements by which the base address is off a 16-byte boundary, rows, dtype)
ROWS = [
    (7, 0, 300, BF16), (8, 1, 300, BF16), (9, 0, 3000, BF16), (15, 3, 300, F16), (5, 0, 3000, F32), (3, 0, 40, F32),
    (2047, 0, 2200, BF16), (2048, 1, 300, BF16), (2049, 0, 2200, BF16), (4095, 5, 300, F16), (8193, 0, 300, BF16),
    (16385, 0, 300, BF16), (24577, 7, 300, BF16), (32001, 0, 300, F16), (32769, 0, 300, BF16), (50257, 0, 700, BF16),
    (50257, 0, 40, F32), (65535, 0, 40, BF16), (65537, 0, 40, BF16), (128257, 0, 300, BF16), (151935, 1, 300, BF16),
    (196607, 0, 40, BF16), (196609, 0, 8, BF16),
]


def _logits(rows, V, off, dtype, dev):
    g = torch.Generator(device=dev).manual_seed(V + off)
    buf = (2 * torch.randn(off + rows * V, generator=g, device=dev)).to(dtype)
    ids = torch.randint(0, V, (rows,), generator=g, device=dev)
    # the last elements (held twice) and the first ones
    edge = torch.arange(rows, device=dev) % 18
    ids = torch.where(edge < 9, (V - 1 - edge).clamp_min(0), ids)
    ids = torch.where(edge == 17, torch.zeros_like(ids), ids)
    return buf[off:].view(rows, V), ids


@pytest.mark.parametrize("V,off,rows,dtype", ROWS)
def test_cross_entropy_odd_rows(V, off, rows, dtype):
    dev = gpu()
    lg, t = _logits(rows, V, off, dtype, dev)
    t[3::11] = -100
    print(f"CE odd rows V={V} off={off} rows={rows} {dtype}", flush=True)
    lg.requires_grad_(True)
    loss = hilda_cross_entropy(lg, t, -100, "none")
    (grad,) = torch.autograd.grad(loss, lg, torch.ones(rows, device=dev))
    sel = torch.cat([torch.arange(min(rows, 18)), torch.arange(max(rows - 18, 0), rows)])
    ts = t.cpu()[sel]
    (l_ref,), (d_ref,) = oracle.fwd_bwd(lambda z: oracle.cross_entropy_ref(z, ts, -100, "none"),
                                        [lg.detach().cpu()[sel]], [torch.ones(len(sel))], dtype=torch.float64)
    lt = dict(rtol=1e-5, atol=1e-5) if dtype == F32 else dict(rtol=2e-3, atol=2e-3)
    assert_close(loss.cpu()[sel], l_ref, name="loss", **lt)
    assert_close(grad.cpu()[sel], d_ref, name="dlogits", **tol(dtype))
    assert rel_fro(grad.cpu()[sel], d_ref.to(dtype)) < (1e-5 if dtype == F32 else 1e-2)
    assert torch.count_nonzero(grad[t == -100]).item() == 0
    # every row: a softmax minus its one-hot sums to 0 (the bound of the aligned rows' test)
    sums = grad[t != -100].float().sum(-1)
    assert sums.abs().max().item() < (1e-4 if dtype == F32 else 2e-2)


@pytest.mark.parametrize("V,off,rows,dtype", ROWS)
def test_grpo_odd_rows(V, off, rows, dtype):
    dev = gpu()
    B = 2
    L = rows // B - 1
    lg, ids = _logits(B * (L + 1), V, off, dtype, dev)
    lg, ids = lg.view(B, L + 1, V), ids.view(B, L + 1)[:, :L].contiguous()
    g = torch.Generator().manual_seed(V)
    adv = torch.randn(B, generator=g)
    old = -math.log(V) + 0.5 * torch.randn(B, L, generator=g)
    ref = -math.log(V) + 0.5 * torch.randn(B, L, generator=g)
    mask = (torch.arange(L)[None, :] < torch.tensor([[L], [max(L // 2, 1)]])).to(torch.int32)
    tail = (1.0, 0.1, 0.2, 0.2)
    print(f"GRPO odd rows V={V} off={off} rows={rows} {dtype}", flush=True)
    lg.requires_grad_(True)
    args = (ids, adv.to(dev), old.to(dev), ref.to(dev), mask.to(dev), *tail)
    loss, kl, clip = hilda_grpo_loss(lg, *args)
    (grad,) = torch.autograd.grad(loss, lg)
    with torch.no_grad():
        infer = hilda_grpo_loss(lg.detach(), *args)
    # the forward-only kernel reduces exactly as the gradient kernel does
    assert all(torch.equal(a, b.detach()) for a, b in zip(infer, (loss, kl, clip)))
    assert torch.count_nonzero(grad[:, -1]).item() == 0
    assert torch.count_nonzero(grad[:, :-1][mask.to(dev) == 0]).item() == 0
    # the oracle on each sequence's leading positions alone would change its mean: take the whole (small) ones
    if rows * V <= 1 << 24:
        f64 = lambda x: x.to(torch.float64)
        z = f64(lg.detach().cpu()).requires_grad_(True)
        lo, _, _ = oracle.grpo_loss_ref(z, ids.cpu(), f64(adv), f64(old), f64(ref), mask, *tail)
        lo.backward()
        assert math.isclose(loss.item(), lo.item(), rel_tol=2e-3, abs_tol=2e-3)
        s = B * float(mask.sum(1).max())  # a live row's gradient at unit scale
        assert_close(grad.float() * s, z.grad * s, name="grad", **tol(dtype))
    # every live row sums to 0 but for the rounding of its entries to their dtype (half an ulp, up to 2^-8 or 2^-11 of
    # each; fp16 may also be subnormal, 2^-25 each) and the 1e-5 of the fp32 arithmetic
    live = grad[:, :-1][mask.to(dev) != 0].double()
    half_ulp = {BF16: 2.0 ** -8, F16: 2.0 ** -11, F32: 0.0}[dtype]
    bound = (half_ulp + 1e-5) * live.abs().sum(-1) + (V * 2.0 ** -25 if dtype == F16 else 0.0)
    assert (live.sum(-1).abs() <= bound).all()
