"""The 16-bit GEMM kernel at the edges of its tiles, stages and splits, through FusedLinearCE.

Every layout the fused-linear plans ask of it: logits (both operands K-contiguous), dX with W^T (both K-contiguous)
and with W MN-contiguous, dW with D^T X^T (both K-contiguous), with D MN-contiguous, and both MN-contiguous (the
vocabulary tiles). Shapes: one row, a tile less or more by one, one to three 64-deep stages (an odd count ends in a
stage of zeros), a K that is no whole number of stages, a short chunk whose dX GEMM splits K.

Against the fp64 oracle on the same inputs, its logits rounded to 16 bits as the GEMM returns them. A gradient entry
then carries the rounding of each dlogit and its own (2^-9 in bf16, each): rtol 1.6e-2, atol 1e-2 at unit scale, 1e-2
in the Frobenius norm. (The vocabulary tiles that sum dX in the 16-bit output add one rounding a tile.)
"""
import pytest
import torch

import oracle
from _util import assert_close, gpu, rel_fro, tol

pytestmark = pytest.mark.gpu

SHAPES = [(1, 64, 8), (255, 128, 257), (257, 192, 255), (70, 320, 520), (300, 1000, 264), (72, 256, 4096)]
FORMS = ["out,wt,dt", "out,wmn,dmn", "vtile,acc,256", "vtile,out,256"]


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("BT,H,V", SHAPES)
def test_wide_gemm_edges(BT, H, V, dtype, form, monkeypatch):
    import kernels.fused_linear_cross_entropy as fl

    g = torch.Generator().manual_seed(BT + H + V)
    h = torch.randn(BT, H, generator=g).to(dtype)
    w = (torch.randn(V, H, generator=g) / H ** 0.5).to(dtype)
    t = torch.randint(0, V, (BT,), generator=g)
    t[1::7] = -100
    # logits in the compute dtype, as the GEMM returns them
    (l_ref,), (dh_ref, dw_ref) = oracle.fwd_bwd(
        lambda a, b: oracle.cross_entropy_ref((a @ b.T).to(dtype).double(), t, -100, "sum"), [h, w],
        dtype=torch.float64)
    monkeypatch.setenv("HILDA_FL_FORM", form)
    dev = gpu()
    print(f"wide gemm {BT}x{H}x{V} {dtype} {form}", flush=True)
    loss, gi, gw, _ = fl.fused_linear_cross_entropy_forward(h.to(dev), w.to(dev), t.to(dev), -100, "sum",
                                                            compute_grad=True, workspace_budget=-1)
    tt = tol(dtype)
    assert_close(loss, l_ref, name="loss", rtol=2e-3, atol=2e-3)
    assert_close(gi, dh_ref, name="dhidden", **tt)
    assert_close(gw, dw_ref, name="dweight", **tt)
    assert rel_fro(gi, dh_ref) < 1e-2 and rel_fro(gw, dw_ref) < 1e-2
    assert torch.count_nonzero(gi[(t == -100).to(dev)]).item() == 0


def _check_sums(BT, H, V, dtype, form, monkeypatch, chunk=8192):
    """A forced form against the fp64 oracle, each gradient entry within the rounding of its terms: with u the unit
    roundoff (2^-8 in bf16, 2^-11 in fp16), every dlogit is rounded once (u; fp16 also 2^-25 where subnormal), the
    entry once and once more for each partial sum before the last (n of them): (n + 2) u sum |d| |w|. One u more for
    logits that an fp32 sum rounds to the other neighbour (about one in 10^4) and for the fp32 arithmetic."""
    import kernels.fused_linear_cross_entropy as fl

    dev = gpu()
    g = torch.Generator(device=dev).manual_seed(BT + H + V)
    h = torch.randn(BT, H, generator=g, device=dev).to(dtype)
    w = (torch.randn(V, H, generator=g, device=dev) / H ** 0.5).to(dtype)
    t = torch.randint(0, V, (BT,), generator=g, device=dev)
    t[1::7] = -100
    hd, wd = h.double(), w.double()
    z = (hd @ wd.T).to(dtype).double().requires_grad_(True)  # logits in the compute dtype, as the GEMM returns them
    l_ref = oracle.cross_entropy_ref(z, t, -100, "sum")
    (d,) = torch.autograd.grad(l_ref, z)
    monkeypatch.setenv("HILDA_FL_FORM", form)
    n = fl.fused_linear_cross_entropy_plan(BT, H, V, dtype, True, chunk, -1)["chunks"]
    print(f"wide gemm {BT}x{H}x{V} {dtype} {form} chunk {chunk}: {n}", flush=True)
    loss, gi, gw, _ = fl.fused_linear_cross_entropy_forward(h, w, t, -100, "sum", compute_grad=True, chunk=chunk,
                                                            workspace_budget=-1)
    assert_close(loss, l_ref, name="loss", rtol=2e-3, atol=2e-3)
    u = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    tiny = 2.0 ** -25 if dtype == torch.float16 else 0.0
    for name, got, ref, terms, rows in (("dhidden", gi, d @ wd, d.abs() @ wd.abs(), wd.abs().sum(0)),
                                        ("dweight", gw, d.T @ hd, d.T.abs() @ hd.abs(), hd.abs().sum(0))):
        err = (got.double() - ref).abs() - (n + 3) * u * terms - tiny * rows - 2 * tiny
        assert err.max().item() <= 0, (name, err.max().item())
        assert rel_fro(got, ref) < 1e-2, name
    assert torch.count_nonzero(gi[t == -100]).item() == 0


# More tiles than CUs, so that workgroups of the persistent kernel take a second one: in the logits GEMM (4 x 67
# tiles, 3 stages), in dW (67 x 4, ragged both ways, over row chunks too: every accumulating epilogue), in dX (17 x 17
# over 9 stages, and over tiles of 4, 4 and 1) and in a split dX (136 tiles, 4 splits). Ignored rows cut M and K on the
# device.
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("BT,H,V,chunk,form", [
    (1000, 192, 17000, 8192, "out,wt,dt"), (1000, 192, 17000, 8192, "out,wmn,dmn"),
    (150, 1000, 17100, 8192, "out,wt,dt"), (150, 1000, 17100, 64, "out,wmn,dmn"),
    (150, 1000, 17100, 64, "acc,wt,dmn"), (150, 1000, 17100, 64, "defer,wt,dt"),
    (4200, 4104, 520, 8192, "out,wt,dt"), (4200, 4104, 520, 8192, "out,wmn,dmn"),
    (4200, 4104, 520, 0, "vtile,acc,256"), (4200, 4104, 520, 0, "vtile,out,256"),
    (2000, 4104, 4200, 8192, "out,wmn,dmn"),
])
def test_wide_gemm_second_tiles(BT, H, V, chunk, form, dtype, monkeypatch):
    _check_sums(BT, H, V, dtype, form, monkeypatch, chunk)


# Tiles wider than 8192 columns, as the planner takes them for few rows: a ragged last tile, one as wide as the
# vocabulary, a hidden size that is padded.
@pytest.mark.parametrize("dx", ["acc", "out"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("BT,H,V,Vt", [(1, 64, 20001, 10240), (40, 72, 32000, 16384), (9, 67, 50257, 16384),
                                       (300, 128, 20001, 20224), (257, 64, 33000, 32768)])
def test_wide_vocab_tiles(BT, H, V, Vt, dtype, dx, monkeypatch):
    _check_sums(BT, H, V, dtype, f"vtile,{dx},{Vt}", monkeypatch, 0)
