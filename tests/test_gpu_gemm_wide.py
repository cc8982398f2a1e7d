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
