"""CPU tier: what the fused-linear planner may not change when its cost model follows faster kernels."""
import ctypes
import os

import pytest

from kernels import _lib

needs_lib = pytest.mark.skipif(not os.path.exists(_lib.LIB_PATH), reason="library not built")

BF16, F16, F32 = 2, 1, 0
M256 = 256 << 20

# (op, BT, H, V, budget, dtype, most roundings of dW and of dX to 16 bits between partial sums). 0, 0: fp32 sums.
SUMS = [
    # few rows: vocabulary tiles with an fp32 dX, not short row chunks with dW in the output
    ("ce", 320, 2048, 128256, 0, BF16, 0, 0), ("ce", 384, 2048, 128256, 0, BF16, 0, 0),
    ("ce", 522, 2048, 128256, 0, BF16, 0, 0), ("ce", 640, 1024, 128256, 0, BF16, 0, 0),
    ("ce", 850, 2048, 32000, 0, BF16, 0, 0), ("ce", 1152, 1024, 50257, 0, BF16, 0, 0),
    ("ce", 3456, 512, 8000, 0, BF16, 0, 0), ("ce", 4309, 4096, 32000, 0, BF16, 0, 0),
    ("ce", 5504, 4096, 32000, M256, BF16, 0, 0), ("ce", 10496, 4096, 32000, M256, BF16, 0, 0),
    ("ce", 11008, 4096, 32000, M256, BF16, 0, 0), ("ce", 15872, 512, 8000, 0, BF16, 0, 0),
    # fp16
    ("ce", 1408, 5120, 32000, 0, F16, 0, 0), ("ce", 14976, 1024, 8000, 0, F16, 0, 0),
    ("ce", 15744, 1024, 8000, 0, F16, 0, 0), ("ce", 9216, 1024, 32000, 0, F16, 0, 15),
    ("ce", 10496, 2048, 128256, 0, F16, 0, 35),
    # 16-bit sums that were, in no more steps
    ("ce", 4736, 2048, 8000, 0, BF16, 0, 1), ("ce", 4992, 2048, 128256, 0, BF16, 0, 31),
    ("ce", 8192, 4096, 32000, 0, BF16, 0, 7), ("ce", 9216, 1024, 128256, 0, BF16, 0, 62),
    ("ce", 9216, 5120, 128256, 0, BF16, 0, 20), ("ce", 16384, 4096, 128256, 0, BF16, 0, 31),
    # one deferred dW GEMM or an fp32 accumulator, not two chunks in the output
    ("jsd", 1920, 512, 50257, M256, BF16, 0, 0), ("jsd", 2176, 512, 8000, 0, BF16, 0, 0),
    ("jsd", 2176, 2048, 50257, 0, BF16, 0, 0), ("jsd", 3072, 2048, 32000, 0, BF16, 0, 0),
    ("jsd", 8192, 4096, 65536, 0, BF16, 0, 0), ("jsd", 13696, 1024, 128256, 0, BF16, 12, 0),
    ("grpo", 3456, 512, 8000, 0, BF16, 0, 0), ("grpo", 4096, 512, 50257, M256, BF16, 0, 0),
    ("grpo", 6656, 512, 8000, 0, BF16, 0, 0),
]


def _plan(op, BT, H, V, budget, dtype, chunk=0):
    info = (ctypes.c_int64 * 8)()
    lib = _lib.load()
    if op == "ce":
        rc = lib.hk_fused_linear_cross_entropy_plan(BT, H, V, chunk, budget, dtype, 1, None, None, info)
    elif op == "jsd":
        rc = lib.hk_fused_linear_jsd_plan(BT, H, H, V, chunk, budget, dtype, 1, 1, None, None, None, None, info)
    else:
        rc = lib.hk_fused_linear_grpo_plan(1, BT - 1, H, V, chunk, budget, dtype, 1, None, None, info)
    _lib.check(rc, "plan")
    return list(info)


@needs_lib
@pytest.mark.parametrize("op,BT,H,V,budget,dtype,dw,dx", SUMS)
def test_gradients_are_rounded_no_more_often(op, BT, H, V, budget, dtype, dw, dx):
    """Each gradient's partial sums are rounded to 16 bits at most as often as stated."""
    _, n, mode, *_ = _plan(op, BT, H, V, budget, dtype)
    steps = {2: (n - 1, 0), 4: (0, n - 1)}.get(mode, (0, 0))
    assert steps[0] <= dw and steps[1] <= dx, (mode, n)


# (BT, H, V, chunk, most bytes): unlimited budget, capped chunks
CAPPED = [
    (51188, 8, 150497, 64, 27740928), (65536, 512, 128256, 2048, 958726656), (65536, 512, 256000, 2048, 1874395648),
    (16384, 512, 32000, 2048, 267584000), (2176, 1024, 8000, 2048, 136162816), (2176, 5120, 128256, 2048, 928271872),
    (4736, 1024, 128256, 2048, 2100510208), (896, 4096, 32000, 2048, 173397504),
    (16384, 4096, 128256, 2048, 6098027008),
]


@needs_lib
@pytest.mark.parametrize("BT,H,V,chunk,most", CAPPED)
def test_capped_chunks_bound_the_workspace(BT, H, V, chunk, most):
    """A caller that caps the chunk also bounds the workspace when the budget does not: no form is forced that keeps
    every chunk's D^T where an accumulator of a fraction of its size does."""
    C, *_, total, _ = _plan("ce", BT, H, V, -1, BF16, chunk)
    assert C <= chunk and total <= most


@needs_lib
@pytest.mark.parametrize("BT,H,V,budget", [(8, 64, 20_000_000, M256), (64, 256, 4_300_000, M256),
                                           (64, 256, 8_000_000, M256), (64, 256, 20_000_000, 1 << 30),
                                           (8, 64, 100_000_000, 1 << 30), (1024, 64, 100_000_000, 0)])
def test_tiles_stay_within_a_gemm_panel(BT, H, V, budget):
    """256 rows of a tile buffer stay below the 2 GiB a GEMM's buffer can address; wider plans fail at launch."""
    cols, _, mode, *_ = _plan("ce", BT, H, V, budget, BF16)
    assert mode in (3, 4) and 256 * cols * 2 < 0x7FF00000
