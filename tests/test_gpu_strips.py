"""GPU: the strip solves, one workgroup per 32 vectors with the blocks dealt out
to waves, and beyond 12288 vectors a side one wave per 32.

Orders of two and three blocks (the smallest strips) against gefa_ref_nopvt, at
the tolerance of the other factor comparisons; orders whose first steps lie
beyond the limit and whose later ones do not by the FP64 backward error of the
refined solution, which no wrong strip reaches.
"""
import os

import numpy as np
import pytest

from hpcc_fpga_amd import Context
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B", [32, 64, 128, 256])
@pytest.mark.parametrize("blocks", [2, 3])
def test_smallest_strips(ctx, B, blocks):
    print(f"strips n={blocks * B} B={B}", flush=True)
    a, _, _, _ = O.generate_ref(blocks * B, seed=B + blocks)
    f = a.copy()
    ctx.gefa(f, B)
    ref = O.gefa_nopvt(a)
    assert np.max(np.abs(f - ref)) <= 2e-5 * np.max(np.abs(ref))


@pytest.mark.parametrize("B,prec", [(256, "fp32"), (128, "fp32"), (256, "fp8"), (128, "fp16")])
def test_both_sides_of_the_limit(ctx, B, prec):
    n = 12288 + 2 * B
    print(f"strips n={n} B={B} {prec}", flush=True)
    ctx.keep_original(True)
    try:
        ctx.generate(n, 1, 11, 1.01)
        r = ctx.solve_ir(B, prec, max_iter=50)
    finally:
        ctx.keep_original(False)
    assert r["converged"]


@pytest.mark.parametrize("n,B", [(16384, 256), (16640, 256)])
def test_both_sides_of_the_bf16_rule(ctx, n, B):
    """BF16 strips by the recurrence up to order 16384, by inverses beyond."""
    print(f"strips n={n} B={B} bf16", flush=True)
    ctx.keep_original(True)
    try:
        ctx.generate(n, 1, 11, 1.01)
        r = ctx.solve_ir(B, "bf16", max_iter=50)
    finally:
        ctx.keep_original(False)
    assert r["converged"]


@pytest.mark.parametrize("B", [64, 128, 256])
def test_strips_by_inverse_at_a_small_order(B):
    """The rule's other side forced at a small order: step 0's strips, which no
    update precedes, to the split product's accuracy (about 2^-17 of the terms,
    ten times that allowed)."""
    n = 4 * B
    print(f"strips by inverse n={n} B={B}", flush=True)
    a, _, _ = O.generate_sized(n, 5, 0)[:3]
    ref = O.gefa_nopvt(a)
    os.environ["HPL_STRIP_SOLVE"] = "inverse"
    try:
        c = Context(0)
    finally:
        os.environ.pop("HPL_STRIP_SOLVE", None)
    try:
        c.upload(a)
        c.gefa_dev(B, "bf16")
        f, _ = c.download(matrix=True, solution=False)
    finally:
        c.close()
    r = np.concatenate([ref[:B, B:].ravel(), ref[B:, :B].ravel()])
    g = np.concatenate([f[:B, B:].ravel(), f[B:, :B].ravel()])
    assert np.max(np.abs(g - r)) <= 10 * 2.0 ** -17 * np.max(np.abs(r))
