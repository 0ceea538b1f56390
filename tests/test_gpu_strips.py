"""GPU: the strip solves, one workgroup per 32 vectors with the blocks dealt out
to waves, and beyond 12288 vectors a side one wave per 32.

Orders of two and three blocks (the smallest strips) against gefa_ref_nopvt, at
the tolerance of the other factor comparisons; orders whose first steps lie
beyond the limit and whose later ones do not by the FP64 backward error of the
refined solution, which no wrong strip reaches.
"""
import numpy as np
import pytest

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
