"""GPU: the substitution and the residual of several right-hand sides at once.

With no correction allowed, hpl_solve_rhs64 returns the FP32 substitution's
solution as it is; it is compared with an FP64 substitution with the same
(downloaded) factor.  The bound is 1e-5 of the solution: the matrices are
diagonally dominant, so L and U are within a small factor of a diagonal
matrix and the FP32 substitution's error is a few units of 6e-8 times the
square root of the number of terms.  The residuals that the refinement
reports are compared with FP64 numpy to 1e-12 of ||M|| ||x|| + ||b||, some
5000 times the rounding of an FP64 sum.
"""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,B,prec,nrhs", [
    (256, 256, "fp32", 2),    # one block
    (288, 32, "fp32", 16),    # the narrowest block, two waves of rows
    (320, 64, "fp32", 3),
    (1024, 128, "fp32", 5),
    (1536, 256, "fp32", 15),
    (1024, 256, "bf16", 16),
    (1024, 512, "fp32", 4),   # no whole inverses: the 32 x 32 solves
    (544, 32, "fp32", 1),
])
def test_substitution_and_residual(ctx, n, B, prec, nrhs):
    print(f"rhs n={n} B={B} {prec} nrhs={nrhs}", flush=True)
    rng = np.random.default_rng(n + nrhs)
    a = (rng.random((n, n), np.float32) - np.float32(0.5)).astype(np.float32)
    a[np.arange(n), np.arange(n)] += np.float32(n)
    b = rng.uniform(-1.0, 1.0, (n, nrhs))
    ctx.keep_original(True)
    ctx.upload(a)
    ctx.gefa_dev(B, prec)
    x, res = ctx.solve_rhs64(b, max_iter=0, check=False)
    f, _ = ctx.download(matrix=True, solution=False)
    ctx.keep_original(False)
    x = x.reshape(n, nrhs)
    for j in range(nrhs):
        ref = O.gesl_nopvt_f64(f.astype(np.float64), b[:, j].copy())
        assert np.max(np.abs(x[:, j] - ref)) <= 1e-5 * np.max(np.abs(ref)), j
    m = a.astype(np.float64).T
    r = b - m @ x
    norm_m = np.max(np.sum(np.abs(m), axis=1))
    for j in range(nrhs):
        scale = norm_m * np.max(np.abs(x[:, j])) + np.max(np.abs(b[:, j]))
        assert abs(res[j]["residual_inf"] - np.max(np.abs(r[:, j]))) <= 1e-12 * scale, j
        assert res[j]["norm_a"] == pytest.approx(norm_m, rel=1e-12)
        assert res[j]["norm_x"] == np.max(np.abs(x[:, j]))
        assert res[j]["norm_b"] == np.max(np.abs(b[:, j]))
