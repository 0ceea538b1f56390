"""GPU: partial pivoting where the panel's split over workgroups changes.

A panel of m rows takes 64 rows per workgroup up to m = 8192 and more beyond,
so one factorisation of a larger order goes through several splits.  The
oracle cannot factorise these orders in test time; a wrong row exchange or
multiplier anywhere leaves a factor that does not refine, so the refined
solution is checked against the FP64 backward error, recomputed on the host.
Below that, orders that leave the last workgroup a few rows are compared with
gefa_ref's restatement, pivots exactly.
"""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,B", [(8448, 256), (8256, 64)])
def test_split_changes_within_a_factorisation(ctx, n, B):
    print(f"pivoted n={n} B={B}", flush=True)
    ctx.keep_original(True)
    ctx.set_pivoting(True)
    try:
        ctx.generate(n, 2, 17)
        a, _ = ctx.download(matrix=True, solution=False)
        _, b, _ = ctx.download_vectors()
        r = ctx.solve_ir(B, "fp32", max_iter=20)
        x = ctx.download_solution64()
        ipvt = ctx.pivots()
    finally:
        ctx.set_pivoting(False)
        ctx.keep_original(False)
    assert r["converged"]
    assert np.all(ipvt >= np.arange(n)) and np.all(ipvt < n)
    res = b.copy()
    norm = np.zeros(n)
    for j in range(0, n, 1024):  # M = a^T: column sums over stored rows
        part = a[j:j + 1024].astype(np.float64)
        res -= part.T @ x[j:j + 1024]
        norm += np.abs(part).sum(axis=0)
    berr = np.max(np.abs(res)) / (np.max(norm) * np.max(np.abs(x)) + np.max(np.abs(b)))
    assert berr <= 1e-14 * n


@pytest.mark.parametrize("n,B", [(96, 32), (160, 32), (224, 32), (448, 64), (576, 64)])
def test_short_last_workgroup(ctx, n, B):
    print(f"pivoted n={n} B={B}", flush=True)
    rng = np.random.default_rng(n)
    a = (rng.random((n, n), np.float32) - np.float32(0.5)).astype(np.float32)
    f = a.copy()
    ipvt, _ = ctx.gefa_pvt(f, B)
    f_ref, ipvt_ref = O.gefa_pvt(a)
    assert np.array_equal(ipvt, ipvt_ref)
    # the first panel's columns (stored rows) bit for bit, the rest to the
    # rounding of another summation order
    assert np.array_equal(f[:B].view(np.uint32), f_ref[:B].view(np.uint32))
    assert np.max(np.abs(f - f_ref)) <= 1e-3 * np.max(np.abs(f_ref))


@pytest.mark.parametrize("n,B", [(32, 32), (96, 32), (320, 64), (512, 256)])
@pytest.mark.parametrize("nrhs", [1, 3, 16])
def test_substitution_in_blocks_of_32(ctx, n, B, nrhs):
    print(f"pivoted n={n} B={B} nrhs={nrhs}", flush=True)
    ctx.keep_original(True)
    ctx.set_pivoting(True)
    try:
        ctx.generate(n, 2, n)
        a, _ = ctx.download(matrix=True, solution=False)
        ctx.gefa_dev(B)
        b = np.random.default_rng(n).random((n, nrhs)) - 0.5
        x, res = ctx.solve_rhs64(b)
    finally:
        ctx.set_pivoting(False)
        ctx.keep_original(False)
    M = a.astype(np.float64).T
    r = np.abs(b - M @ x).max(axis=0)
    scale = np.abs(M).sum(axis=1).max() * np.abs(x).max(axis=0) + np.abs(b).max(axis=0)
    assert all(q["converged"] for q in res)
    assert np.all(r <= 1e-14 * n * scale)
