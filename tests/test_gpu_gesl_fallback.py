"""GPU: substitutions whose single launch cannot hold all its workgroups at once.

The single-launch substitutions wait for each other's workgroups with a bound.
Where a wait gives up -- here with HPL_GESL_SPIN=0, at the first value that is
not there yet -- every workgroup leaves and the call solves again launch after
launch, from the untouched right-hand side.  HPL_GESL_GROUPS selects that path
from the start.
"""
import os

import numpy as np
import pytest
import torch  # before the library: one HIP runtime for both

from hpcc_fpga_amd import Context
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _env(monkeypatch, env):
    for k in [k for k in os.environ if k.startswith("HPL_")]:
        monkeypatch.delenv(k)
    for k, v in env.items():
        monkeypatch.setenv(k, v)


@pytest.mark.parametrize("env", [{}, {"HPL_GESL_GROUPS": "1"}, {"HPL_GESL_SPIN": "0"}])
@pytest.mark.parametrize("n", [64, 128, 640, 1024])
def test_fp64(monkeypatch, env, n):
    # every path keeps gesl_ref_nopvt's order of operations: the same bits
    print(f"f64 gesl {env} n={n}", flush=True)
    _env(monkeypatch, env)
    A, b = O.generate_ref_f64(n, seed=3)
    F = O.gefa_nopvt_f64(A)
    ref = O.gesl_nopvt_f64(F, b)
    with Context(0) as c:
        for _ in range(2):
            x = b.copy()
            c.gesl_f64(F, x)
            assert np.array_equal(x.view(np.uint64), ref.view(np.uint64))


@pytest.mark.parametrize("n,B,pivot", [(2048, 256, False), (1152, 128, False), (1088, 64, False),
                                       (544, 32, False), (576, 64, True), (2048, 256, True)])
def test_fp32(monkeypatch, n, B, pivot):
    """Giving up ends in the launches per block: the bits of a call that starts there
    (one workgroup cannot own more than 16 slices of 64, or 32, entries)."""
    g = np.random.default_rng(n + B)
    a = (g.random((n, n)) - 0.5).astype(np.float32)
    if not pivot:
        a[np.arange(n), np.arange(n)] += n
    b = g.uniform(-1, 1, n)
    out = {}
    for name, env in (("groups", {"HPL_GESL_GROUPS": "1"}), ("spin", {"HPL_GESL_SPIN": "0"})):
        print(f"fp32 gesl {env} n={n} B={B} pivot={pivot}", flush=True)
        _env(monkeypatch, env)
        with Context(0) as c:
            c.keep_original(True)
            c.set_pivoting(pivot)
            c.upload(a)
            c.upload_rhs64(b)
            c.gefa_dev(B)
            c.gesl_dev()
            x = c.download(matrix=False)[1]
            c.solve_ir(B, "fp32", tol=1e-15)
            r = c.download_solution64()
            c.solve_gmres(B, "fp32", tol=1e-15)
            out[name] = (x, r, c.download_solution64(), c.solve_rhs64(b)[0],
                         c.solve_rhs64(np.stack([b, -2.0 * b[::-1], b ** 2], axis=1))[0])
    for p, q in zip(out["groups"], out["spin"]):
        assert np.all(np.isfinite(p)) and np.array_equal(p, q)
    ref = np.linalg.solve(a.T.astype(np.float64), b)
    assert np.max(np.abs(out["spin"][1] - ref)) <= 1e-9 * np.max(np.abs(ref))


@pytest.mark.parametrize("n", [544, 1088, 2048])
def test_noalloc_shows_that_it_gave_up(monkeypatch, n):
    """hpl_gesl_noalloc only enqueues work and cannot solve again: NaN in x instead."""
    print(f"noalloc n={n}", flush=True)
    a, b, _, _ = O.generate_ref(n, seed=n)
    f = O.gefa_nopvt(a)
    F = torch.from_numpy(f).cuda()
    with Context(0) as c:
        ref = b.copy()
        _env(monkeypatch, {})
        c._check(c._L.hpl_gesl(c._c, f.ctypes.data, ref.ctypes.data, n, n, None))
        for env in ({"HPL_GESL_SPIN": "0"}, {}):
            _env(monkeypatch, env)
            x = torch.from_numpy(b).cuda()
            assert c._L.hpl_gesl_noalloc(F.data_ptr(), n, n, x.data_ptr(), None) == 0
            torch.cuda.synchronize()
            x = x.cpu().numpy()
            if env:
                assert np.any(np.isnan(x))
            else:
                assert np.array_equal(x, ref)


@pytest.mark.parametrize("n,B,prec,pivot", [(96, 32, "fp32", False), (320, 64, "fp32", False),
                                            (512, 128, "bf16", False), (1024, 256, "fp32", False),
                                            (96, 32, "fp32", True), (768, 256, "fp32", True)])
@pytest.mark.parametrize("nrhs", [1, 3, 16])
def test_without_whole_inverses(monkeypatch, n, B, prec, pivot, nrhs):
    """What is left where the inverses find no room: a launch per block that solves the
    diagonal system by its 32 x 32 inverses, for each width of right-hand sides."""
    print(f"no inverses n={n} B={B} {prec} pivot={pivot} nrhs={nrhs}", flush=True)
    _env(monkeypatch, {"HPL_GESL_INVERSES": "0"})
    g = np.random.default_rng(n + nrhs)
    a = (g.random((n, n)) - 0.5).astype(np.float32)
    if not pivot:
        a[np.arange(n), np.arange(n)] += n
    b = g.uniform(-1, 1, (n, nrhs))
    with Context(0) as c:
        c.keep_original(True)
        c.set_pivoting(pivot)
        c.upload(a, b[:, 0].astype(np.float32))
        c.gefa_dev(B, prec)
        c.gesl_dev()
        x0 = c.download(matrix=False)[1]
        x, res = c.solve_rhs64(b)
        c.upload_rhs64(b[:, 0])
        c.solve_gmres(B, prec)  # (raises where it does not converge)
        y = c.download_solution64()
    M = a.astype(np.float64).T
    r = np.abs(b - M @ x).max(axis=0)
    scale = np.abs(M).sum(axis=1).max() * np.abs(x).max(axis=0) + np.abs(b).max(axis=0)
    assert all(q["converged"] for q in res) and np.all(r <= 1e-14 * n * scale)
    assert np.abs(b[:, 0] - M @ y).max() <= 1e-14 * n * scale[0]
    # unrefined: the FP32 backward error grows like sqrt(n); BF16's own update error apart
    if prec == "fp32":
        r0 = np.abs(b[:, 0] - M @ x0).max()
        assert r0 <= 64 * np.sqrt(n) * 2.0 ** -24 * (scale[0] + np.abs(b).max())


@pytest.mark.parametrize("n,B", [(32, 32), (64, 32), (64, 64), (128, 64), (256, 128), (256, 256)])
def test_few_panels(monkeypatch, n, B):
    """Small pivoted factors are solved by a launch per panel block: no further off than
    gesl_ref in FP32, whether or not there is room for whole inverses."""
    print(f"few panels n={n} B={B}", flush=True)
    g = np.random.default_rng(n + B)
    a = (g.random((n, n)) - 0.5).astype(np.float32)
    b = g.uniform(-1, 1, n).astype(np.float32)
    x = []
    for env in ({}, {"HPL_GESL_INVERSES": "0"}):
        _env(monkeypatch, env)
        with Context(0) as c:
            c.set_pivoting(True)
            c.upload(a, b)
            c.gefa_dev(B)
            c.gesl_dev()
            x.append(c.download(matrix=False)[1])
            f, _ = c.download(matrix=True, solution=False)
            ipvt = c.pivots()
    assert np.array_equal(x[0], x[1])
    ref = np.linalg.solve(a.T.astype(np.float64), b.astype(np.float64))
    seq = O.gesl_pvt(f, b.copy(), ipvt)
    err = np.max(np.abs(x[0] - ref))
    assert err <= 8 * max(np.max(np.abs(seq - ref)), 2.0 ** -24 * np.max(np.abs(ref)))
