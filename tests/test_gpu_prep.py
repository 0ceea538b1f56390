"""GPU: the 32 x 32 inverses of hpl_gesl_noalloc and of an uploaded factor.

They come from a kernel that solves for the unit vectors, an element per lane;
the substitution that applies them is compared with an FP64 substitution of the
same factor, over orders of one block to several and every inner block (the
largest power of two up to 256 that divides n).  Bound: the factor is well
conditioned (diagonally dominant), so the FP32 result differs by a modest
multiple of the unit roundoff times the root of the number of terms.
"""
import numpy as np
import pytest

from oracle import oracle as O

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _x64(f, b):
    """Substitution with gefa_ref_nopvt's factor in FP64: stored rows are M's
    columns; negated multipliers right of the diagonal, -1/u_kk on it."""
    n = len(b)
    F = f.astype(np.float64).T  # M's factor
    L = np.tril(-F, -1) + np.eye(n)
    U = np.triu(F, 1) + np.diag(-1.0 / np.diag(F))
    return np.linalg.solve(U, np.linalg.solve(L, b.astype(np.float64)))


@pytest.mark.parametrize("n", [32, 64, 96, 128, 160, 256, 512, 768, 1056, 1088])
def test_noalloc(ctx, n):
    print(f"noalloc n={n}", flush=True)
    a, b, _, _ = O.generate_ref(n, seed=n)
    f = O.gefa_nopvt(a)
    F = torch.from_numpy(f).cuda()
    x = torch.from_numpy(b).cuda()
    for _ in range(2):  # the flags of a launch before are cleared
        x.copy_(torch.from_numpy(b))
        assert ctx._L.hpl_gesl_noalloc(F.data_ptr(), n, n, x.data_ptr(), None) == 0
        torch.cuda.synchronize()
    ref = _x64(f, b)
    err = np.max(np.abs(x.cpu().numpy() - ref)) / np.max(np.abs(ref))
    assert err <= 8 * np.sqrt(n) * 2.0 ** -21


@pytest.mark.parametrize("n", [32, 128, 1024])
def test_nan_of_every_pattern_ends(ctx, n):
    """Published values announce themselves by not being the cleared pattern, a
    NaN: right-hand sides of that very NaN (and of its payload's neighbours)
    still come out as NaN, without a wait that gives up."""
    print(f"gesl of NaN n={n}", flush=True)
    a, _, _, _ = O.generate_ref(n, seed=n)
    f = O.gefa_nopvt(a)
    for bits in (0xFFFFFFFF, 0x7FFFFFFF, 0xFFBFFFFF, 0x7FC00000):
        x = np.full(n, bits, np.uint32).view(np.float32)
        st = ctx._L.hpl_gesl(ctx._c, f.ctypes.data, x.ctypes.data, n, n, None)
        assert st == 0, (hex(bits), st)
        assert np.all(np.isnan(x)), hex(bits)


@pytest.mark.parametrize("n", [64, 1024])
def test_nan_of_every_pattern_ends_f64(ctx, n):
    print(f"f64 gesl of NaN n={n}", flush=True)
    a, _ = O.generate_ref_f64(n, seed=n)
    f = O.gefa_nopvt_f64(a)
    for bits in (0xFFFFFFFFFFFFFFFF, 0x7FFFFFFFFFFFFFFF, 0xFFF7FFFFFFFFFFFF):
        x = np.full(n, bits, np.uint64).view(np.float64)
        ctx.gesl_f64(f, x)
        assert np.all(np.isnan(x)), hex(bits)
