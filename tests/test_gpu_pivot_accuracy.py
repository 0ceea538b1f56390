"""GPU: the unrefined answer of a pivoted factor is no further off than by whole blocks.

A pivoted factor is substituted in blocks of 32, so a sum over the order has n / 32
terms where whole panel blocks had n / B; the substitutions carry the sums' rounding
errors along.  The bounds are the mean backward errors that the substitution by whole
blocks reached (16 columns; 10 matrices of order 8192 with block 64, 24 of order 1024
with block 128; the means' standard errors were 0.7e-8 and 0.25e-8).
"""
import numpy as np
import pytest

from hpcc_fpga_amd import Context

pytestmark = pytest.mark.gpu


def _backward_errors(monkeypatch, env, n, B, seeds, together):
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    out = []
    with Context(0) as c:
        c.keep_original(True)
        c.set_pivoting(True)
        for seed in seeds:
            print(f"pivoted accuracy n={n} B={B} seed={seed} {env}", flush=True)
            c.generate(n, 2, seed)
            c.gefa_dev(B)
            b = np.random.default_rng(seed).uniform(-1, 1, (n, 16))
            for part in ([b] if together else b.T):
                res = c.solve_rhs64(part, max_iter=0, tol=1e-300, check=False)[1]
                out += [r["backward_error"] for r in res]
    return np.mean(out)


def test_several_columns(monkeypatch):
    assert _backward_errors(monkeypatch, {}, 8192, 64, range(3), True) <= 4.97e-7


# one column; by the launches that follow where the single launch gives up; and by
# whole blocks again, where the inverses find no room
@pytest.mark.parametrize("env", [{}, {"HPL_GESL_GROUPS": "1"}, {"HPL_GESL_INVERSES": "0"}])
def test_one_column(monkeypatch, env):
    bound = 1.87e-7 + (3 * 0.43e-8 if "HPL_GESL_INVERSES" in env else 0.0)  # its own mean, 8 of 24
    assert _backward_errors(monkeypatch, env, 1024, 128, range(8), False) <= bound
