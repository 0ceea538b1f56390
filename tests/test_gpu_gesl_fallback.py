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
