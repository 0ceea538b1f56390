"""GPU: the pivot panel's splits over workgroups of 64, 128 and 256 rows give one factor.

A panel takes 256 rows per workgroup only beyond 16384 rows, where no oracle
follows in test time; HPL_PANEL_ROWS asks for the same split at small orders.
Every row sees the same operations in each split, so factor and pivots agree
bit for bit, and the pivots with gefa_ref's restatement.
"""
import numpy as np
import pytest

from hpcc_fpga_amd import Context
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,B", [(32, 32), (224, 32), (576, 64), (960, 64), (896, 128), (1152, 128),
                                 (768, 256)])
def test_rows_per_workgroup(monkeypatch, n, B):
    rng = np.random.default_rng(n + B)
    a = (rng.random((n, n), np.float32) - np.float32(0.5)).astype(np.float32)
    got = {}
    for rows in (64, 128, 256):
        print(f"pivoted n={n} B={B} rows={rows}", flush=True)
        monkeypatch.setenv("HPL_PANEL_ROWS", str(rows))
        with Context(0) as c:
            for _ in range(2):
                f = a.copy()
                got[rows] = f, c.gefa_pvt(f, B)[0]
    f_ref, ipvt_ref = O.gefa_pvt(a)
    for f, ipvt in got.values():
        assert np.array_equal(ipvt, ipvt_ref)
        assert np.array_equal(f.view(np.uint32), got[64][0].view(np.uint32))
    assert np.array_equal(got[64][0][:B].view(np.uint32), f_ref[:B].view(np.uint32))


@pytest.mark.parametrize("rows", [128, 256])
def test_ties(monkeypatch, rows):
    """Equal magnitudes in several workgroups and waves: the first row wins."""
    n, B = 768, 64
    print(f"pivoted ties rows={rows}", flush=True)
    rng = np.random.default_rng(rows)
    a = rng.choice(np.array([-2.0, -1.0, 1.0, 2.0], np.float32), (n, n)).astype(np.float32)
    monkeypatch.setenv("HPL_PANEL_ROWS", str(rows))
    with Context(0) as c:
        f = a.copy()
        ipvt = c.gefa_pvt(f, B)[0]
    f_ref, ipvt_ref = O.gefa_pvt(a)
    assert np.array_equal(ipvt[:B], ipvt_ref[:B])
    assert np.array_equal(f[:B].view(np.uint32), f_ref[:B].view(np.uint32))
