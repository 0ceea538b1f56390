"""GPU: copies between host and device through the pinned staging buffers.

Copies are exact, so every comparison is bit for bit.  Sizes: a row narrower
than the device's pitch, several pieces per copy with a short last one, host
rows longer than the system, more than one buffer's worth of contiguous bytes.
"""

import numpy as np
import pytest

from hpcc_fpga_amd import Batch, Context

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,pad", [(32, 0), (96, 5), (1056, 0), (1056, 33), (3000, 1)])
def test_matrix_round_trip(n, pad):
    print(f"transfer n={n} host pitch {n + pad}", flush=True)
    rng = np.random.default_rng(n + pad)
    a = rng.random((n, n + pad), np.float32)
    d = rng.random((n, n + pad))
    b = rng.random(n, np.float32)
    with Context(0) as c:
        for rep in range(2):  # the second call finds the buffers in use
            c.upload(a, b)
            out = np.full((n, n + pad), -1.0, np.float32)
            c._check(c._L.hpl_download(c._c, out.ctypes.data, n + pad, None, None))
            assert np.array_equal(out[:, :n], a[:, :n])
            assert np.all(out[:, n:] == -1.0)  # nothing written past a row
            assert np.array_equal(c.download_vectors()[0], b)
            a = a[::-1].copy()
        if n % 64 == 0:
            c.upload_f64(d)
            o64 = np.empty((n, n))
            c._check(c._L.hpl_download_f64(c._c, o64.ctypes.data, n, None, None))
            assert np.array_equal(o64, d[:, :n])


def test_batch_solutions_after_every_solve():
    """Solutions fetched one by one, then from the common copy, of this solve
    and not the last one; results of more bytes than one buffer holds."""
    count = 50000
    print(f"batch get, {count} systems", flush=True)
    with Context(0) as c:
        bt = Batch(c, np.full(count, 3, np.int32))
        for seed in (1, 2):
            bt.generate(seed)
            st = bt.solve("fp32")
            assert st["failed"] == 0
            for s in (0, 1, 2, count - 1, 3, 4, 5, count // 2, 0):
                x, it, berr = bt.get(s)
                m, b = bt.get_system(s)
                ref = np.linalg.solve(m[:3, :3].astype(np.float64).T, b[:3])
                assert np.max(np.abs(x - ref)) <= 1e-12
        # another right-hand side for one system: its own new solution
        m, b = bt.get_system(7)
        bt.set_system(7, m[:3, :3], 2.0 * b[:3])
        x0, _, _ = bt.get(7)  # still the last solve's
        bt.solve("fp32")
        x1, _, _ = bt.get(7)
        assert np.max(np.abs(x1 - 2.0 * x0)) <= 1e-12
        bt.close()
