"""GPU: the serving engine in every update precision that its configuration names."""
import numpy as np
import pytest

from hpcc_fpga_amd import Server

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["fp32", "bf16", "fp16", "fp8"])
def test_every_precision(prec):
    print(f"serve {prec}", flush=True)
    g = np.random.default_rng(5)
    srv = Server(hbm_budget=4 * 10 ** 9, prec=prec, max_n=1100)
    try:
        for n, nrhs in ((64, 1), (300, 3), (1000, 16)):
            a = (g.random((n, n)) - 0.5).astype(np.float32)
            a[np.arange(n), np.arange(n)] += n
            b = g.uniform(-1, 1, (n, nrhs))
            x, r = srv.wait(srv.submit(b if nrhs > 1 else b[:, 0], a=a))
            x = x.reshape(n, nrhs)
            M = a.astype(np.float64).T
            scale = np.abs(M).sum(axis=1).max() * np.abs(x).max() + np.abs(b).max()
            assert np.abs(b - M @ x).max() <= 1e-14 * n * scale, (prec, n)
    finally:
        srv.close()
