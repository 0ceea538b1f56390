"""GPU: the pipelined schedule, its serial end and the grouped schedule give one factor.

Below an order of serial_m (HPL_SERIAL_M, read when a context is created) the
pipelined schedule goes on launch after launch on one stream.  Every element
still gets each step's update once, in step order, through the same products,
so wherever the change falls the factor agrees bit for bit -- also with 0,
where the groups run to the last block.
"""
import os

import numpy as np
import pytest

from hpcc_fpga_amd import Context

pytestmark = pytest.mark.gpu


def _factor(monkeypatch, env, n, B, prec):
    for k in [k for k in os.environ if k.startswith("HPL_")]:
        monkeypatch.delenv(k)
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    print(f"{env} n={n} B={B} {prec}", flush=True)
    with Context(0) as c:
        c.generate(n, 0, 5)
        c.gefa_dev(B, prec)
        a, _ = c.download(matrix=True, solution=False)
        c.gesl_dev()  # with the inverses that the factorisation left
        _, x = c.download(matrix=False, solution=True)
    return a, x


@pytest.mark.parametrize("n,B,prec,depth", [
    (2048, 128, "fp32", 3),
    (1792, 256, "fp32", 4),
    (1056, 32, "fp32", 4),
    (2560, 512, "fp32", 2),
    (3072, 256, "bf16", 5),
    (2048, 128, "fp16", 4),
    (3072, 256, "fp8", 5),
])
def test_serial_end(monkeypatch, n, B, prec, depth):
    d = {"HPL_UPDATE_DEPTH": str(depth)}
    g, xg = _factor(monkeypatch, {"HPL_SCHEDULE": "grouped", **d}, n, B, prec)
    for serial in (0, B, n // 2, n):
        p, x = _factor(monkeypatch, {"HPL_SERIAL_M": str(serial), **d}, n, B, prec)
        assert np.array_equal(g.view(np.uint32), p.view(np.uint32)), serial
        # the generator's solution is 1; FP32 substitution, low-precision factors
        # to their update's rounding (2^-4 for E4M3 on entries of size 1 / n)
        assert np.max(np.abs(x - 1.0)) <= np.max(np.abs(xg - 1.0)) + 1e-5, serial


@pytest.mark.parametrize("n,depth", [(64, 8), (192, 2), (1600, 6), (2688, 8)])
def test_serial_end_fp64(monkeypatch, n, depth):
    """The FP64 schedules (blocks of 64): grouped, pipelined to the end, and
    with the serial end from several orders on."""
    d = {"HPL_F64_DEPTH": str(depth)}
    out = []
    for env in ({"HPL_SCHEDULE": "grouped"}, {"HPL_SERIAL_M": "0"}, {"HPL_SERIAL_M": "640"},
                {"HPL_SERIAL_M": "640", "HPL_TAIL_M": "1000", "HPL_TAIL_DEPTH": "2"}, {}):
        for k in [k for k in os.environ if k.startswith("HPL_")]:
            monkeypatch.delenv(k)
        for k, v in {**env, **d}.items():
            monkeypatch.setenv(k, v)
        print(f"{env} n={n} FP64", flush=True)
        with Context(0) as c:
            c.generate_f64(n, 0, 3)
            c.gefa_dev_f64()
            out.append(c.download_f64(matrix=True, solution=False)[0])
    for a in out[1:]:
        assert np.array_equal(out[0].view(np.uint64), a.view(np.uint64))
