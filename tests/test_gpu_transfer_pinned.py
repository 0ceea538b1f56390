"""GPU: host buffers that the runtime already knows (pinned) are copied directly.

Copies are exact: bit for bit, also at pitches beyond the order, beside ordinary
buffers in the same context, and where the caller reuses a buffer after the call.
"""
import numpy as np
import pytest
import torch  # before the library: one HIP runtime for both

from hpcc_fpga_amd import Context

pytestmark = pytest.mark.gpu


def _pinned(shape, dtype):
    t = torch.empty(shape, dtype={np.float32: torch.float32, np.float64: torch.float64}[dtype],
                    pin_memory=True)
    return t.numpy()


@pytest.mark.parametrize("n,pad", [(32, 0), (96, 5), (1024, 0), (1056, 33)])
def test_pinned_round_trip(n, pad):
    print(f"pinned n={n} host pitch {n + pad}", flush=True)
    rng = np.random.default_rng(n + pad)
    want = rng.random((n, n + pad), np.float32)
    bw = rng.random(n)
    a, out = _pinned((n, n + pad), np.float32), _pinned((n, n + pad), np.float32)
    b = _pinned((n,), np.float64)
    with Context(0) as c:
        for _ in range(2):
            a[:], b[:], out[:] = want, bw, -1.0
            c.upload(a)
            c.upload_rhs64(b)
            a[:], b[:] = 0.0, 0.0  # the calls are over: the buffers are the caller's again
            c._check(c._L.hpl_download(c._c, out.ctypes.data, n + pad, None, None))
            assert np.array_equal(out[:, :n], want[:, :n]) and np.all(out[:, n:] == -1.0)
            assert np.array_equal(c.download_vectors()[1], bw)
            c.upload(want)  # ordinary memory in between
            part = out[1:, 1:]  # inside a pinned buffer, at its pitch
            out[:] = -1.0
            if n > 32:
                c.upload(np.ascontiguousarray(want[:32, :32]))
                c._check(c._L.hpl_download(c._c, part.ctypes.data, n + pad, None, None))
                assert np.array_equal(part[:32, :32], want[:32, :32])


def test_pinned_right_hand_sides():
    n, nrhs = 512, 5
    print("pinned right-hand sides", flush=True)
    g = np.random.default_rng(1)
    a = (g.random((n, n)) - 0.5).astype(np.float32)
    a[np.arange(n), np.arange(n)] += n
    b, x = _pinned((nrhs, n + 3), np.float64), _pinned((nrhs, n + 7), np.float64)
    b[:] = g.uniform(-1, 1, b.shape)
    with Context(0) as c:
        c.keep_original(True)
        c.upload(a)
        c.gefa_dev(128)
        ref = c.solve_rhs64(np.ascontiguousarray(b[:, :n].T))[0]
        from hpcc_fpga_amd.linpack import _IRResult

        res = (_IRResult * nrhs)()
        c._check(c._L.hpl_solve_rhs64(c._c, nrhs, b.ctypes.data, n + 3, x.ctypes.data, n + 7, 50,
                                      1e-14 * n, res))
    assert np.array_equal(x[:, :n].T, ref)


@pytest.mark.parametrize("n", [1, 124, 128, 132, 8192, 8196])
def test_around_the_small_buffers(n):
    """Transfers of up to 64 KiB take small staging buffers, longer ones large ones:
    matrices and vectors on either side, in turn."""
    print(f"small transfers n={n}", flush=True)
    rng = np.random.default_rng(n)
    a = rng.random((n, n), np.float32)
    with Context(0) as c:
        for rep in range(5):  # more calls than buffers
            b = rng.random(n)
            c.upload(a, b.astype(np.float32))
            c.upload_rhs64(b)
            f, b64, _ = c.download_vectors()
            assert np.array_equal(b64, b) and np.array_equal(f, b.astype(np.float32))
            if n < 8192 or rep == 0:
                assert np.array_equal(c.download(matrix=True, solution=False)[0], a)
