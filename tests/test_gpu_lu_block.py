"""GPU: the diagonal-block LU where its fast path does not apply.

The kernel forms each pivot's -1/p from the hardware reciprocal and Newton
steps, which holds only away from the ends of the exponent range; a panel with
a pivot outside goes through divisions instead.  Either way every element gets
gefa_ref_nopvt's operations in its order (LINPACK/src/host/linpack_data.cpp:166-196),
so the factor is compared bit for bit.
"""
import numpy as np
import pytest

from hpcc_fpga_amd import HplError
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _matrix(B, kind):
    rng = np.random.default_rng(B)
    a = (rng.random((B, B), np.float32) - np.float32(0.5)).astype(np.float32)
    a[np.arange(B), np.arange(B)] += np.float32(B)
    if kind == "huge":
        a *= np.float32(2.0 ** 110)
    elif kind == "tiny":  # pivots below 2^-100, off-diagonal entries partly denormal
        a *= np.float32(2.0 ** -125)
    elif kind == "one huge pivot":  # in the last panel only
        a[B - 3] *= np.float32(2.0 ** 115)
    elif kind == "zeros":  # exact zeros of both signs, as padding has them
        a[rng.random((B, B)) < 0.5] = np.float32(0.0)
        a[rng.random((B, B)) < 0.2] = np.float32(-0.0)
        a[np.arange(B), np.arange(B)] = np.float32(B)
    return a


@pytest.mark.parametrize("kind", ["plain", "huge", "tiny", "one huge pivot", "zeros"])
@pytest.mark.parametrize("B", [32, 64, 128])
def test_lu_block_range(ctx, B, kind):
    print(f"lu block B={B} {kind}", flush=True)
    a = _matrix(B, kind)
    f = a.copy()
    ctx.gefa(f, B)
    assert np.array_equal(f.view(np.uint32), O.gefa_nopvt(a).view(np.uint32))


@pytest.mark.parametrize("row", [0, 37, 95, 127])
def test_zero_pivot_in_any_panel(ctx, row):
    print(f"lu block zero pivot at {row}", flush=True)
    a = np.diag(np.full(128, 3.0, np.float32))
    a[row, row] = 0.0
    with pytest.raises(HplError) as e:
        ctx.gefa(a, 128)
    assert e.value.status == 4


@pytest.mark.parametrize("B", [256, 512])
def test_recursive_block(ctx, B):
    """Blocks of several leaves: the whole factor as the parity tests take it."""
    print(f"recursive block B={B}", flush=True)
    a, b, _, _ = O.generate_ref(2 * B, seed=9)
    f = a.copy()
    ctx.gefa(f, B)
    ref = O.gefa_nopvt(a)
    assert np.max(np.abs(f - ref)) <= 2e-5 * np.max(np.abs(ref))


def test_block_beside_a_large_update(ctx):
    """The narrower workgroup of large orders: the first diagonal block, which no
    update precedes, bit for bit."""
    n, B = 6656, 128
    print(f"lu block B={B} of n={n}", flush=True)
    ctx.generate(n, 0, 5)
    a, _ = ctx.download(matrix=True, solution=False)
    ctx.gefa_dev(B)
    f, _ = ctx.download(matrix=True, solution=False)
    ref = O.gefa_nopvt(np.ascontiguousarray(a[:B, :B]))
    assert np.array_equal(np.ascontiguousarray(f[:B, :B]).view(np.uint32), ref.view(np.uint32))
