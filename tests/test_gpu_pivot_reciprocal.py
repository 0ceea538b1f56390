"""GPU: the -1/p of the diagonal-block LU against the division, mantissa by mantissa.

The kernel forms -1/p from the hardware reciprocal and one Newton step in FMA and
claims the correctly rounded quotient.  The factor of a diagonal matrix with a one
beside every other pivot holds the quotients themselves: -1/p on the diagonal and,
as each row is scaled by it, beside it (1 * -1/p).  Near both ends of a binade every mantissa is tried, between them an
even sample; each end's own values in every place of a 128-wide block.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

N = 4096


def _check(ctx, bits):
    p = bits.astype(np.uint32).view(np.float32)
    a = np.zeros((N, N), np.float32)
    i = np.arange(N)
    a[i, i] = p
    a[i[::2], i[1::2]] = 1.0  # (every one: the inverses' products would overflow)
    ctx.gefa(a, 128)
    want = (np.float32(-1.0) / p).view(np.uint32)
    assert np.array_equal(a[i, i].view(np.uint32), want)
    assert np.array_equal(a[i[::2], i[1::2]].view(np.uint32), want[::2])


@pytest.mark.parametrize("sign", [0, 1])
@pytest.mark.parametrize("exponent", [64, 127, 190])
def test_ends_of_a_binade(ctx, sign, exponent):
    print(f"reciprocals sign={sign} exponent={exponent}", flush=True)
    head = (sign << 31) | (exponent << 23)
    low, high = np.arange(N), (1 << 23) - 1 - np.arange(N)
    for m in (low, high, np.resize([0, 1, 2, (1 << 23) - 1, (1 << 23) - 2], N)):
        _check(ctx, head | m)


@pytest.mark.parametrize("part", range(4))
def test_sample_of_a_binade(ctx, part):
    print(f"reciprocals part={part}", flush=True)
    rng = np.random.default_rng(part)
    for _ in range(32):  # a mantissa of each 2048 consecutive ones
        m = (np.arange(N) << 11) + rng.integers(0, 1 << 11, N)
        sign = rng.integers(0, 2, N)
        exponent = rng.integers(40, 215, N)
        _check(ctx, (sign << 31) | (exponent << 23) | rng.permutation(m))
