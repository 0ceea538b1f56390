"""GPU: hpl_batch_get in any order, from any thread, gives the last solve's solutions.

Systems read in ascending order are copied ahead, many read in another order are
copied together; each of those paths against the solutions read one at a time after
a solve of its own, in orders that start, break off and resume an ascending run.
"""
import threading
from contextlib import closing

import numpy as np
import pytest

from hpcc_fpga_amd import Batch, Context

pytestmark = pytest.mark.gpu


def _orders(count):
    up = np.arange(count)
    g = np.random.default_rng(count)
    return {"up": up, "down": up[::-1], "random": g.permutation(count), "even": up[::2],
            "twice": np.repeat(up, 2), "broken": np.concatenate([up[:7], up[3:9], up[count // 2:],
                                                                 up[:count // 2]])}


@pytest.mark.parametrize("count,lo,hi", [(1, 5, 6), (9, 1, 40), (700, 1, 200), (90, 900, 1025)])
def test_every_order(count, lo, hi):
    print(f"batch get of {count} systems", flush=True)
    n = np.random.default_rng(count).integers(lo, hi, count).astype(np.int32)
    with Context(0) as c, closing(Batch(c, n)) as bt:
        for seed in (1, 2):
            bt.generate(seed)
            bt.solve("fp16")
            ref = []
            for s in range(count)[::-1][:40]:  # few, descending: each by itself
                ref.append((s, bt.get(s)))
            for name, order in _orders(count).items():
                bt.solve("fp16")
                got = {int(s): bt.get(int(s)) for s in order}
                for s, (x, it, berr) in ref:
                    if s in got:
                        assert np.array_equal(got[s][0], x), (name, s)
                        assert got[s][1:] == (it, berr), (name, s)
            for s, (x, _, berr) in got.items():
                assert x.shape == (n[s],) and np.max(np.abs(x - 1.0)) <= 1e-9


def test_from_several_threads():
    count = 400
    print("batch get from several threads", flush=True)
    n = np.random.default_rng(0).integers(1, 150, count).astype(np.int32)
    with Context(0) as c, closing(Batch(c, n)) as bt:
        bt.generate(3)
        bt.solve("fp16")
        ref = [bt.get(s) for s in range(count)]
        for rep in range(3):
            bt.solve("fp16")
            out = [[None] * count for _ in range(4)]

            def read(k):
                order = (np.arange(count), np.arange(count)[::-1], np.arange(count),
                         np.random.default_rng(rep).permutation(count))[k]
                for s in order:
                    out[k][s] = bt.get(int(s))

            th = [threading.Thread(target=read, args=(k,)) for k in range(4)]
            for t in th:
                t.start()
            for t in th:
                t.join()
            for k in range(4):
                for s in range(count):
                    assert np.array_equal(out[k][s][0], ref[s][0]) and out[k][s][1:] == ref[s][1:]
