"""LambdaRank's derivatives over more queries than a launch has blocks of 512
threads (2^32 threads of them): the oracle's bits, and in about the time of a
few queries less (a launch of that many blocks runs the remainder only, here
five: 80 ms became 4 s)."""
import time

import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu


def test_more_queries_than_blocks():
    from mojoboost_amd import device

    rng = np.random.default_rng(3)
    seconds = []
    for nq in ((1 << 23) - 5, (1 << 23) + 5):
        counts = np.where(np.arange(nq) % 2 == 0, 2, 1).astype(np.int32)
        n = int(counts.sum())
        y = rng.integers(0, 3, size=n).astype(np.float64)
        raw = rng.normal(size=n)
        ds = device.Dataset(np.zeros((1, n), np.uint8), n, 1, 2, y)
        ds.set_groups(counts)
        best = float("inf")
        for _ in range(3):
            t = time.time()
            g, h = ds.lambdarank(raw)
            best = min(best, time.time() - t)
        seconds.append(best)
        ds.free()
    wg, wh = O.lambdarank(raw, y, counts)
    assert np.array_equal(g.view(np.uint64), wg.view(np.uint64))
    assert np.array_equal(h.view(np.uint64), wh.view(np.uint64))
    assert seconds[1] < 5 * seconds[0], seconds
