"""LambdaRank's derivatives over more queries than a launch has blocks of 512
threads (2^32 threads of them): the oracle's bits, and in about the time of a
few queries less (a launch of that many blocks runs the remainder only, here
five: 80 ms became 4 s). And over queries on both sides of the smaller blocks'
rule."""
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


@pytest.mark.parametrize("few", [2047, 2048, 2051])
@pytest.mark.parametrize("others", [(), (33, 34, 500, 2048), (33, 2049)])
@pytest.mark.parametrize("trunc,norm", [(30, True), (3, False)])
def test_queries_of_few_documents(few, others, trunc, norm):
    """The blocks of two waves, alone and beside the larger ones: queries of 1
    to 32 documents, tied scores, grades up to 30."""
    from mojoboost_amd import device

    rng = np.random.default_rng(few + len(others))
    counts = rng.permutation(np.concatenate([rng.integers(1, 33, size=few - 4), [1, 31, 32, 32], others])).astype(np.int32)
    n = int(counts.sum())
    y = rng.integers(0, 5, size=n).astype(np.float64)
    y[:50] = rng.integers(0, 31, size=50)
    raw = np.round(rng.normal(size=n), 1)
    bins = rng.integers(0, 8, size=(2, n), dtype=np.uint8)
    ds = device.Dataset(bins, n, 2, 8, y)
    ds.set_groups(counts)
    g, h = ds.lambdarank(raw, lambdarank_truncation_level=trunc, lambdarank_norm=int(norm))
    wg, wh = O.lambdarank(raw, y, counts, truncation=trunc, sigma=1.0, norm=norm)
    assert np.array_equal(g.view(np.uint64), wg.view(np.uint64))
    assert np.array_equal(h.view(np.uint64), wh.view(np.uint64))
    # a training takes the magnitudes from both launches
    kw = dict(num_iterations=3, num_leaves=7, min_data_in_leaf=5, use_quantized_grad=1,
              lambdarank_truncation_level=trunc, lambdarank_norm=int(norm))
    fit = ds.train(objective=3, **kw)
    p, starts = O.rank_params(counts, **kw)
    ref = O.train(bins, n, 2, 8, y, p)
    assert fit.n_trees == ref.n_trees
    for k in ("feature", "threshold", "left", "right"):
        assert np.array_equal(getattr(fit, k), getattr(ref, k)), k
    assert np.array_equal(fit.train_raw().view(np.uint64), ref.train_raw(n).view(np.uint64))
