"""Calls on one dataset share its slabs of device memory one after another:
runs of different kinds and sizes in turn, on two datasets and from two
threads, give the results each gives alone."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _data(n, f, nb, seed, k=2):
    rng = np.random.default_rng(seed)
    bins = rng.integers(0, nb, size=(f, n), dtype=np.uint8)
    z = bins[0] / nb + (bins[1] / nb) * (bins[2] / nb) + 0.3 * rng.normal(size=n)
    y = np.floor(np.clip((z - z.min()) / (z.max() - z.min()), 0, 0.999) * k)
    return bins, y


def _same(a, b):
    assert a.n_trees == b.n_trees
    for k in ("feature", "threshold", "left", "right", "value", "gain", "count"):
        assert np.array_equal(getattr(a, k), getattr(b, k)), k
    assert np.array_equal(a.train_raw(), b.train_raw())


KINDS = [
    dict(objective=1, num_leaves=31, num_iterations=4),
    dict(objective=0, num_leaves=255, num_iterations=2),
    dict(objective=1, num_leaves=15, num_iterations=3, bagging_fraction=0.6, bagging_freq=1),
    dict(objective=1, num_leaves=31, num_iterations=13, goss=1, top_rate=0.2, other_rate=0.2, learning_rate=0.2),
    dict(objective=1, num_leaves=31, num_iterations=3, quant_scale_rule=1),
    dict(objective=1, num_leaves=31, num_iterations=3, partition_mode=1),
]


def test_calls_in_turn():
    from mojoboost_amd import device

    bins, y = _data(30_011, 9, 64, 1)
    alone = [device.Dataset(bins, 30_011, 9, 64, y).train(**k) for k in KINDS]
    ds = device.Dataset(bins, 30_011, 9, 64, y)
    for i in (0, 1, 2, 3, 4, 5, 5, 4, 3, 2, 1, 0):
        _same(ds.train(**KINDS[i]), alone[i])


@pytest.mark.parametrize("n,k", [(1, 3), (63, 2), (64, 17), (70_001, 10), (130, 33)])
def test_multiclass_scores_row_major(n, k):
    """train_raw's row-major scores, at the edges of the transpose's tiles:
    each row's scores are the base plus its leaves."""
    from mojoboost_amd import device

    rng = np.random.default_rng(n)
    bins = rng.integers(0, 16, size=(3, n), dtype=np.uint8)
    y = rng.integers(0, k, size=n).astype(np.float64)
    fit = device.Dataset(bins, n, 3, 16, y).train(objective=2, num_class=k, num_iterations=2, num_leaves=4,
                                                  min_data_in_leaf=1)
    want = fit.predict_binned(bins, n, 3)
    assert np.array_equal(fit.train_raw(), want)


def test_threads():
    from mojoboost_amd import device

    data = [_data(20_000 + 7 * i, 6, 32, 5 + i) for i in range(2)]
    sets = [device.Dataset(b, b.shape[1], 6, 32, y) for b, y in data]
    alone = [[sets[i].train(**k) for k in KINDS[:3]] for i in range(2)]
    got = [[], []]

    def work(i):
        for _ in range(3):
            for k in KINDS[:3]:
                got[i].append(sets[i].train(**k))

    ts = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    for i in range(2):
        for j, fit in enumerate(got[i]):
            _same(fit, alone[i][j % 3])
