"""mbh_predict_binned on trees whose nodes are reached twice or not at all,
which a model file may hold: the scores of a plain walk, with the tree alone,
followed by trees that would fill another chunk, and in one class of three.
Leaf values are small dyadic fractions and the learning rate is 1/2, so the
sums are exact."""
import ctypes as C

import numpy as np
import pytest

from test_gpu_predict_shapes import _tree, _walk

pytestmark = pytest.mark.gpu

# features, left and right children; thresholds and values are drawn
SHARED = {
    # visits as many nodes as it has, four of them leaves of its two
    "leaves": ([0, 1, 1, 1, 2, -1, -1], [3, 2, 5, 5, 6, -1, -1], [4, 5, 6, 6, 5, -1, -1]),
    # one leaf for every split
    "one_leaf": ([0, 0, 0, -1], [3, 3, 3, -1], [3, 3, 3, -1]),
    # siblings neighbours, both subtrees the same nodes
    "siblings": ([0, 1, 2, -1, -1], [1, 3, 3, -1, -1], [2, 4, 4, -1, -1]),
}


def _shared(rng, name, nb):
    feat, left, right = (np.array(v, np.int32) for v in SHARED[name])
    m = len(feat)
    return (feat, np.where(feat >= 0, rng.integers(nb, size=m), -1).astype(np.int32), left, right,
            rng.integers(-64, 65, size=m) / 64.0, np.zeros(m, np.int32), np.full(m, -1, np.int32),
            np.zeros((m, 4), np.uint64))


@pytest.mark.parametrize("name", sorted(SHARED))
@pytest.mark.parametrize("n,after,k", [(300, 0, 1), (300, 5, 1), (300, 5, 3), (262_000, 5, 1)])
def test_shared_nodes(name, n, after, k):
    from mojoboost_amd import _lib
    from mojoboost_amd._lib import ptr

    rng = np.random.default_rng(n + after + k)
    f, nb = 4, 32
    forest = [_shared(rng, name, nb)] + [_tree(rng, 500, f, nb, False, t % 2 == 1) for t in range(after)]
    off = np.cumsum([0] + [len(t[0]) for t in forest]).astype(np.int64)
    feat, thr, left, right, value, dl, mb, _ = (np.concatenate([t[i] for t in forest]) for i in range(8))
    bins = rng.integers(0, nb, size=(f, n), dtype=np.uint8)
    base = np.arange(1.0, k + 1.0)
    want = np.tile(base, (n, 1))
    for t, tree in enumerate(forest):
        want[:, t % k] += 0.5 * _walk(tree, bins, n)
    out = np.zeros(n * k)
    err = C.create_string_buffer(512)
    rc = _lib.lib().mbh_predict_binned(ptr(bins), n, f, k, 0.5, ptr(base), ptr(off), 0, len(forest), ptr(feat),
                                       ptr(thr), ptr(left), ptr(right), ptr(value), ptr(dl), ptr(mb), None, ptr(out),
                                       err, 512)
    assert rc == 0, err.value
    assert np.array_equal(out.reshape(n, k), want)
