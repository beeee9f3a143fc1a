"""mbh_predict_binned of a matrix that its device copy takes in several batches
of rows: columns gathered in groups (a last group and a last batch of few), and
columns long enough for copies of their own. Scores against a plain walk."""
import ctypes as C

import numpy as np
import pytest

from test_gpu_predict_shapes import _tree, _walk

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,f,k", [
    (4_101, 600_000, 1),   # batches of 4096 and 5 rows, the last group of columns short
    (270_000, 8, 2_000),   # 134K rows, then the rest: gathered, the scores set the batch
    (300_000, 8, 900),     # 297K rows on their own, the rest gathered
])
def test_batches(n, f, k):
    from mojoboost_amd import _lib
    from mojoboost_amd._lib import ptr

    rng = np.random.default_rng(f)
    nb, trees = 64, 3
    # the trees split on the first columns, the last ones and some between
    forest = [_tree(rng, 20, 40, nb, False, t % 2 == 1) for t in range(trees)]
    names = np.unique(np.concatenate([[0, f - 1], rng.integers(0, f, size=38)])).astype(np.int32)
    forest = [(np.where(t[0] >= 0, names[t[0] % len(names)], -1).astype(np.int32),) + t[1:] for t in forest]
    off = np.cumsum([0] + [len(t[0]) for t in forest]).astype(np.int64)
    feat, thr, left, right, value, dl, mb, _ = (np.concatenate([t[i] for t in forest]) for i in range(8))
    bins = np.empty((f, n), np.uint8)
    block = rng.integers(0, nb, size=1 << 20, dtype=np.uint8)
    flat = bins.reshape(-1)
    for at in range(0, flat.size, len(block) - 7):
        part = flat[at:at + len(block) - 7]
        part[:] = block[:len(part)]
    for c in names:
        bins[c] = rng.integers(0, nb, size=n, dtype=np.uint8)
    base = np.arange(1.0, k + 1.0)
    out = np.zeros(n * k)
    err = C.create_string_buffer(512)
    rc = _lib.lib().mbh_predict_binned(ptr(bins), n, f, k, 0.5, ptr(base), ptr(off), 0, trees, ptr(feat), ptr(thr),
                                       ptr(left), ptr(right), ptr(value), ptr(dl), ptr(mb), None, ptr(out), err, 512)
    assert rc == 0, err.value
    want = np.tile(base[:trees], (n, 1))
    for t, tree in enumerate(forest):
        want[:, t % k] += 0.5 * _walk(tree, bins, n)
    out = out.reshape(n, k)
    assert np.array_equal(out[:, :trees], want)
    assert k <= trees or (out[:, k - 1] == base[k - 1]).all()
