"""mbh_predict_binned over the splits of its work: rows per block from one
per thread down to the fewest, chunks of many and of few trees, bins in LDS
and not, trees too large for a chunk, missing bins, category sets, several
classes, single-leaf trees, a tree range. Leaf values are small dyadic
fractions and the learning rate is 1/2, so every sum is exact and a plain
walk gives the scores' bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _tree(rng, n_inner, f, nb, cat, shuffle):
    """A random tree of n_inner splits: children after their parents,
    siblings neighbours or not."""
    feat, thr, left, right, dl, mb = [-1], [-1], [-1], [-1], [0], [-1]
    leaves = [0]
    for _ in range(n_inner):
        at = leaves.pop(rng.integers(len(leaves)))
        a = len(feat)
        for _ in range(2):
            feat.append(-1), thr.append(-1), left.append(-1), right.append(-1), dl.append(0), mb.append(-1)
        feat[at] = int(rng.integers(f))
        thr[at] = -1 if cat and rng.random() < 0.3 else int(rng.integers(nb))
        l, r = (a + 1, a) if shuffle and rng.random() < 0.5 else (a, a + 1)
        left[at], right[at] = l, r
        dl[at] = int(rng.integers(2))
        mb[at] = int(rng.choice([-1, nb - 1])) if thr[at] >= 0 else -1
        leaves += [a, a + 1]
    value = rng.integers(-64, 65, size=len(feat)) / 64.0
    bits = rng.integers(0, 2**63, size=(len(feat), 4), dtype=np.uint64)
    return (np.array(feat, np.int32), np.array(thr, np.int32), np.array(left, np.int32), np.array(right, np.int32),
            value, np.array(dl, np.int32), np.array(mb, np.int32), bits)


def _walk(tree, bins, n):
    feat, thr, left, right, value, dl, mb, bits = tree
    at = np.zeros(n, np.int64)
    rows = np.arange(n)
    while True:
        inner = feat[at] >= 0
        if not inner.any():
            return value[at]
        b = bins[np.maximum(feat[at], 0), rows].astype(np.int64)
        word = bits[at, b >> 6] >> (b & 63).astype(np.uint64)
        go = np.where(thr[at] < 0, (word & np.uint64(1)) != 0, np.where(b == mb[at], dl[at] != 0, b <= thr[at]))
        at = np.where(inner, np.where(go, left[at], right[at]), at)


@pytest.mark.parametrize("n,f,nb,inner,trees,k,cat,begin", [
    (1, 1, 2, (1, 2), 3, 1, False, 0),               # fewest rows of a block
    (17, 5, 256, (0, 3), 40, 1, False, 0),           # single-leaf trees among them
    (501, 28, 255, (30, 30), 100, 1, False, 0),      # more trees than a chunk's leaf values
    (5_003, 13, 63, (20, 60), 65, 1, True, 0),       # category sets
    (180_001, 29, 255, (5, 254), 24, 3, True, 3),    # three classes, a range without tree 0
    (261_632, 7, 16, (14, 14), 9, 1, False, 0),      # the last size of k_predict_wide
    (261_633, 7, 16, (14, 14), 9, 1, False, 0),      # the first of k_predict_rows, a ragged last block
    (300_000, 130, 64, (30, 31), 6, 1, False, 0),    # bins past the budget of a row a thread
    (900, 20_000, 64, (30, 31), 4, 1, True, 0),      # bins read from global memory
    (3_000, 9, 255, (1_000, 1_023), 5, 1, False, 0),  # a tree a chunk
    (2_000, 9, 255, (2_500, 2_600), 3, 1, True, 0),  # trees past a chunk's nodes
])
def test_predict_shapes(n, f, nb, inner, trees, k, cat, begin):
    import ctypes as C

    from mojoboost_amd import _lib
    from mojoboost_amd._lib import ptr

    rng = np.random.default_rng(n + f)
    forest = [_tree(rng, int(rng.integers(inner[0], inner[1] + 1)), f, nb, cat, t % 2 == 1) for t in range(trees)]
    off = np.cumsum([0] + [len(t[0]) for t in forest]).astype(np.int64)
    feat, thr, left, right, value, dl, mb, bits = (np.concatenate([t[i] for t in forest]) for i in range(8))
    bins = rng.integers(0, nb, size=(f, n), dtype=np.uint8) if nb < 256 else rng.integers(0, 256, size=(f, n)).astype(np.uint8)
    base = np.arange(1.0, k + 1.0)
    want = np.tile(base if begin == 0 else np.zeros(k), (n, 1))
    for t in range(begin, trees):
        want[:, t % k] += 0.5 * _walk(forest[t], bins, n)
    out = np.zeros(n * k)
    err = C.create_string_buffer(512)
    rc = _lib.lib().mbh_predict_binned(
        ptr(bins), n, f, k, 0.5, ptr(base) if begin == 0 else None, ptr(off), begin, trees, ptr(feat), ptr(thr),
        ptr(left), ptr(right), ptr(value), ptr(dl), ptr(mb), ptr(bits) if cat else None, ptr(out), err, 512)
    assert rc == 0, err.value
    assert np.array_equal(out.reshape(n, k), want)
