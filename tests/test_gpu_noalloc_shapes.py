"""mbh_histogram_noalloc at the edges of its feature tiles, row chunks and
merge blocks, bit for bit against numpy sums."""
import numpy as np
import pytest

from test_zz_no_alloc import _case, _Hip, _noalloc

pytestmark = pytest.mark.gpu


def _want(bins, qg, qh, rows, f, nb):
    r = np.arange(bins.shape[1]) if rows is None else rows
    want = np.zeros((f, nb, 3), np.int64)
    for j in range(f):
        for k, v in enumerate((qg[r], qh[r], np.ones(len(r)))):
            want[j, :, k] = np.bincount(bins[j, r], weights=v.astype(np.float64), minlength=nb)
    return want


@pytest.mark.parametrize("n,f,nb,sel", [
    (1, 1, 2, None),             # one row, one feature
    (63, 8, 256, None),          # one tile exactly
    (1025, 9, 255, None),        # one row past a chunk, two tiles
    (2049, 17, 33, 1),           # a single selected row
    (70_001, 15, 255, 33_333),   # ragged list, the last tile short
    (300_000, 3, 7, 299_999),    # the hottest bins
    (1_200_000, 28, 255, None),  # chunks above the smallest
    (200, 9_000, 2, 150),        # more than kMaxTiles x kTileFeatures features
    (40, 256, 256, None),        # the first cells merged by a thread each, one partial
    (3_000, 2_100, 255, 2_500),  # three partials, a ragged last merge block
    (9_000, 255, 256, None),     # just below them
    (40_000, 300, 255, None),    # eight partials, a cell's threads each one
])
def test_noalloc_shapes(n, f, nb, sel):
    rng = np.random.default_rng(n + f)
    bins, qg, qh = _case(rng, n, f, nb, 4)
    # any order, repeats among them
    rows = None if sel is None else rng.integers(0, n, size=sel).astype(np.int32)
    hip = _Hip()
    try:
        got, status = _noalloc(hip, bins, n, f, nb, qg, qh, rows)
    finally:
        hip.free()
    assert status == 0
    assert np.array_equal(got.astype(np.int64), _want(bins, qg, qh, rows, f, nb))
