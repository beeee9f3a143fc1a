"""Histograms of the magnitude-sum lattice where the cells' layout changes:
bin-major up to the tile and bin counts whose cells fit a workgroup's LDS,
feature-major above, one tile or several; bit for bit against numpy."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,f,nb,sel", [
    (1, 1, 2, None), (5_000, 14, 256, 1), (40_001, 15, 255, 20_000),
    (40_001, 28, 255, None),  # the widest bin-major tile at 255 bins
    (40_001, 29, 255, 33),    # feature-major
    (20_003, 60, 64, None),   # 64-byte records, bin-major
    (9_999, 62, 100, 5_000),
    (3_001, 130, 33, None),   # several tiles
])
def test_wide_cells(n, f, nb, sel):
    from mojoboost_amd import device

    rng = np.random.default_rng(n + f)
    bins = rng.integers(0, nb, size=(f, n)).astype(np.uint8)
    most = min(1 << 30, ((1 << 31) - 1) // n)
    qg = rng.integers(-most, most + 1, size=n).astype(np.int32)
    qh = rng.integers(0, most + 1, size=n).astype(np.int32)
    rows = None if sel is None else np.sort(rng.choice(n, sel, replace=False)).astype(np.int32)
    got = device.Dataset(bins, n, f, nb, np.zeros(n)).histogram32(qg, qh, rows)
    r = np.arange(n) if rows is None else rows
    for j in range(f):
        for k, v in enumerate((qg[r].astype(np.int64), qh[r].astype(np.int64), np.ones(len(r), np.int64))):
            want = np.zeros(nb, np.int64)
            np.add.at(want, bins[j, r], v)
            assert np.array_equal(got[j, :, k], want), (j, k)
