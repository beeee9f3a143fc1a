"""Small batches' accumulation in feature slices: histograms and trees at the
edges of the slices (8 features), of the root's chunks (1536 rows) and of the
rule that takes them, binary32, binary64 (GOSS-weighted) and magnitude-sum
cells."""
import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,f,nb,sel", [
    (1, 9, 2, None), (1_536, 16, 255, None), (1_537, 17, 64, 700), (20_001, 31, 255, None),
    (98_304, 28, 255, None), (98_305, 29, 100, 50_000), (60_000, 70, 33, 1),
])
def test_slice_histograms(n, f, nb, sel):
    from mojoboost_amd import device

    rng = np.random.default_rng(n + f)
    bins = rng.integers(0, nb, size=(f, n)).astype(np.uint8)
    g = (rng.integers(-512, 513, size=n) / 256.0).astype(np.float32)  # sums exact in binary64
    h = (rng.integers(0, 513, size=n) / 256.0).astype(np.float32)
    rows = None if sel is None else np.sort(rng.choice(n, sel, replace=False)).astype(np.int32)
    gh, cnt = device.Dataset(bins, n, f, nb, np.zeros(n)).histogram_fp32(g, h, rows)
    r = np.arange(n) if rows is None else rows
    gh, cnt = gh.reshape(f, nb, 2), cnt.reshape(f, nb)
    for j in range(f):
        for got, v in ((gh[j, :, 0], g[r].astype(np.float64)), (gh[j, :, 1], h[r].astype(np.float64)),
                       (cnt[j], np.ones(len(r)))):
            assert np.array_equal(got, np.bincount(bins[j, r], weights=v, minlength=nb)), j


@pytest.mark.parametrize("n,f,kw", [
    (3_000, 9, dict(objective=0)),
    (40_000, 20, dict(objective=1)),
    (30_000, 17, dict(objective=1, goss=1, top_rate=0.3, other_rate=0.3, learning_rate=0.5)),
    (12_000, 33, dict(objective=1, bagging_fraction=0.5, bagging_freq=1)),
])
def test_slice_training(n, f, kw):
    """The same splits as the oracle's, scores within 1e-5 (binary64 sums in
    another order)."""
    from mojoboost_amd import device

    rng = np.random.default_rng(n)
    x = rng.normal(size=(f, n))
    z = x[0] + x[1] * x[2] + 0.5 * rng.normal(size=n)
    y = z if kw["objective"] == 0 else (z > 0).astype(np.float64)
    bins = O.bin_equal_width(x.ravel(), n, f, 200)
    p = dict(num_iterations=6, num_leaves=24, min_data_in_leaf=20, lambda_l2=1.0, learning_rate=0.1)
    p.update(kw)
    fit = device.Dataset(bins, n, f, 200, y).train(**p, use_quantized_grad=0)
    ref = O.train(bins, n, f, 200, y, O.default_params(**p, use_quantized_grad=0))
    assert fit.n_trees == ref.n_trees
    want = ref.train_raw(n)
    assert np.max(np.abs(fit.train_raw() - want)) <= 1e-5 * np.max(np.abs(want))
    for k in ("feature", "threshold", "left", "right"):
        assert np.array_equal(getattr(fit, k), getattr(ref, k)), k
