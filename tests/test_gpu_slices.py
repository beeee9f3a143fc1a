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


@pytest.mark.parametrize("n,f,nb,kw", [
    (1, 1, 4, dict(min_data_in_leaf=1)),
    (1_023, 8, 256, {}), (1_025, 9, 63, {}),           # chunks and slices of one launch
    (65_536, 20, 255, {}), (65_537, 20, 255, {}),      # the last rows of one launch, the first of two
    (20_000, 48, 33, {}), (20_000, 49, 33, {}),        # the most slices, and one more
    (30_000, 12, 64, dict(quant_scale_rule=1, bagging_fraction=0.7, bagging_freq=1)),
    (30_000, 12, 64, dict(goss=1, top_rate=0.2, other_rate=0.2, learning_rate=0.5)),
    (9_000, 6, 40, dict(num_leaves=255, min_data_in_leaf=2)),
])
def test_one_launch_expansion(n, f, nb, kw):
    """Quantized trees of small data, where one launch partitions and
    accumulates: the CPU oracle's, bit for bit, missing bins among them."""
    from mojoboost_amd import device

    rng = np.random.default_rng(n + f)
    bins = rng.integers(0, nb, size=(f, n)).astype(np.uint8)
    missing = np.where(np.arange(f) % 3 == 0, nb - 1, -1).astype(np.int32)
    z = bins[0] / nb + (bins[-1] / nb) ** 2 + 0.4 * rng.normal(size=n)
    y = (z > np.median(z)).astype(np.float64)
    p = dict(objective=1, num_iterations=5, num_leaves=20, min_data_in_leaf=10, lambda_l2=1.0, learning_rate=0.1)
    p.update(kw)
    fit = device.Dataset(bins, n, f, nb, y, missing_bin=missing).train(**p)
    ref = O.train(bins.ravel(), n, f, nb, y, O.default_params(**p, use_quantized_grad=1), missing_bin=missing)
    assert fit.n_trees == ref.n_trees
    for k in ("feature", "threshold", "left", "right", "default_left"):
        assert np.array_equal(getattr(fit, k), getattr(ref, k)), k
    for k in ("value", "gain", "count"):
        assert np.array_equal(getattr(fit, k).view(np.uint64), getattr(ref, k).view(np.uint64)), k
