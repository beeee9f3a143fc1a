"""The bag's root list at the edges of its tiles of 4096 rows (and of its
grid of them): quantized trees equal to the CPU oracle's, bit for bit."""
import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,fraction,kw", [
    (63, 0.5, dict(min_data_in_leaf=3)),
    (4_095, 0.9, {}), (4_096, 0.1, {}), (4_097, 0.5, {}),
    (50_001, 0.02, {}),                        # tiles with a few rows each
    (40_000, 0.7, dict(quant_scale_rule=1)),   # pairs written beside the list
])
def test_bag_tiles(n, fraction, kw):
    from mojoboost_amd import device

    rng = np.random.default_rng(n)
    f, nb = 5, 32
    x = rng.normal(size=(f, n))
    y = (x[0] + 0.5 * x[1] * x[2] + rng.normal(size=n) > 0).astype(np.float64)
    bins = O.bin_equal_width(x.ravel(), n, f, nb)
    p = dict(objective=1, num_iterations=3, num_leaves=7, min_data_in_leaf=10, lambda_l2=1.0, learning_rate=0.1,
             bagging_fraction=fraction, bagging_freq=1)
    p.update(kw)
    fit = device.Dataset(bins, n, f, nb, y).train(**p)
    ref = O.train(bins, n, f, nb, y, O.default_params(**p, use_quantized_grad=1))
    assert fit.n_trees == ref.n_trees
    for k in ("feature", "threshold", "left", "right"):
        assert np.array_equal(getattr(fit, k), getattr(ref, k)), k
    for k in ("value", "gain", "count"):
        assert np.array_equal(getattr(fit, k).view(np.uint64), getattr(ref, k).view(np.uint64)), k
