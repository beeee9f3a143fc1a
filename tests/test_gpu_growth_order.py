"""The planner's replay commits runs of splits at once: tree for tree the
oracle's one-split-at-a-time order, at the edges of the frontier's layout (64
slots a lane group), on equal gains (copies of the same rows, whose subtrees
tie split for split) and where growth ends early."""
import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("leaves", [2, 3, 15, 63, 64, 65, 127, 256, 257, 440])
@pytest.mark.parametrize("copies", [1, 4])
def test_growth_order(leaves, copies):
    from mojoboost_amd import device

    rng = np.random.default_rng(leaves)
    n0, f = 6_000, 6
    bins0 = rng.integers(0, 60, size=(f, n0)).astype(np.uint8)
    y0 = ((bins0[0].astype(int) * 7 + bins0[1] * bins0[2]) % 11 < 5).astype(np.float64)
    # each copy of the rows has its own value of one more feature
    n = n0 * copies
    bins = np.vstack([np.tile(bins0, copies), np.repeat(np.arange(copies, dtype=np.uint8), n0)[None, :]])
    y = np.tile(y0, copies)
    p = dict(num_iterations=3, num_leaves=leaves, min_data_in_leaf=5, lambda_l2=1.0, learning_rate=0.3, objective=1)
    bins = np.ascontiguousarray(bins)
    fit = device.Dataset(bins, n, f + 1, 60, y).train(**p, use_quantized_grad=1)
    ref = O.train(bins, n, f + 1, 60, y, O.default_params(**p, use_quantized_grad=1))
    assert fit.n_trees == ref.n_trees
    for k in ("feature", "threshold", "left", "right"):
        assert np.array_equal(getattr(fit, k), getattr(ref, k)), k
