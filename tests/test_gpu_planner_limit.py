"""num_leaves at the planner's limit: the largest that a dataset accepts grows
the oracle's trees, and every larger one is refused, before any launch."""
import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu


def _refused(ds, leaves, **kw):
    from mojoboost_amd import _lib

    try:
        ds.train(num_leaves=leaves, **kw)
    except _lib.MojoTreesError as e:
        assert "planner" in str(e), e
        assert e.code == _lib.ERROR_UNSUPPORTED, e
        return True
    return False


@pytest.mark.parametrize("features,quantized", [(6, 1), (28, 1), (28, 0)])
def test_largest_accepted(features, quantized):
    from mojoboost_amd import device

    rng = np.random.default_rng(features)
    n, nb = 12_000, 60
    bins = rng.integers(0, nb, size=(features, n)).astype(np.uint8)
    y = ((bins[0].astype(int) * 7 + bins[1] * bins[2]) % 11 < 5).astype(np.float64)
    ds = device.Dataset(bins, n, features, nb, y)
    # no tree is grown while the limit is looked for
    lo, hi = 440, 1024
    while hi - lo > 1:
        mid = (lo + hi) // 2
        if _refused(ds, mid, num_iterations=0):
            hi = mid
        else:
            lo = mid
    assert 473 <= lo <= 512
    for leaves in (lo + 1, lo + 2, 502, 512, 513, 600, 655, 1024):
        if leaves > lo:
            assert _refused(ds, leaves, num_iterations=2), leaves
    p = dict(num_iterations=2, num_leaves=lo, min_data_in_leaf=3, lambda_l2=1.0, learning_rate=0.3, objective=1,
             use_quantized_grad=quantized)
    fit = ds.train(**p)
    ref = O.train(bins, n, features, nb, y, O.default_params(**p))
    assert fit.n_trees == ref.n_trees
    assert max(np.diff(fit.off)) == 2 * lo - 1  # the trees have that many leaves
    for k in ("feature", "threshold", "left", "right"):
        assert np.array_equal(getattr(fit, k), getattr(ref, k)), k
