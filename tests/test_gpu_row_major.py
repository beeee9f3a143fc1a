"""train_raw's row-major scores where the transpose's blocks take several runs
of 64 rows each: every row's scores are the base plus its leaves."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(1 << 22) - 1, (1 << 22) + 1, 3 * (1 << 22) + 65])
def test_rows_past_the_blocks(n):
    from mojoboost_amd import device

    rng = np.random.default_rng(n)
    k = 3
    bins = rng.integers(0, 16, size=(2, n), dtype=np.uint8)
    y = ((bins[0] // 3 + bins[1] // 5) % k).astype(np.float64)
    fit = device.Dataset(bins, n, 2, 16, y).train(objective=2, num_class=k, num_iterations=1, num_leaves=7)
    assert np.array_equal(fit.train_raw(), fit.predict_binned(bins, n, 2))
