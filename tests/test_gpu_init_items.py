"""k-means++ steps on both sides of the row count at which an item grows from 256 to 1024
rows (init_step_kernel): the chosen rows equal the oracle's, bit for bit, on every width
of a row's pieces, with bounds (32 MB of rows and more) and without."""

import numpy as np
import pytest

from conftest import gaussian_mixture

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [255, 257, 400000, 400001])
@pytest.mark.parametrize("d,dtype", [(1, np.float32), (5, np.float32), (13, np.float32), (33, np.float32),
                                     (1, np.float64), (3, np.float64), (7, np.float64), (20, np.float64)])
def test_plus_plus_items(engine, oracle, n, d, dtype):
    x = gaussian_mixture(n, d, 8, seed=n + d, center_range=10.0, dtype=dtype)
    assert np.array_equal(engine.init_centroids(x, 7, 2, seed=d), oracle.init_centroids(x, 7, 2, d))
