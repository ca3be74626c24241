"""k-means++ steps that leave out rows by the triangle inequality (init_step_kernel):
the chosen rows equal the oracle's, bit for bit, on sizes that keep bounds (32 MB of
rows and more) and on every width of a row's pieces."""

import numpy as np
import pytest

from conftest import gaussian_mixture

pytestmark = pytest.mark.gpu

PLUS_PLUS = 2

CASES = [
    # n, d, k, dtype, clustered: bounds kept with whole and partial pieces, on clustered
    # rows (most are left out) and on uniform ones (few are); then narrow rows
    (70001, 127, 40, np.float32, True),
    (70001, 127, 25, np.float32, False),
    (263000, 32, 30, np.float32, True),
    (300001, 15, 20, np.float64, True),
    (33000, 128, 30, np.float64, False),
    (9001, 1, 12, np.float32, True),
    (9001, 5, 12, np.float32, True),
    (9001, 13, 12, np.float32, False),
    (9001, 1, 12, np.float64, True),
    (9001, 7, 12, np.float64, True),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "n%d_d%d_k%d_%s_%s" % (c[0], c[1], c[2], c[3].__name__, c[4]))
def test_plus_plus_with_bounds(engine, oracle, case):
    n, d, k, dtype, clustered = case
    if clustered:
        x = gaussian_mixture(n, d, 24, seed=d, center_range=10.0, dtype=dtype)
    else:
        x = np.random.default_rng(d).uniform(-1, 1, size=(n, d)).astype(dtype)
    got = engine.init_centroids(x, k, PLUS_PLUS, seed=n)
    want = oracle.init_centroids(x, k, PLUS_PLUS, n)
    assert np.array_equal(got, want)


def test_plus_plus_with_bounds_and_duplicate_rows(engine, oracle):
    """Every row many times: distances of exactly zero, and nothing left to choose."""
    base = gaussian_mixture(12, 128, 12, seed=2)
    x = np.tile(base, (6000, 1))
    got = engine.init_centroids(x, 15, PLUS_PLUS, seed=5)
    assert np.array_equal(got, oracle.init_centroids(x, 15, PLUS_PLUS, 5))
