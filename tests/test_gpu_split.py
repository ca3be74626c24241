"""FP32 assignment with split BF16 products (km_assign_split.hpp) against the oracle's
exact-form argmin: equal labels at the edges of its tiles, halves and index bits, and
where the error band decides (rows far from the origin, tiny and huge values,
values that are not finite)."""

import numpy as np
import pytest

from conftest import gaussian_mixture
from test_gpu_parity import set_path

pytestmark = pytest.mark.gpu

# n, d, k: one row, a tile and a row, widths around the halves' edges and with
# every remainder mod 4, one block and a centroid, the largest k and the first past it
SHAPES = [(1, 5, 1), (257, 1, 2), (129, 30, 33), (256, 31, 32), (130, 33, 129), (255, 62, 7), (513, 65, 128),
          (128, 127, 128), (1000, 128, 257), (5000, 16, 4096), (5000, 16, 4097), (300, 129, 40)]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "n%d_d%d_k%d" % s)
def test_labels_equal_exact_form(engine, oracle, shape):
    n, d, k = shape
    set_path(engine, "mfma_f32")
    x = gaussian_mixture(max(n, k), d, min(k, 50), seed=n + d, sigma=(0.5, 2.0))
    c = x[np.random.default_rng(k).permutation(x.shape[0])[:k]].copy()
    x = x[:n].copy()
    lab, obj = engine.infer(x, c, objective=True)
    wl, _ = oracle.canonical_assign(x, c)
    assert np.array_equal(lab, wl)
    assert obj == oracle.canonical_objective(x, c, wl)


@pytest.mark.parametrize("scale,offset", [(1.0, 1e4), (1e-20, 0.0), (1e-38, 0.0), (3e18, 0.0), (1.0, -3e5)])
def test_labels_inside_the_band(engine, oracle, scale, offset):
    set_path(engine, "mfma_f32")
    x = (gaussian_mixture(3000, 24, 20, seed=8, dtype=np.float64) * scale + offset).astype(np.float32)
    c = x[:40].copy()
    lab, _ = engine.infer(x, c)
    assert np.array_equal(lab, oracle.canonical_assign(x, c)[0])


def test_rows_that_are_not_finite(engine, oracle):
    set_path(engine, "mfma_f32")
    x = gaussian_mixture(1000, 12, 9, seed=3)
    x[17, 3], x[400, 0], x[401, 11], x[999, 5] = np.nan, np.inf, -np.inf, 3e38
    c = gaussian_mixture(9, 12, 9, seed=5)
    lab, _ = engine.infer(x, c)
    assert np.array_equal(lab, oracle.canonical_assign(x, c)[0])
