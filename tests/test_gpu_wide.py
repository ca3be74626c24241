"""FP32 assignment of wide rows (km_assign_wide.hpp) against the oracle's exact-form
argmin: equal labels at the edges of its tiles and feature chunks, where the error
band decides, and past its limits."""

import numpy as np
import pytest

from conftest import gaussian_mixture
from test_gpu_parity import assert_bit_exact, set_path

pytestmark = pytest.mark.gpu

# n, d, k: both tile widths with one centroid more and less, one row and a tile and a
# row, one to three chunks of 32 features past 128 with every remainder mod 4 and
# mod 32, several centroid tiles, the last k of the kernel and the first past it, the widest rows
SHAPES = [(1, 129, 1), (127, 160, 127), (129, 161, 129), (128, 256, 128), (257, 257, 256), (130, 258, 257),
          (300, 287, 5), (1000, 513, 300), (2049, 768, 64), (700, 131, 4096), (700, 259, 4097), (200, 4096, 9),
          (5000, 512, 600)]


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


@pytest.mark.parametrize("scale,offset", [(1e-20, 0.0), (1e-38, 0.0), (1e18, 0.0), (1.0, -3e5)])
def test_labels_inside_the_band(engine, oracle, scale, offset):
    set_path(engine, "mfma_f32")
    x = (gaussian_mixture(900, 301, 20, seed=8, dtype=np.float64) * scale + offset).astype(np.float32)
    x[17, 3], x[400, 0], x[401, 300], x[899, 5] = np.nan, np.inf, -np.inf, 3e38
    c = x[20:60].copy()
    lab, _ = engine.infer(x, c)
    assert np.array_equal(lab, oracle.canonical_assign(x, c)[0])


@pytest.mark.parametrize("d,k", [(200, 40), (320, 150)])
def test_training_takes_open_rows(engine, oracle, d, k):
    set_path(engine, "mfma_f32")
    x = gaussian_mixture(4001, d, 30, seed=k, sigma=(2.0, 4.0))
    c0 = x[:k].copy()
    got = engine.train(x, c0, 12, 0.0)
    assert_bit_exact(got, oracle.canonical_lloyd(x, c0, 12, 0.0))
