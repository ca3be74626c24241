"""BF16 inference straight from the float rows (assign_split_kernel with one piece), whose open
rows take the three-piece kernel and then the re-scores: equal to the oracle's
exact-form argmin at the edges of its tiles, planes and index bits, where the band decides,
and on inputs that send every row down the whole chain."""

import numpy as np
import pytest

from conftest import gaussian_mixture
from test_gpu_parity import set_path
from test_gpu_split import SHAPES

pytestmark = pytest.mark.gpu

# two row blocks at every padded width (32, 64, 128), a tile and a row, one block of centroids
# and one more, every remainder of a width mod 4
MORE = [(1, 128, 1), (256, 32, 32), (257, 31, 33), (513, 64, 129), (511, 126, 128), (2000, 125, 257), (700, 3, 40),
        (3000, 128, 4096)]


@pytest.mark.parametrize("shape", SHAPES + MORE, ids=lambda s: "n%d_d%d_k%d" % s)
def test_labels_equal_exact_form(engine, oracle, shape):
    n, d, k = shape
    set_path(engine, "bf16")
    x = gaussian_mixture(max(n, k), d, min(k, 50), seed=n + d, sigma=(0.5, 2.0))
    c = x[np.random.default_rng(k).permutation(x.shape[0])[:k]].copy()
    x = x[:n].copy()
    lab, obj = engine.infer(x, c, objective=True, bf16=True)
    wl, _ = oracle.canonical_assign(x, c)
    assert np.array_equal(lab, wl)
    assert obj == oracle.canonical_objective(x, c, wl)


@pytest.mark.parametrize("d", [24, 60, 127])
@pytest.mark.parametrize("scale,offset", [(1.0, 1e4), (1e-20, 0.0), (1e-38, 0.0), (1e18, 0.0), (3e18, 0.0), (1.0, -3e5)])
def test_labels_inside_the_band(engine, oracle, d, scale, offset):
    set_path(engine, "bf16")
    x = (gaussian_mixture(3000, d, 20, seed=8, dtype=np.float64) * scale + offset).astype(np.float32)
    x[17, 3], x[400, 0], x[401, d - 1], x[899, 5] = np.nan, np.inf, -np.inf, 3e38
    c = x[20:60].copy()
    lab, _ = engine.infer(x, c, bf16=True)
    assert np.array_equal(lab, oracle.canonical_assign(x, c)[0])


@pytest.mark.parametrize("n,d,k", [(5000, 128, 200), (3001, 33, 40), (2000, 64, 3)])
def test_every_row_down_the_chain(engine, oracle, n, d, k):
    set_path(engine, "bf16")
    x = (np.random.default_rng(d).uniform(-1, 1, (n, d)) + 300.0).astype(np.float32)
    c = x[:k].copy()
    lab, _ = engine.infer(x, c, bf16=True)
    st = engine.stats()
    assert st["refined_candidate_rows"] + st["refined_collect_rows"] > 0.99 * n
    assert np.array_equal(lab, oracle.canonical_assign(x, c)[0])
