"""Rows and clusters that a training iteration skips (km_bounds.hpp): a row whose
bounds prove its label, a cluster whose members did not change.  Skipping changes
no result, so every training equals the oracle bit for bit: labels, centroids,
objective and iteration count."""

import numpy as np
import pytest

from conftest import gaussian_mixture
from test_gpu_parity import assert_bit_exact, set_path

pytestmark = pytest.mark.gpu

CASES = [
    # name, n, d, k, iterations, scale, threshold: run to the fixed point (nothing
    # left to assign), the edges of the 4096-row runs, squares near underflow and
    # distances past the bounds' largest (every row assigned again), the stop rule,
    # k above the counting sort's (clusters not tracked)
    ("to_fixed_point", 30011, 17, 23, 30, 1.0, 0.0),
    ("one_run_exact", 4096, 8, 5, 12, 1.0, 0.0),
    ("one_run_and_a_row", 4097, 33, 40, 12, 1.0, 0.0),
    ("tiny_values", 5000, 12, 9, 10, 1e-21, 0.0),
    ("huge_values", 5000, 12, 9, 10, 3e17, 0.0),
    ("offset_rows", 20000, 20, 16, 10, 1.0, 0.0),
    ("stop_rule", 12001, 64, 30, 40, 1.0, 1e-3),
    ("k_above_counting_sort", 9000, 4, 4500, 3, 1.0, 0.0),
    # the largest grouping in one workgroup and the first past it; rows staged for
    # their d64 in several pieces (odd widths)
    ("small_group_largest", 16384, 3, 1024, 4, 1.0, 0.0),
    ("small_group_past", 16385, 3, 1025, 4, 1.0, 0.0),
    ("d64_pieces", 5001, 51, 7, 4, 1.0, 1e-3),
]


@pytest.mark.parametrize("path,dtype", [("mfma_f32", np.float32), ("generic", np.float32), ("bf16", np.float32),
                                        ("mfma_f32", np.float64)], ids=["f32", "generic", "bf16", "f64"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: c[0])
def test_skipped_rows_and_clusters_change_nothing(engine, oracle, case, path, dtype):
    name, n, d, k, iters, scale, thr = case
    bf16 = set_path(engine, path)
    x = gaussian_mixture(n, d, min(k, 64), seed=n + d, center_range=10.0, sigma=(0.5, 2.0), dtype=np.float64)
    if name == "offset_rows":  # a wide error band: few rows are certain
        x = x + 500.0
    x = (x * scale).astype(dtype)
    c0 = x[np.random.default_rng(n).choice(n, size=k, replace=False)].copy()
    got = engine.train(x, c0, iters, thr, bf16=bf16)
    assert_bit_exact(got, oracle.canonical_lloyd(x, c0, iters, thr))


def test_moved_and_refilled_clusters(engine, oracle):
    """Two coincident groups of centroids start empty, are refilled with far rows and
    take members in later iterations, while other clusters stay unchanged."""
    set_path(engine, "mfma_f32")
    x = gaussian_mixture(20000, 6, 12, seed=4)
    c0 = np.concatenate([x[:4], x[:4], x[:4]]).copy()
    got = engine.train(x, c0, 15, 0.0)
    assert engine.stats()["empty_cluster_events"] >= 1
    assert_bit_exact(got, oracle.canonical_lloyd(x, c0, 15, 0.0))
