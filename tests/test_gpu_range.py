"""Rows and centroids near the end of the float range, where a squared norm is still a
float but twice it is not: 2 x.c passes the largest float for the very centroid that is
nearest.  Such rows are re-scored in the exact form, so the labels are the oracle's."""

import numpy as np
import pytest

from test_gpu_parity import set_path

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("norm2", [0.9e38, 1.75e38, 3.2e38])
@pytest.mark.parametrize("d", [12, 33, 128, 200, 513])
@pytest.mark.parametrize("path", ["auto", "bf16"])
def test_norms_near_the_float_range(engine, oracle, path, d, norm2):
    set_path(engine, "bf16")  # option 0; the flag below asks for BF16 distances
    rng = np.random.default_rng(d)
    u = rng.standard_normal((10, d))
    u *= np.sqrt(norm2) / np.linalg.norm(u, axis=1, keepdims=True)
    # a direction's own centroid, and one at 0.8 of it, whose products stay in range
    c = np.concatenate([0.8 * u, u]).astype(np.float32)
    x = (u[rng.integers(0, 10, 400)] * (1.0 - 1e-3 * rng.random((400, 1)))).astype(np.float32)
    want = oracle.canonical_assign(x, c)[0]
    assert np.array_equal(engine.infer(x, c, bf16=path == "bf16")[0], want)
    assert np.array_equal(engine.train(x, c, 0, 0.0, bf16=path == "bf16")[1], want)
