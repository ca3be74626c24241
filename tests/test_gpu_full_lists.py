"""The full re-score (refine_full_vec_kernel) of lists on both sides of the lengths at
which four, two or one wave take a row: rows far from the origin, nearly all of which
have more candidates than a list entry holds."""

import numpy as np
import pytest

from test_gpu_parity import assert_bit_exact, set_path

pytestmark = pytest.mark.gpu


def far_rows(n, d):
    return (np.random.default_rng(n).uniform(-1, 1, (n, d)) + 3000.0).astype(np.float32)


@pytest.mark.parametrize("n", [700, 8300, 16700, 33000])
@pytest.mark.parametrize("k", [60, 100, 300])
def test_labels_of_long_lists(engine, oracle, n, k):
    set_path(engine, "bf16")
    x = far_rows(n, 20)
    c = x[np.random.default_rng(k).permutation(n)[:k]].copy()
    lab, _ = engine.infer(x, c)
    assert engine.stats()["refined_full_rows"] > 0.97 * n
    assert np.array_equal(lab, oracle.canonical_assign(x, c)[0])


@pytest.mark.parametrize("n", [8300, 16700])
def test_training_with_long_lists(engine, oracle, n):
    set_path(engine, "bf16")
    x = far_rows(n, 12)
    got = engine.train(x, x[:150].copy(), 4, 0.0)
    assert_bit_exact(got, oracle.canonical_lloyd(x, x[:150].copy(), 4, 0.0))
