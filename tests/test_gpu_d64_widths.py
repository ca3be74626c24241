"""The objective on rows of one to nine 16-byte vectors (row_d64_kernel's pieces), whole and
ragged, with a wave's last rows missing: equal to the oracle's, bit for bit."""

import numpy as np
import pytest

from conftest import gaussian_mixture
from test_gpu_parity import set_path

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("d", [1, 2, 3, 4, 5, 8, 9, 15, 16, 17, 33])
def test_objective_of_narrow_rows(engine, oracle, d, dtype):
    set_path(engine, "bf16")
    for n in (1, 63, 65, 4097):
        x = gaussian_mixture(max(n, 6), d, 6, seed=n + d, dtype=dtype)[:n].copy()
        c = gaussian_mixture(6, d, 6, seed=d, dtype=dtype)
        lab, obj = engine.infer(x, c, objective=True)
        wl, _ = oracle.canonical_assign(x, c)
        assert np.array_equal(lab, wl)
        assert obj == oracle.canonical_objective(x, c, wl)
