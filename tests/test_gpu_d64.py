"""Row distances of the objective (row_d64_kernel): the objective equals the oracle's bit
for bit at the edges of a wave's rows and of a row's pieces, in both types, with rows
and centroids at any alignment, and a value that is not finite."""

import numpy as np
import pytest

from conftest import gaussian_mixture

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("n,d", [(1, 1), (63, 2), (64, 3), (65, 15), (255, 16), (256, 17), (257, 31), (300, 32),
                                 (301, 33), (1000, 65), (500, 257)])
def test_objective_bits(engine, oracle, n, d, dtype):
    import torch

    k = min(n, 5)
    x = gaussian_mixture(n, d, k, seed=n + d, dtype=np.float64).astype(dtype)
    if n == 301:
        x[7, 3] = np.inf
    c = x[:k].copy()
    want, _ = oracle.canonical_assign(x, c)
    obj = oracle.canonical_objective(x, c, want)
    for shift in (0, 1):  # elements past a 16-byte boundary
        flat = torch.empty(n * d + k * d + 2, dtype=getattr(torch, np.dtype(dtype).name), device="cuda")
        xs = flat[shift:shift + n * d].view(n, d)
        cs = flat[shift + n * d:shift + n * d + k * d].view(k, d)
        xs.copy_(torch.from_numpy(x))
        cs.copy_(torch.from_numpy(c))
        torch.cuda.synchronize()
        lab, got = engine.infer(xs, cs, objective=True)
        assert np.array_equal(lab.cpu().numpy(), want)
        assert got == obj or (np.isnan(got) and np.isnan(obj))
