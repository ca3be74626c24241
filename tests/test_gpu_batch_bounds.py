"""Batched training over enough iterations to keep bounds (five and more): every
instance equals the oracle's training of it alone, bit for bit, whatever tile
variant assigns it."""

import numpy as np
import pytest

from conftest import gaussian_mixture

pytestmark = pytest.mark.gpu

# n, d, k: one row, one cluster, an item and a row, odd widths, every matrix-core
# width, tiles of several chunks of features, and clusters that start empty
SIZES = [(1, 3, 1), (50, 4, 50), (129, 16, 7), (4097, 8, 5), (5000, 33, 40), (9000, 17, 12), (3000, 64, 128),
         (2500, 100, 33), (1500, 200, 20), (6000, 128, 65), (700, 300, 9), (800, 12, 130)]


@pytest.mark.parametrize("iters", [4, 5, 12])
@pytest.mark.parametrize("variant", [0, 1, 4, 8], ids=["default", "tile64x8", "tile16x8", "matrix_cores"])
@pytest.mark.parametrize("graph", [False, True])
def test_batch_with_bounds(engine, oracle, variant, iters, graph):
    import torch

    from onedal_amd.engine import KM_OPT_BATCH_TILE

    xs, c0s = [], []
    for i, (n, d, k) in enumerate(SIZES):
        x = gaussian_mixture(n, d, max(1, min(k, 12)), seed=i, sigma=(0.5, 2.0))
        pick = np.random.default_rng(i).choice(n, size=k, replace=False)
        if i == 3:
            pick[:] = pick[0]  # all but one cluster start empty
        xs.append(x)
        c0s.append(x[pick].copy())
    engine.set_option(KM_OPT_BATCH_TILE, variant)
    try:
        cs, ls, objs, its = engine.train_batch_device([torch.from_numpy(x).cuda() for x in xs],
                                                      [torch.from_numpy(c).cuda() for c in c0s], iters, graph=graph)
    finally:
        engine.set_option(KM_OPT_BATCH_TILE, 0)
    for x, c0, c, lab, obj, it in zip(xs, c0s, cs, ls, objs, its):
        wc, wl, wo, wi = oracle.canonical_lloyd(x, c0, iters, 0.0)[:4]
        assert it == wi
        assert np.array_equal(lab.cpu().numpy(), wl)
        assert np.array_equal(c.cpu().numpy(), wc)
        assert obj == wo
