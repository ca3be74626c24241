"""Batches on both sides of the rule on a plan's work, which tells the tile its instances
take: equal to the oracle bit for bit."""

import numpy as np
import pytest

from conftest import gaussian_mixture

pytestmark = pytest.mark.gpu


def run(engine, shapes, iters, graph=True):
    import torch

    xs = [gaussian_mixture(n, d, min(k, 20), seed=n + d + k, sigma=(0.5, 2.0)) for n, d, k in shapes]
    c0s = [x[:k].copy() for x, (_, _, k) in zip(xs, shapes)]
    cs, ls, objs, _ = engine.train_batch_device([torch.from_numpy(x).cuda() for x in xs],
                                                [torch.from_numpy(c).cuda() for c in c0s], iters, graph=graph)
    return xs, c0s, [c.cpu().numpy() for c in cs], [l.cpu().numpy() for l in ls], objs


# work 2e6, 5e8 and 1.7e9 (narrow tiles, the table twice), and 2e8 with a mean k of 9 (narrow tiles);
# k on both sides of 8 and 16
PLANS = [([(1000, 8, 4), (1500, 32, 8), (900, 64, 16), (700, 16, 17)], 6),
         ([(20000, 64, 128), (30000, 128, 80), (5000, 32, 8), (9000, 32, 16)], 6),
         ([(70000, 128, 128), (40000, 64, 100), (8000, 32, 8), (9000, 128, 16), (3000, 33, 30)], 16),
         ([(300000, 64, 9), (60000, 128, 8), (2000, 32, 40)], 5)]


@pytest.mark.parametrize("plan", PLANS, ids=["small", "middle", "large", "few_clusters"])
def test_plans_equal_the_oracle(engine, oracle, plan):
    shapes, iters = plan
    xs, c0s, cs, ls, objs = run(engine, shapes, iters)
    for x, c0, c, l, o in zip(xs, c0s, cs, ls, objs):
        wc, wl, wo, _ = oracle.canonical_lloyd(x, c0, iters, 0.0)[:4]
        assert np.array_equal(l, wl)
        assert np.array_equal(c.view(np.uint8), wc.view(np.uint8))
        assert o == wo
