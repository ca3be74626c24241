"""Batches on both sides of the rules on a plan's work: which tile its instances take and
whether it keeps bounds.  Equal to the oracle bit for bit, and small batches keep no
bounds (their memory tells)."""

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


# work 2e6, 5e8 and 1.7e9 (narrow tiles, the table twice), 2e8 with a mean k of 9
# (narrow tiles), and with one kind either way (the table);
# iterations times work below and above 2e10; k on both sides of 8 and 16
PLANS = [([(1000, 8, 4), (1500, 32, 8), (900, 64, 16), (700, 16, 17)], 6),
         ([(20000, 64, 128), (30000, 128, 80), (5000, 32, 8), (9000, 32, 16)], 6),
         ([(70000, 128, 128), (40000, 64, 100), (8000, 32, 8), (9000, 128, 16), (3000, 33, 30)], 16),
         ([(300000, 64, 9), (60000, 128, 8), (2000, 32, 40)], 5), ([(900000, 16, 10)], 5)]


@pytest.mark.parametrize("plan", PLANS, ids=["small", "middle", "large", "few_clusters", "one_kind"])
def test_plans_equal_the_oracle(engine, oracle, plan):
    shapes, iters = plan
    xs, c0s, cs, ls, objs = run(engine, shapes, iters)
    for x, c0, c, l, o in zip(xs, c0s, cs, ls, objs):
        wc, wl, wo, _ = oracle.canonical_lloyd(x, c0, iters, 0.0)[:4]
        assert np.array_equal(l, wl)
        assert np.array_equal(c.view(np.uint8), wc.view(np.uint8))
        assert o == wo


def test_a_small_batch_keeps_no_bounds():
    """Four million rows of 2 columns and 2 clusters: labels, ids, d64 and chunk sums are 17 bytes a
    row; labels before and gaps would be 8 more."""
    import torch

    from onedal_amd.engine import Engine

    eng = Engine(0)
    n = 4_000_000
    x = torch.rand((n, 2), device="cuda")
    c = x[:2].clone()
    out = ([torch.empty_like(c)], [torch.empty(n, device="cuda", dtype=torch.int32)])
    eng.train_batch_device([x[:1000]], [c], 5, graph=False)
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    eng.train_batch_device([x], [c], 5, graph=False, outs=out)
    torch.cuda.synchronize()
    got = free - torch.cuda.mem_get_info()[0]
    eng.close()
    assert got < 20 * n
