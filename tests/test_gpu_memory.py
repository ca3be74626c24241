"""Device memory that a call leaves with its context, in bytes a row of the data."""

import pytest

pytestmark = pytest.mark.gpu

N = 8_000_000


def taken(call):
    """Bytes that the device has less after call()."""
    import torch

    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    call()
    torch.cuda.synchronize()
    return free - torch.cuda.mem_get_info()[0]


@pytest.fixture(scope="module")
def rows():
    import torch

    return torch.rand((N, 4), device="cuda", generator=torch.Generator("cuda").manual_seed(1))


def test_the_objective_takes_no_memory_of_its_own(rows):
    from onedal_amd.engine import Engine

    eng = Engine(0)
    c = rows[:5].clone()
    eng.infer(rows, c)
    got = taken(lambda: eng.infer(rows, c, objective=True))
    eng.close()
    assert got < 2 * N  # chunk sums, and the allocator's granularity


def test_training_takes_no_more_than_without_bounds(rows):
    """Without bounds: norm 4, lists 44, ids 4, d64 8, labels out 4, chunk sums, histograms
    and granularity 4; with them 16 a row for gap, bound, label before and open rows."""
    from onedal_amd.engine import Engine

    eng = Engine(0)
    c = rows[:5].clone()
    eng.infer(rows[:1000], c)
    got = taken(lambda: eng.train(rows, c, 3, 0.0))
    eng.close()
    assert got < 68 * N
