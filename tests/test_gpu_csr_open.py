"""Sparse training with bounds where they settle little or nothing: rows in random
columns, copied and nearly copied centroids, every number of centroids per lane, values
near the ends of the type.  Equal to the oracle bit for bit, with the objective (the
closest distances of settled and of assigned rows) needed in every iteration or not."""
import numpy as np
import pytest

from test_gpu_csr import check_train
from test_oracle_csr import sparse_blobs

pytestmark = pytest.mark.gpu


def random_rows(n, d, m, seed, dtype, base):
    from oracle.oracle import Csr

    rng = np.random.default_rng(seed)
    cols = np.sort(rng.permuted(np.tile(np.arange(d), (n, 1)), axis=1)[:, :m], axis=1)
    vals = rng.uniform(1.0, 6.0, size=n * m).astype(dtype)
    return Csr(vals, cols.reshape(-1).astype(np.int64) + base, np.arange(n + 1, dtype=np.int64) * m + base, d, base)


@pytest.mark.parametrize("thr", [0.0, 1e-9])
@pytest.mark.parametrize("n,d,m,k,dtype", [(4001, 60, 9, 20, np.float32), (3000, 300, 70, 300, np.float32),
                                           (3000, 90, 16, 140, np.float64)])
def test_random_columns(engine, oracle, n, d, m, k, dtype, thr):
    x = random_rows(n, d, m, k, dtype, 1)
    check_train(engine, oracle, x, x.to_dense()[:k], 7, thr)


@pytest.mark.parametrize("iters,thr", [(0, 0.0), (3, 0.0), (3, 1e-6)])
@pytest.mark.parametrize("k,dtype,scale", [(1, np.float32, 1.0), (256, np.float32, 1e-20), (257, np.float32, 1.0),
                                           (512, np.float32, 1.0), (513, np.float32, 1.0), (1024, np.float32, 1e17),
                                           (1025, np.float32, 1.0), (128, np.float64, 1e-23), (129, np.float64, 1.0),
                                           (256, np.float64, 1.0), (257, np.float64, 1.0), (512, np.float64, 1e60),
                                           (513, np.float64, 1.0)])
def test_centroids_per_lane_and_ties(engine, oracle, k, dtype, scale, iters, thr):
    x, _ = sparse_blobs(2000, 70, 30, 0.3, seed=k, dtype=dtype, base=1)
    x.values *= dtype(scale)
    c = x.to_dense()[:k].copy()
    c[1::2] = c[: c[1::2].shape[0] * 2 : 2]
    c[3::4] *= dtype(1.0 + 1e-6)
    check_train(engine, oracle, x, c, iters, thr)
