"""Sparse training that leaves out rows whose bounds prove their label (km_csr.hpp):
equal to the oracle bit for bit when most rows are skipped, with the objective needed in
every iteration or only at the end, with refilled clusters, and where the bounds
cannot be used (repeated columns, a norm far above the others)."""
import numpy as np
import pytest

from test_gpu_csr import check_train
from test_oracle_csr import reorder, sparse_blobs

pytestmark = pytest.mark.gpu

# n, d, k, density, iterations, threshold, dtype: one row a run and several, rows of
# more than 64 entries, a run's remainder, one block of centroids and several
CASES = [(1, 5, 1, 0.9, 3, 0.0, np.float32), (3001, 40, 7, 0.3, 25, 0.0, np.float32),
         (140003, 60, 9, 0.1, 12, 0.0, np.float64), (20011, 400, 20, 0.25, 15, 1e-6, np.float32),
         (5003, 30, 1100, 0.3, 6, 0.0, np.float32), (3000, 4096, 12, 0.01, 8, 0.0, np.float32),
         (3000, 17, 256, 0.4, 8, 1e-6, np.float64)]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "n%d_d%d_k%d_%s" % (c[0], c[1], c[2], np.dtype(c[6]).name))
def test_skipped_rows_change_nothing(engine, oracle, case):
    n, d, k, dens, iters, thr, dtype = case
    x, _ = sparse_blobs(n, d, min(k, 40), dens, seed=n + d, dtype=dtype, base=0)
    c0 = x.to_dense()[np.random.default_rng(k).choice(n, k, replace=False)]
    check_train(engine, oracle, x, c0, iters, thr)


@pytest.mark.parametrize("thr", [0.0, 1e-6])
def test_refilled_clusters(engine, oracle, thr):
    x, _ = sparse_blobs(6000, 50, 8, 0.2, seed=3, dtype=np.float32, base=1)
    c0 = np.repeat(x.to_dense()[:4], 3, axis=0)
    check_train(engine, oracle, x, c0, 12, thr)
    assert engine.stats()["empty_cluster_events"] >= 1


def test_one_huge_row_and_reordered_columns(engine, oracle):
    x, _ = sparse_blobs(4000, 50, 8, 0.2, seed=5, dtype=np.float32, base=0)
    c0 = x.to_dense()[:8]
    check_train(engine, oracle, reorder(x, 2, 0), c0, 8, 0.0)
    x.values[7] = 1e12  # every band is far wider than the distances
    check_train(engine, oracle, x, x.to_dense()[:8], 8, 0.0)


@pytest.mark.parametrize("k,dtype,scale", [(1, np.float32, 1.0), (256, np.float32, 1e-20), (257, np.float32, 1.0),
                                           (1024, np.float32, 1e17), (1025, np.float32, 1.0), (128, np.float64, 1e-23),
                                           (129, np.float64, 1.0), (512, np.float64, 1e60), (513, np.float64, 1.0)])
def test_rough_distances_and_ties(engine, oracle, k, dtype, scale):
    """Edges of the centroids per lane; every second centroid is a copy or nearly one, so
    rough distances cannot tell them apart; values near and past the float range."""
    x, _ = sparse_blobs(2000, 70, 30, 0.3, seed=k, dtype=dtype, base=1)
    x.values *= dtype(scale)
    c = x.to_dense()[:k].copy()
    c[1::2] = c[: c[1::2].shape[0] * 2 : 2]
    c[3::4] *= dtype(1.0 + 1e-6)
    labels, obj = engine.infer_csr(x.values, x.cols, x.offs, x.d, c, base=1, objective=True)
    rl, closest = oracle.csr_assign(x, c)
    assert np.array_equal(labels, rl)
    assert obj == oracle.csr_objective(closest)
