"""Precision of the products that float rows are assigned by.  The rows that an
assignment re-scores are those with a second centroid inside the error band, and the
band is proven from the products' error: their number tells which products ran."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def rows_in_fp32_band(x, c):
    """Rows whose second centroid lies within the band of FP32 products (km_common.hpp)."""
    d = x.shape[1]
    x, c = x.astype(np.float64), c.astype(np.float64)
    xn, cn = (x * x).sum(1), (c * c).sum(1)
    dist = np.sort(xn[:, None] - 2.0 * x @ c.T + cn, axis=1)
    u, ua = 2.0 ** -24, 2.0 ** -23
    cmax = np.sqrt(cn.max())
    da = (2.0 * d * ua + 2.01 * u) * np.sqrt(xn) * cmax + 2.01 * u * cmax * cmax
    g = (d + 2) * u
    return int((dist[:, 1] - dist[:, 0] <= 2.0 * da + 2.0 * g * (dist[:, 0] + da)).sum())


def data(d):
    """Rows far from the origin without clusters: about a fifth have two near centroids."""
    rng = np.random.default_rng(d)
    return (rng.uniform(-10, 10, (20000, d)) + 100.0).astype(np.float32)


@pytest.mark.parametrize("d", [16, 64, 127, 200])
def test_fp32_products_can_be_asked_for(engine, oracle, d):
    """KM_OPT_ASSIGN_PATH 2: the band is that of FP32 products (5%: values near its edge)."""
    from onedal_amd.engine import KM_OPT_ASSIGN_PATH

    x = data(d)
    c = x[:200].copy()
    engine.set_option(KM_OPT_ASSIGN_PATH, 2)
    lab, _ = engine.infer(x, c)
    engine.set_option(KM_OPT_ASSIGN_PATH, 0)
    st = engine.stats()
    want = rows_in_fp32_band(x, c)
    assert want > 300
    assert abs(st["refined_candidate_rows"] + st["refined_full_rows"] - want) < 0.05 * want
    assert np.array_equal(lab, oracle.canonical_assign(x, c)[0])


def test_fp32_option_past_256_columns(engine):
    from onedal_amd.engine import KM_OPT_ASSIGN_PATH

    x = data(257)[:500]
    engine.set_option(KM_OPT_ASSIGN_PATH, 2)
    engine.infer(x, x[:20].copy())
    engine.set_option(KM_OPT_ASSIGN_PATH, 0)
    assert engine.stats()["assign_path"] == 1
