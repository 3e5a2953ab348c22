"""The packet walk where there are few queries: one or several per wave up to whole
packets, given as queries or as a list of short rows; rows equal those of groups."""
import numpy as np
import pytest

import rtnn_amd
from oracle import mlp_ref as M

pytestmark = pytest.mark.gpu


def check(ctx, qs, r, k, search, **opts):
    ctx.set_options(queries_per_wave=4)  # 16 lanes over the cells
    wi, wd, _ = ctx.search(qs, mode="knn", radius=r, k=k)
    ctx.set_options(**opts)
    try:
        idx, d2, st = search(qs, radius=r, k=k)
    finally:
        ctx.set_options()
    assert np.array_equal(idx, wi) and np.array_equal(d2, wd)
    return st


# one query a wave up to 4 waves a CU and SIMD (1024, 2048 or 4096 waves), two a
# wave from there on, packets of 64
@pytest.mark.parametrize("k", [4, 16, 32, 64])
@pytest.mark.parametrize("nq", [1, 5, 1023, 1025, 2049, 4095, 4097, 65537, 300001])
def test_few_queries(ctx, nq, k):
    pts = rtnn_amd.gen_gaussian_mixture(5, 50000, 20000)
    qs = rtnn_amd.gen_gaussian_mixture(5, 51000, nq)
    qs[nq // 2] = [np.nan, 0, 0]
    ctx.set_points(pts)
    st = check(ctx, qs, 15.0, k, ctx.search_partitioned)
    assert st.lanes_per_query == 1


# short rows of a stage: none, fewer than the waves of a launch, about one or two a
# wave, a whole packet for some
@pytest.mark.parametrize("nq", [1, 63, 8191, 8193, 70001, 600001])
def test_short_rows_over_the_waves(ctx, nq):
    pts = rtnn_amd.gen_gaussian_mixture(5, 50000, 50000)
    qs = rtnn_amd.gen_gaussian_mixture(5, 51000, nq)
    ctx.set_points(pts)
    ctx.set_mlp_weights(np.concatenate([np.zeros(M.NP), [0.25, 1.0]]).astype(np.float32))
    st = check(ctx, qs, 15.0, 8, ctx.search_learned, grid_levels=5, tree_fallback=1)
    assert st.fallback_queries > 0.5 * nq
