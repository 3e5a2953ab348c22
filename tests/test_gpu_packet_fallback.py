"""KNN of the proposal methods on hierarchical grids: packets at r whatever lanes are
asked for (no row is short, however poor the network); rows equal the plain search's."""
import numpy as np
import pytest

import rtnn_amd
from oracle import mlp_ref as M

pytestmark = pytest.mark.gpu


def check(ctx, qs, r, k, search, **opts):
    ctx.set_options()
    wi, wd, _ = ctx.search(qs, mode="knn", radius=r, k=k)
    ctx.set_options(**opts)
    try:
        idx, d2, st = search(qs, radius=r, k=k)
    finally:
        ctx.set_options()
    assert np.array_equal(idx, wi) and np.array_equal(d2, wd)
    return st


@pytest.mark.parametrize("opts", [{}, {"queries_per_wave": 16}, {"queries_per_wave": 4},
                                  {"learned_cap": 1}, {"queries_per_wave": 32, "group_buffer": 3}])
@pytest.mark.parametrize("k", [1, 16, 64])
def test_no_short_rows(ctx, k, opts):
    if k > 16 and opts.get("queries_per_wave") == 32:
        k = 16
    pts = rtnn_amd.gen_uniform(3, 60000, 0.0, 40.0)
    qs = rtnn_amd.gen_uniform(4, 5000, -1.0, 41.0)
    ctx.set_points(pts)
    # o = 0: the network proposes its least radius for every query
    ctx.set_mlp_weights(np.concatenate([np.zeros(M.NP), [0.25, 1.0]]).astype(np.float32))
    st = check(ctx, qs, 3.0, k, ctx.search_learned, grid_levels=5, **opts)
    assert st.fallback_queries == 0 and st.lanes_per_query == 1
    st = check(ctx, qs, 3.0, k, ctx.search_partitioned, grid_levels=5, **opts)
    assert st.fallback_queries == 0 and st.lanes_per_query == 1
