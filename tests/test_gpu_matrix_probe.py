"""The choice between the matrix kernel and groups of lanes for many queries: by how
far apart the queries of a wave lie.  Either kernel gives the rows of four-lane
groups and of the CPU oracle."""
import numpy as np
import pytest

import oracle
import rtnn_amd

pytestmark = pytest.mark.gpu

MANY = 1 << 19  # queries from which a single cloud takes the matrix kernel


def clumps(seed, n, box=1000.0):
    rng = np.random.default_rng(seed)
    c = np.random.default_rng(1).uniform(0, box, (40, 3))
    return (c[rng.integers(0, 40, n)] + rng.normal(0, 5.0, (n, 3))).astype(np.float32)


def even(seed, n, side):
    return np.random.default_rng(seed).uniform(0, side, (n, 3)).astype(np.float32)


def check(ctx, pts, qs, r, k, want):
    ctx.set_points(pts)
    ctx.set_options()
    idx, d2, st = ctx.search(qs, mode="radius", radius=r, k=k)
    ctx.set_options(queries_per_wave=16)  # four lanes per query
    wi, wd, _ = ctx.search(qs, mode="radius", radius=r, k=k)
    ctx.set_options()
    assert np.array_equal(idx, wi) and np.array_equal(d2, wd)
    q = (pts if qs is None else qs)[7::4999]
    oi, od = oracle.grid_search(pts, q, oracle.MODE_RADIUS, r, k)
    assert np.array_equal(idx[7::4999], oi) and np.array_equal(d2[7::4999], od)
    assert st.lanes_per_query == want


@pytest.mark.parametrize("k", [5, 16, 17, 32])
@pytest.mark.parametrize("extra", [0, 1, 63])
def test_queries_unlike_the_points(ctx, k, extra):
    qs = even(k, MANY + extra, 1000.0)  # uniform over the box of the clumps
    qs[1000] = [np.nan, 1, 1]
    qs[2000] = [np.inf, 1, 1]
    qs[3000] = [3e38, -3e38, 0]
    pts = clumps(2, 300_000)
    check(ctx, pts, qs, 5.0, k, 16)


@pytest.mark.parametrize("k", [8, 32])
def test_queries_like_the_points(ctx, k):
    check(ctx, clumps(3, 200_000), clumps(4, MANY), 2.0, k, 1)
    check(ctx, even(5, MANY, 87.0), even(6, MANY, 87.0), 2.0, k, 1)


@pytest.mark.parametrize("r,want", [(0.2, 16), (1.5, 1)])
def test_points_as_queries(ctx, r, want):
    # one point for 150 cells (too far apart), and 2.7 a cell
    check(ctx, even(7, MANY, 87.0), None, r, 16, want)


@pytest.mark.parametrize("like,want", [(False, 2), (True, 1)])
def test_knn_at_proposed_radii(ctx, like, want):
    pts = clumps(8, 500_000)
    qs = clumps(9, MANY) if like else even(9, MANY, 1000.0)
    ctx.set_points(pts)
    ctx.mlp_train(5.0, 16, n_samples=20000, steps=40, batch=1000, seed=1)
    want_rows = ctx.search(qs, mode="knn", radius=5.0, k=16)
    ctx.set_options(cell_factor=2.0, queries_per_wave=32, grid_levels=1, group_buffer=2)
    try:
        got = ctx.search_learned(qs, radius=5.0, k=16)
    finally:
        ctx.set_options()
    assert np.array_equal(got[0], want_rows[0]) and np.array_equal(got[1], want_rows[1])
    assert got[2].lanes_per_query == want
