"""Plain KNN by the cells or by packets of queries, as the cells' filling has it:
every route at its edges (numbers of queries, list sizes, all points or a sample
of them, hashed or exact counters) gives the rows of the packet walk."""
import numpy as np
import pytest

import oracle
import rtnn_amd

pytestmark = pytest.mark.gpu

PACKETS = 1 << 10  # cells per axis of the packet walk's order


def route(st):
    return 0 if list(st.grid_dims) == [PACKETS] * 3 else st.lanes_per_query


def both(ctx, qs, r, k):
    ctx.set_options()
    idx, d2, st = ctx.search(qs, mode="knn", radius=r, k=k)
    ctx.set_options(queries_per_wave=64)
    wi, wd, ws = ctx.search(qs, mode="knn", radius=r, k=k)
    ctx.set_options()
    assert route(ws) == 0
    assert np.array_equal(idx, wi) and np.array_equal(d2, wd)
    return idx, d2, route(st)


# points per unit cell -> lanes (0: packets), 20,000 queries or 150,000
@pytest.mark.parametrize("k", [1, 8, 9, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("n,mean,few,many", [
    (16384, 40.0, 16, None), (16384, 90.0, 0, None), (30000, 1.5, 4, None),
    (30000, 10.0, 16, None), (30000, 40.0, 0, None),
    (131072, 1.0, 4, None), (131073, 1.0, 4, {1: 1, 8: 1}), (200000, 40.0, 0, {}),
    (400000, 5.0, 16, {1: 1, 8: 1, 9: 16, 16: 16})])
def test_uniform(ctx, k, n, mean, few, many):
    side = (n / mean) ** (1 / 3)
    pts = rtnn_amd.gen_uniform(n % 97 + k, n, 0.0, side)
    ctx.set_points(pts)
    qs = pts if n <= 20000 else pts[:20000] + np.float32(0.1)
    idx, d2, got = both(ctx, qs, 1.0, k)
    assert got == (16 if len(qs) <= 1 << 14 and mean < 60 else few)
    sub = slice(0, 300)
    wi, wd = oracle.grid_search(pts, qs[sub], oracle.MODE_KNN, 1.0, k)
    assert np.array_equal(idx[sub], wi) and np.array_equal(d2[sub], wd)
    if many is not None:
        want = 0 if not many else many.get(k, 4)
        assert both(ctx, pts[:150000], 1.0, k)[2] == want


def test_uneven_points(ctx):
    # a hot cell; a far point that makes more cells than counters (hashed) and
    # one that makes the cells grow until everything is in one; one place, one
    # point; a grid held to few cells
    rng = np.random.default_rng(5)
    spread = rng.uniform(0, 60, (170000, 3)).astype(np.float32)
    hot = spread.copy()
    hot[::3] = rng.normal(30, 0.2, (len(hot[::3]), 3))
    ctx.set_points(hot)
    assert both(ctx, hot[:140000], 1.0, 8)[2] == 0
    for at, want in ((160.0, 1), (9000.0, 0)):
        far = spread.copy()
        far[7] = at
        ctx.set_points(far)
        assert both(ctx, far[:140000], 1.0, 8)[2] == want
    for p in (np.full((5000, 3), 2.5, np.float32), np.full((1, 3), 2.5, np.float32)):
        ctx.set_points(p)
        both(ctx, p, 1.0, 5)
    ctx.set_points(spread[:3000])
    ctx.set_options(max_cells=64)
    idx, d2, _ = ctx.search(spread[:500], mode="knn", radius=4.0, k=7)
    ctx.set_options()
    wi, wd = oracle.bruteforce(spread[:3000], spread[:500], oracle.MODE_KNN, 4.0, 7)
    assert np.array_equal(idx, wi) and np.array_equal(d2, wd)
