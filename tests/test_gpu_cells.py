"""Raster grids built by counting (up to 2^20 points): edges of the scan's
blocks (4096 cells, one block up to 65536), hot cells, and one context whose
counters serve grids of many sizes in turn.  Rows against the CPU oracle."""
import numpy as np
import pytest

import oracle
import rtnn_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells", [(1, 1, 1), (3, 1, 2), (16, 16, 16), (17, 241, 1), (64, 32, 32),
                                   (65, 32, 32), (41, 41, 39), (90, 7, 200)])
def test_table_sizes(ctx, cells):
    # the box is cells x edge r, so the table holds exactly these cells
    rng = np.random.default_rng(sum(cells))
    n = int(rng.integers(700, 4000))
    pts = (rng.uniform(0, 1, (n, 3)) * np.array(cells) * 0.999).astype(np.float32)
    pts[0] = 0
    ctx.set_points(pts)
    idx, d2, st = ctx.search(None, mode="radius", radius=1.0, k=24)
    assert st.sort_passes == 0  # counted, not sorted
    wi, wd = oracle.grid_search(pts, pts, oracle.MODE_RADIUS, 1.0, 24)
    assert np.array_equal(idx, wi) and np.array_equal(d2, wd)


def test_hot_cells_and_regrown_tables(ctx):
    # almost all points in one cell, in input order and shuffled; then smaller
    # and larger tables on the same counters
    rng = np.random.default_rng(3)
    hot = np.concatenate([rng.uniform(0, 0.5, (3000, 3)), rng.uniform(0, 30, (300, 3))])
    for p in (hot, rng.permutation(hot)):
        p = p.astype(np.float32)
        ctx.set_points(p)
        for r in (0.4, 1.5, 0.2, 9.0):
            idx, d2, _ = ctx.search(None, mode="radius", radius=r, k=16)
            wi, wd = oracle.bruteforce(p, p, oracle.MODE_RADIUS, r, 16)
            assert np.array_equal(idx, wi) and np.array_equal(d2, wd)


def test_counting_and_sorting_agree(ctx):
    # just above and below 2^20 points: the same rows for the common queries
    pts = rtnn_amd.gen_uniform(7, (1 << 20) + 64, 0.0, 100.0)
    qs = rtnn_amd.gen_uniform(8, 5000, 0.0, 100.0)
    rows = []
    for n in (1 << 20, (1 << 20) + 1):
        p = pts[:n].copy()
        p[1 << 20:] = 500.0  # outside every query's reach
        ctx.set_points(p)
        idx, d2, st = ctx.search(qs, mode="radius", radius=2.0, k=48)
        rows.append((idx, d2, st.sort_passes))
    assert rows[0][2] == 0 and rows[1][2] > 0
    assert np.array_equal(rows[0][0], rows[1][0]) and np.array_equal(rows[0][1], rows[1][1])
