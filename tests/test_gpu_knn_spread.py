"""Plain KNN at the lines of its rule on many points: few queries (a smaller
sample of the points' cells), a list of up to four keys, and lists of 9 to 16 with
more than 2^19 queries.  The rows are those of the packet walk."""
import numpy as np
import pytest

import oracle
import rtnn_amd

pytestmark = pytest.mark.gpu

PACKETS = [1 << 10] * 3  # cells per axis of the packet walk's order


# points per cell of edge 1 (one more in a point's own) -> lanes (0: packets); 2^18
# points is the largest set whose sums the runtime waits for
@pytest.mark.parametrize("n,nq,mean,k,want", [
    (1 << 18, 1 << 14, 40.0, 8, 16), ((1 << 18) + 1, 1 << 14, 40.0, 16, 16),
    (600000, 1 << 14, 90.0, 8, 0), (600000, (1 << 14) + 1, 40.0, 8, 0),
    (600000, 1, 5.0, 4, 16), (600000, 150000, 18.0, 4, 1), (600000, 150000, 18.0, 5, 0),
    (600000, 150000, 23.0, 4, 0),
    (600000, 1 << 19, 4.0, 16, 16), (600000, (1 << 19) + 1, 4.0, 16, 1),
    (600000, (1 << 19) + 1, 4.0, 9, 1), (600000, (1 << 19) + 1, 2.2, 16, 4),
    (600000, (1 << 19) + 1, 7.0, 16, 0)])
def test_lines(ctx, n, nq, mean, k, want):
    pts = rtnn_amd.gen_uniform(n % 89 + k, n, 0.0, (n / mean) ** (1 / 3))
    ctx.set_points(pts)
    qs = pts[:nq]
    idx, d2, st = ctx.search(qs, mode="knn", radius=1.0, k=k)
    got = 0 if list(st.grid_dims) == PACKETS else st.lanes_per_query
    assert got == want
    ctx.set_options(queries_per_wave=64)
    wi, wd, _ = ctx.search(qs, mode="knn", radius=1.0, k=k)
    ctx.set_options()
    assert np.array_equal(idx, wi) and np.array_equal(d2, wd)
    sub = slice(0, 200)
    oi, od = oracle.grid_search(pts, qs[sub], oracle.MODE_KNN, 1.0, k)
    assert np.array_equal(idx[sub], oi) and np.array_equal(d2[sub], od)


def test_few_queries_crowded_cells(ctx):
    # a third of the points in few cells: what a query reads is far over the line
    rng = np.random.default_rng(8)
    pts = rng.uniform(0, 60, (300000, 3)).astype(np.float32)
    pts[::3] = rng.normal(30, 0.5, (100000, 3))
    ctx.set_points(pts)
    idx, d2, st = ctx.search(pts[:9000], mode="knn", radius=1.0, k=8)
    assert list(st.grid_dims) == PACKETS
    oi, od = oracle.grid_search(pts, pts[:200], oracle.MODE_KNN, 1.0, 8)
    assert np.array_equal(idx[:200], oi) and np.array_equal(d2[:200], od)
