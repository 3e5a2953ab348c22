"""The packet walk of the plain KNN (packet.hip) against the CPU oracle at the
edges of its tree (leaves of 8 points, nodes of 64 leaves, 64-query packets)
and list sizes, and against the group kernel on what its dispatch accepts."""
import numpy as np
import pytest

import oracle
import rtnn_amd

pytestmark = pytest.mark.gpu


def check(ctx, pts, qs, r, k):
    ctx.set_options(queries_per_wave=64)  # sparse points would go by their cells
    idx, d2, st = ctx.search(qs, mode="knn", radius=r, k=k)
    ctx.set_options()
    assert st.lanes_per_query == 1
    wi, wd = oracle.grid_search(pts, pts if qs is None else qs, oracle.MODE_KNN, r, k)
    assert np.array_equal(idx, wi) and np.array_equal(d2, wd)


@pytest.mark.parametrize("n", [1, 7, 8, 9, 63, 65, 511, 512, 513, 32767, 32769, 40000])
@pytest.mark.parametrize("k", [1, 8, 9, 33])
def test_tree_edges(ctx, n, k):
    rng = np.random.default_rng(n * 100 + k)
    pts = rng.uniform(-3, 7, (n, 3)).astype(np.float32)
    qs = rng.uniform(-5, 9, (n % 130 + 3, 3)).astype(np.float32)
    ctx.set_points(pts)
    check(ctx, pts, qs, 2.5, k)
    check(ctx, pts, None, 1.0, k)


@pytest.mark.parametrize("k", [2, 4, 5, 7, 16, 17, 31, 32, 50, 63, 64])
def test_list_sizes_and_uneven_points(ctx, k):
    # clusters, exact duplicates (more than a leaf of them), one far point that
    # flattens the key grid, queries far outside, NaN and infinite
    rng = np.random.default_rng(k)
    pts = np.concatenate([rng.normal(0, 0.5, (6000, 3)), rng.uniform(-50, 50, (3000, 3)),
                          np.repeat(rng.normal(0, 0.5, (20, 3)), 30, axis=0),
                          [[4000.0, 0, 0]]]).astype(np.float32)
    qs = np.concatenate([rng.normal(0, 1, (700, 3)), rng.uniform(-60, 60, (700, 3)), pts[-40:],
                         [[np.nan, 0, 0], [np.inf, 0, 0], [0, -np.inf, 0], [1e30, 0, 0]]])
    qs = qs.astype(np.float32)
    ctx.set_points(pts)
    for r in (0.3, 8.0):
        idx, d2, _ = ctx.search(qs, mode="knn", radius=r, k=k)
        wi, wd = oracle.bruteforce(pts, qs, oracle.MODE_KNN, r, k)
        assert np.array_equal(idx, wi) and np.array_equal(d2, wd)


def test_lattice_ties_and_flat_boxes(ctx):
    # every distance tied many times; then all points in a plane, on a line and
    # in one place
    g = np.arange(24, dtype=np.float32)
    pts = np.stack(np.meshgrid(g, g, g), -1).reshape(-1, 3)
    ctx.set_points(pts)
    check(ctx, pts, None, 3.0, 20)
    rng = np.random.default_rng(1)
    for keep in ((0, 1), (2,), ()):
        p = np.full((3000, 3), 0.25, np.float32)
        for a in keep:
            p[:, a] = rng.uniform(0, 5, 3000)
        ctx.set_points(p)
        check(ctx, p, None, 0.5, 12)


@pytest.mark.parametrize("order", [0, 1, 2])
def test_equals_the_group_kernel(ctx, order):
    # query_order = 1 keeps the cell walk (queries in input order)
    pts = rtnn_amd.gen_gaussian_mixture(2, 20, 60000)
    qs = rtnn_amd.gen_gaussian_mixture(2, 21, 20011)
    ctx.set_points(pts)
    try:
        for k in (6, 16, 48):
            ctx.set_options(queries_per_wave=16)
            want = ctx.search(qs, mode="knn", radius=20.0, k=k)
            for qpw in (0, 64):
                ctx.set_options(queries_per_wave=qpw, query_order=order)
                got = ctx.search(qs, mode="knn", radius=20.0, k=k)
                assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
    finally:
        ctx.set_options()
