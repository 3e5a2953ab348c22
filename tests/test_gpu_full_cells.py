"""Raster grids whose cells are full keep the input order inside a cell (sorted, not
counted) where one lane takes a query or few lanes a batch's; rows are the oracle's
either way, and sort_passes tells which build it was."""
import numpy as np
import pytest
import torch

import oracle
import rtnn_amd

pytestmark = pytest.mark.gpu


def lattice(side, h=0.1):
    i = np.arange(side, dtype=np.float32) * np.float32(h)
    z, y, x = np.meshgrid(i, i, i, indexing="ij")
    return np.ascontiguousarray(np.stack([x, y, z], -1).reshape(-1, 3))


def rows_equal(pts, idx, d2, mode, r, k):
    m = oracle.MODE_KNN if mode == "knn" else oracle.MODE_RADIUS
    wi, wd = oracle.grid_search(pts, pts[::7], m, r, k)
    assert np.array_equal(idx[::7], wi) and np.array_equal(d2[::7], wd)


# a 21^3 lattice: 9.3 points a cell of edge 0.22, 3.4 of edge 0.15
@pytest.mark.parametrize("qpw,r,counted", [(64, 0.22, False), (64, 0.15, True), (0, 0.22, True),
                                           (16, 0.3, True)])
def test_range(ctx, qpw, r, counted):
    pts = lattice(21)
    ctx.set_points(pts)
    ctx.set_options(queries_per_wave=qpw)
    try:
        idx, d2, st = ctx.search(None, mode="radius", radius=r, k=20)
    finally:
        ctx.set_options()
    rows_equal(pts, idx, d2, "radius", r, 20)
    assert (st.sort_passes == 0) == counted


@pytest.mark.parametrize("qpw,r,counted", [(0, 0.44, False), (0, 0.3, True), (32, 0.44, True)])
def test_partitioned(ctx, qpw, r, counted):
    pts = lattice(21)
    ctx.set_points(pts)
    ctx.set_options(queries_per_wave=qpw, grid_levels=1, cell_factor=2.0)
    try:
        idx, d2, st = ctx.search_partitioned(pts, radius=r, k=9)
    finally:
        ctx.set_options()
    rows_equal(pts, idx, d2, "knn", r, 9)
    assert (st.sort_passes == 0) == counted


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("mode,qpw,r,counted", [
    ("radius", 64, 0.22, False), ("radius", 64, 0.15, True), ("radius", 0, 0.6, True),
    ("radius", 16, 0.6, False), ("knn", 16, 0.3, True), ("knn", 0, 0.6, True)])
def test_batches(ctx, mode, qpw, r, counted, graph):
    sides = [21, 12, 21]
    clouds = [lattice(s) for s in sides]
    offs = np.concatenate([[0], np.cumsum([len(c) for c in clouds])]).astype(np.uint64)
    dev = torch.from_numpy(np.concatenate(clouds)).cuda()
    torch.cuda.synchronize()
    ctx.set_options(queries_per_wave=qpw)
    try:
        if graph:
            g = ctx.graph_batched(dev, offs, mode=mode, radius=r, k=12)
            for _ in range(3):
                g.launch()
            idx, d2 = g.idx.cpu().numpy(), g.d2.cpu().numpy()
            g.close()
        else:
            idx, d2, st = ctx.search_batched(dev, offs, mode=mode, radius=r, k=12)
            idx, d2 = idx.cpu().numpy(), d2.cpu().numpy()
            assert (st.sort_passes == 0) == counted
    finally:
        ctx.set_options()
    for a, b, c in zip(offs[:-1].astype(int), offs[1:].astype(int), clouds):
        rows_equal(c, idx[a:b], d2[a:b], mode, r, 12)
