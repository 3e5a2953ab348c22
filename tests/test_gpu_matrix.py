"""The matrix-core kernel (range search of many queries or of batches, k <= 32; KNN
at proposed radii): rows equal to the group kernel's and to the CPU oracle at the
edges of its tiles (64 queries, 32 and 768 points, 16 keys)."""
import numpy as np
import pytest
import torch

import oracle
import rtnn_amd

pytestmark = pytest.mark.gpu

MANY = 1 << 19  # queries from which single clouds take it


def equal_to_groups(ctx, qs, r, k, sample, pts):
    ctx.set_options()
    idx, d2, _ = ctx.search(qs, mode="radius", radius=r, k=k)
    ctx.set_options(queries_per_wave=16)  # four lanes per query
    wi, wd, _ = ctx.search(qs, mode="radius", radius=r, k=k)
    ctx.set_options()
    assert np.array_equal(idx, wi) and np.array_equal(d2, wd)
    q = (pts if qs is None else qs)[sample]
    oi, od = oracle.grid_search(pts, q, oracle.MODE_RADIUS, r, k)
    assert np.array_equal(idx[sample], oi) and np.array_equal(d2[sample], od)


@pytest.mark.parametrize("k", [1, 15, 16, 17, 32])
def test_points_as_queries(ctx, k):
    rng = np.random.default_rng(k)
    # even points, hot cells (several lists of points, rows far beyond 32 hits),
    # duplicates, a far offset
    pts = np.concatenate([rng.uniform(0, 100, (MANY - 4000, 3)), rng.normal(50, 0.3, (3000, 3)),
                          np.repeat(rng.uniform(0, 100, (50, 3)), 21, axis=0)])
    pts = (pts + 1000.0).astype(np.float32)
    ctx.set_points(pts)
    sample = np.concatenate([np.arange(0, len(pts), 997), np.arange(MANY - 4000, MANY - 3900)])
    equal_to_groups(ctx, None, 1.0, k, sample, pts)
    equal_to_groups(ctx, None, 2.3, k, sample[::4], pts)


@pytest.mark.parametrize("n", [1, 31, 33, 5000, 2 * MANY + 1])
def test_other_queries(ctx, n):
    # far, infinite and NaN queries among them; n = 2 MANY + 1 is the densest
    # point set half as many queries take the kernel for
    rng = np.random.default_rng(n)
    pts = rng.uniform(0, 60, (n, 3)).astype(np.float32)
    qs = rng.uniform(-3, 63, (MANY, 3)).astype(np.float32)
    qs[:3] = [[1e30, 0, 0], [np.inf, 1, 1], [np.nan, 2, 2]]
    ctx.set_points(pts)
    r = 2.0 if n > 100 else 20.0
    equal_to_groups(ctx, qs, r, 24, np.arange(3, MANY, 1499), pts)


@pytest.mark.parametrize("k", [1, 16, 32])
@pytest.mark.parametrize("scale,r", [(1.0, 0.2), (1.0, 5.0), (1e15, 2e14), (1e18, 5e18),
                                     (1e-18, 2e-19)])
def test_batches(ctx, k, scale, r):
    # sizes at the edges of waves, blocks and lists; radii from a few hits to whole
    # clouds; squares near overflow and underflow
    rng = np.random.default_rng(7)
    sizes = [1, 2, 31, 32, 33, 63, 64, 65, 255, 256, 257, 511, 769, 1500]
    offs = np.concatenate([[0], np.cumsum(sizes)]).astype(np.uint64)
    xyz = (rng.uniform(0, 1, (int(offs[-1]), 3)) * scale).astype(np.float32)
    dev = torch.from_numpy(xyz).cuda()
    torch.cuda.synchronize()
    ctx.set_options()
    idx, d2, _ = ctx.search_batched(dev, offs, radius=r, k=k)
    idx, d2 = idx.cpu().numpy(), d2.cpu().numpy()
    for a, b in zip(offs[:-1].astype(int), offs[1:].astype(int)):
        wi, wd = oracle.bruteforce(xyz[a:b], xyz[a:b], oracle.MODE_RADIUS, r, k)
        assert np.array_equal(idx[a:b], wi) and np.array_equal(d2[a:b], wd)


@pytest.mark.parametrize("k", [1, 5, 16])
def test_knn_at_proposed_radii(ctx, k):
    rng = np.random.default_rng(k + 40)
    n = MANY + 77
    v = rng.normal(size=(n, 3))
    pts = (rng.integers(0, 40, (n, 1)) * 25.0 +
           20.0 * v / np.linalg.norm(v, axis=1, keepdims=True)).astype(np.float32)
    ctx.set_points(pts)
    ctx.mlp_train(4.0, k, n_samples=20000, steps=40, batch=1000, seed=1)
    want = ctx.search(pts, mode="knn", radius=4.0, k=k)
    ctx.set_options(cell_factor=2.0, queries_per_wave=32, grid_levels=1, group_buffer=2)
    got = ctx.search_learned(pts, radius=4.0, k=k)
    ctx.set_options()
    assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])


@pytest.mark.parametrize("k", [1, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("r", [0.2, 0.5, 5.0])
def test_knn_batches(ctx, k, r):
    rng = np.random.default_rng(9)
    sizes = [1, 2, 31, 33, 64, 65, 255, 257, 769, 1500]
    offs = np.concatenate([[0], np.cumsum(sizes)]).astype(np.uint64)
    xyz = rng.uniform(0, 1, (int(offs[-1]), 3)).astype(np.float32)
    xyz[-40:] = xyz[-1]  # duplicates are no neighbours of each other
    dev = torch.from_numpy(xyz).cuda()
    torch.cuda.synchronize()
    ctx.set_options()
    idx, d2, _ = ctx.search_batched(dev, offs, mode="knn", radius=r, k=k)
    idx, d2 = idx.cpu().numpy(), d2.cpu().numpy()
    for a, b in zip(offs[:-1].astype(int), offs[1:].astype(int)):
        wi, wd = oracle.bruteforce(xyz[a:b], xyz[a:b], oracle.MODE_KNN, r, k)
        assert np.array_equal(idx[a:b], wi) and np.array_equal(d2[a:b], wd)
