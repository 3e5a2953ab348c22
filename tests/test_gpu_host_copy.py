"""Rows copied to the caller's host memory: around the size from which they
travel through the pinned ring, whole and partial chunks, slots used again,
without distances, and into pinned memory.  Equal to the rows on the device."""
import numpy as np
import pytest
import torch

import rtnn_amd

pytestmark = pytest.mark.gpu


def device_rows(ctx, pts, k):
    dev = torch.from_numpy(pts).cuda()
    torch.cuda.synchronize()
    idx, d2, _ = ctx.search(dev, mode="radius", radius=1.5, k=k)
    return idx.cpu().numpy(), d2.cpu().numpy()


# 8 * n * k bytes: 4 MiB and a row around it, 1 MiB chunks and partial ones, 4 MiB
# chunks and more of them than slots
@pytest.mark.parametrize("n,k", [(8191, 64), (8192, 64), (8193, 64), (9999, 129), (40001, 33),
                                 (130000, 50)])
def test_rows_equal(ctx, n, k):
    pts = rtnn_amd.gen_uniform(n, n, 0.0, float((n / 2) ** (1 / 3)))
    ctx.set_points(pts)
    wi, wd = device_rows(ctx, pts, k)
    for _ in range(2):
        out = (np.full((n, k), 7, np.int32), np.full((n, k), 7, np.float32))
        ctx.search(pts, mode="radius", radius=1.5, k=k, out=out)
        assert np.array_equal(out[0], wi) and np.array_equal(out[1], wd)
    pin = (torch.empty((n, k), dtype=torch.int32, pin_memory=True),
           torch.empty((n, k), dtype=torch.float32, pin_memory=True))
    out = tuple(t.numpy() for t in pin)
    ctx.search(pts, mode="radius", radius=1.5, k=k, out=out)
    assert np.array_equal(out[0], wi) and np.array_equal(out[1], wd)
    # one array, not on a page's or a word's boundary of the chunks
    raw = np.zeros(n * k + 3, np.int32)
    idx = raw[3:].reshape(n, k)
    ctx.search(pts, mode="radius", radius=1.5, k=k, with_d2=False, out=(idx, None))
    assert np.array_equal(idx, wi) and not raw[:3].any()


def test_partitioned_rows_equal(ctx):
    pts = rtnn_amd.gen_uniform(3, 60000, 0.0, 30.0)
    ctx.set_points(pts)
    dev = torch.from_numpy(pts).cuda()
    torch.cuda.synchronize()
    wi, wd, _ = ctx.search_partitioned(dev, radius=1.5, k=20)
    idx, d2, _ = ctx.search_partitioned(pts, radius=1.5, k=20)
    assert np.array_equal(idx, wi.cpu().numpy()) and np.array_equal(d2, wd.cpu().numpy())
