"""Set-up of the points (copy, bounding box and the check for non-finite
coordinates in one launch): sizes around the kernel's four-point words and
blocks, views at every 4-byte offset from a 16-byte boundary, extreme and bad
points at either end.  Rows against the CPU oracle."""
import numpy as np
import pytest
import torch

import oracle
import rtnn_amd

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 3, 4, 5, 1023, 1024, 1025, 1031, 4099]


def _view(p, off):
    """p on the GPU, `off` floats after a 16-byte boundary."""
    buf = torch.full((p.size + 16,), float("nan"), device="cuda")
    v = buf[off:off + p.size].view(-1, 3)
    v.copy_(torch.from_numpy(p))
    torch.cuda.synchronize()
    assert v.data_ptr() % 16 == 4 * off
    return v


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("off", [0, 1, 2, 3])
def test_box_and_rows(ctx, n, off):
    rng = np.random.default_rng(n * 4 + off)
    p = rng.uniform(0.25, 0.75, (n, 3)).astype(np.float32)
    for low, high in ((0, n - 1), (n - 1, 0)):
        c = p.copy()
        c[low] = -0.25
        c[high] = (3.5, 5.5, 7.5) if n > 1 else -0.25
        ctx.set_points(_view(c, off))
        idx, d2, st = ctx.search(None, mode="radius", radius=1.0, k=12)
        assert list(st.grid_dims) == ([4, 6, 8] if n > 1 else [1, 1, 1])
        wi, wd = oracle.grid_search(c, c, oracle.MODE_RADIUS, 1.0, 12)
        assert np.array_equal(idx.cpu(), wi) and np.array_equal(d2.cpu(), wd)


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("off", [0, 1])
def test_non_finite_points_are_counted(ctx, n, off):
    rng = np.random.default_rng(n)
    p = rng.uniform(0, 1, (n, 3)).astype(np.float32)
    bad = sorted({0, n // 2, n - 1})
    for i, row in enumerate(bad):
        p[row, i % 3] = (np.nan, np.inf, -np.inf)[i]
    for src in (_view(p, off), p):
        with pytest.raises(rtnn_amd.RtnnError, match=f"{len(bad)} non-finite"):
            ctx.set_points(src)
    # the same buffers serve the next points
    q = rng.uniform(0, 1, (n, 3)).astype(np.float32)
    ctx.set_points(_view(q, off))
    idx, d2, _ = ctx.search(None, mode="radius", radius=0.3, k=8)
    wi, wd = oracle.grid_search(q, q, oracle.MODE_RADIUS, 0.3, 8)
    assert np.array_equal(idx.cpu(), wi) and np.array_equal(d2.cpu(), wd)


@pytest.mark.parametrize("large", [[], [70000, 9001]])
@pytest.mark.parametrize("shift", [0, 1, 2, 3])
def test_cloud_boxes(ctx, shift, large):
    # clouds that start and end at every remainder of four points, some empty;
    # with the large ones the average cloud takes the wide blocks
    sizes = [0, 1, 2, 3, 4, 5, 6, 7, 1030, 0, 257, 1021] + large
    off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.uint64)
    n = int(off[-1])
    rng = np.random.default_rng(shift)
    p = rng.uniform(0, 20 if large else 6, (n, 3)).astype(np.float32)
    idx, d2, _ = ctx.search_batched(_view(p, shift), off, mode="radius", radius=1.0, k=9)
    idx, d2 = idx.cpu().numpy(), d2.cpu().numpy()
    for a, b in zip(off[:-1].astype(int), off[1:].astype(int)):
        if a == b:
            continue
        wi, wd = oracle.grid_search(p[a:b], p[a:b], oracle.MODE_RADIUS, 1.0, 9)
        assert np.array_equal(idx[a:b], wi) and np.array_equal(d2[a:b], wd)
