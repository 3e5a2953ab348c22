"""lanes_per_query of the statistics names the kernel that ran: 1 for the matrix
kernel (a query per lane) where groups of lanes were asked for, 16 for long KNN rows
of a batch, the lanes asked for otherwise."""
import numpy as np
import pytest
import torch

import rtnn_amd

pytestmark = pytest.mark.gpu

MANY = 1 << 19  # queries from which a single cloud takes the matrix kernel


@pytest.mark.parametrize("mode,k,qpw,want", [
    ("radius", 32, 0, 1), ("radius", 33, 0, 16), ("radius", 32, 16, 4), ("radius", 32, 4, 1),
    ("knn", 32, 0, 1), ("knn", 33, 0, 16), ("knn", 33, 64, 16), ("knn", 16, 16, 4)])
def test_batches(ctx, mode, k, qpw, want):
    offs = np.array([0, 700, 1500], np.uint64)
    xyz = torch.rand(1500, 3, generator=torch.Generator().manual_seed(1)).cuda()
    torch.cuda.synchronize()
    ctx.set_options(queries_per_wave=qpw)
    try:
        assert ctx.search_batched(xyz, offs, mode=mode, radius=0.2, k=k)[2].lanes_per_query == want
    finally:
        ctx.set_options()


@pytest.mark.parametrize("n,want", [(MANY, 1), (MANY - 1, 16)])
def test_points_as_queries(ctx, n, want):
    ctx.set_points(np.random.default_rng(n).uniform(0, 80, (n, 3)).astype(np.float32))
    assert ctx.search(None, mode="radius", radius=1.0, k=8)[2].lanes_per_query == want
