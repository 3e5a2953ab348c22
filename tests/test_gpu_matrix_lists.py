"""The matrix-core kernel where its lists of candidates fill: 15 tiles of 32 points
(480) for rows of up to 16 keys, 24 (768) beyond.  Clouds that one radius covers
list every point of theirs; the rows are the oracle's."""
import numpy as np
import pytest
import torch

import oracle
import rtnn_amd

pytestmark = pytest.mark.gpu

SIZES = [447, 448, 449, 479, 480, 481, 511, 512, 513, 735, 736, 737, 767, 768, 769, 959, 960,
         961, 1439, 1440, 1441, 1535, 1536, 1537]


@pytest.mark.parametrize("k", [1, 16, 17, 32])
@pytest.mark.parametrize("mode", ["radius", "knn"])
@pytest.mark.parametrize("near_last", [False, True])
def test_full_lists(ctx, k, mode, near_last):
    # near_last: the row's points are the last that the list takes in
    rng = np.random.default_rng(k)
    offs = np.concatenate([[0], np.cumsum(SIZES)]).astype(np.uint64)
    xyz = rng.uniform(0, 1, (int(offs[-1]), 3)).astype(np.float32)
    if near_last:
        for a, b in zip(offs[:-1].astype(int), offs[1:].astype(int)):
            xyz[a:b] = xyz[a:b][np.argsort(xyz[a:b, 2], kind="stable")]
            xyz[b - 2:b, 2] = 1.0
    dev = torch.from_numpy(xyz).cuda()
    torch.cuda.synchronize()
    ctx.set_options()
    idx, d2, _ = ctx.search_batched(dev, offs, mode=mode, radius=2.0, k=k)
    idx, d2 = idx.cpu().numpy(), d2.cpu().numpy()
    om = oracle.MODE_RADIUS if mode == "radius" else oracle.MODE_KNN
    for a, b in zip(offs[:-1].astype(int), offs[1:].astype(int)):
        wi, wd = oracle.bruteforce(xyz[a:b], xyz[a:b], om, 2.0, k)
        assert np.array_equal(idx[a:b], wi) and np.array_equal(d2[a:b], wd)
