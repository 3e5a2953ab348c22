"""Stream-ordered KNN: by cells or packets as the points lie, measured once per points
and radius; rows equal the synchronous search's after new points, other radii and
other cell budgets, with earlier work still in flight."""
import numpy as np
import pytest

import rtnn_amd

pytestmark = pytest.mark.gpu


def sets(n):
    rng = np.random.default_rng(n)
    even = rng.uniform(0, (n / 0.8) ** (1 / 3), (n, 3))
    return [even, even[:1] + rng.normal(0, 3.0, (n, 3)), np.repeat(even[: n // 8 + 1], 8, axis=0),
            even * [1, 1, 40.0]]


@pytest.mark.parametrize("n", [1, 300, 20000, 140000, 600000])
def test_rows(n):
    import torch
    s = torch.cuda.Stream()
    with rtnn_amd.Context(0) as ctx:
        for pts in sets(n):
            pts = np.ascontiguousarray(pts, np.float32)
            ctx.set_points(pts)
            got = []
            for r, k, cells in ((1.2, 16, 0), (2.0, 4, 0), (1.2, 64, 0), (1.2, 16, 4096)):
                q = torch.from_numpy(pts[::3].copy()).cuda()
                out = (torch.empty((len(q), k), dtype=torch.int32, device="cuda"),
                       torch.empty((len(q), k), dtype=torch.float32, device="cuda"))
                torch.cuda.synchronize()
                ctx.set_options(max_cells=cells)
                ctx.search_async(q, out[0], out[1], mode="knn", radius=r, stream=s)
                got.append((q, r, k, out))
            s.synchronize()
            ctx.set_options(queries_per_wave=4)
            for q, r, k, out in got:
                wi, wd, _ = ctx.search(q, mode="knn", radius=r, k=k)
                assert torch.equal(out[0], wi) and torch.equal(out[1], wd)
            ctx.set_options()
