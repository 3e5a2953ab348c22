"""The scratch of rtnn_search_noalloc: every piece holds what its kernels write
(the sorts of points and queries share one workspace, whose size is not monotone
in the number of pairs), and sizes around the sort's change of tiles give the rows
of rtnn_search."""
import ctypes

import numpy as np
import pytest

import rtnn_amd

SCRATCH = 128 << 20
MIN_CELLS = 1 << 16
LINE = 1 << 19  # pairs up to which the radix sort takes its small tiles
NAMES = ("status offs bb grid keys vals spts tmp qkeys qvals qs ovf cells").split()


class Layout(ctypes.Structure):
    _fields_ = [(n, ctypes.c_uint64) for n in NAMES]


def layout(n, nq, own_q, pooled):
    f = getattr(rtnn_amd.lib(), "_ZN4rtnn14noalloc_layoutEmmbb")
    f.restype = Layout
    f.argtypes = [ctypes.c_uint64, ctypes.c_uint64, ctypes.c_bool, ctypes.c_bool]
    return f(n, nq, own_q, pooled)


def radix_words(n):
    f = getattr(rtnn_amd.lib(), "_ZN4rtnn15radix_tmp_wordsEm")
    f.restype = ctypes.c_uint64
    f.argtypes = [ctypes.c_uint64]
    return f(n)


def cell_words(n):
    f = getattr(rtnn_amd.lib(), "_ZN4rtnn21cell_bounds_tmp_wordsEm")
    f.restype = ctypes.c_uint64
    f.argtypes = [ctypes.c_uint64]
    return f(n)


@pytest.mark.parametrize("pooled", [False, True])
@pytest.mark.parametrize("own_q", [False, True])
def test_pieces_hold_what_is_written(own_q, pooled):
    sizes = [1, 63, 1000, 4096, 150_000, LINE - 1024, LINE - 1, LINE, LINE + 1, 520_000, 530_000,
             550_000, 571_000, 600_000, 1_000_000, 2_000_000]
    cells = [1, 1 << 8, 1 << 16, 1 << 20, 1 << 21, (1 << 22) + 1, 1 << 24, SCRATCH // 4]
    for n in sizes:
        for nq in sizes if own_q else [n]:
            l = layout(n, nq, own_q, pooled)
            need = {"status": 16, "offs": 16, "bb": 24, "grid": 48, "keys": 4 * n, "vals": 4 * n,
                    "spts": 16 * n + 4096,
                    "tmp": 4 * max(radix_words(n), radix_words(nq) if own_q else 0,
                                   8 * 1024,  # the box reduction's partial boxes
                                   max(cell_words(c) for c in cells))}
            if own_q:
                need.update(qkeys=4 * nq, qvals=4 * nq, qs=16 * nq)
            if pooled:
                need["ovf"] = 4 * (nq + 64)
            used = [x for x in NAMES if x in need] + ["cells"]
            for a, b in zip(used, used[1:]):
                assert getattr(l, a) % 256 == 0
                assert getattr(l, a) + need[a] <= getattr(l, b), (n, nq, a)


@pytest.mark.parametrize("n,nq", [(3_306_736, 0), (2_076_336, 2_076_336)])
def test_largest_inputs_fit(n, nq):
    assert layout(n, nq, nq > 0, False).cells + 4 * (MIN_CELLS + 1) <= SCRATCH


@pytest.mark.gpu
@pytest.mark.parametrize("n,nq", [(530_000, 520_000), (LINE + 1, LINE), (LINE, LINE + 1)])
def test_rows_around_the_change_of_tiles(n, nq):
    import torch
    g = torch.Generator(device="cuda").manual_seed(n + nq)
    side = (n / 0.8) ** (1 / 3)
    p = torch.rand(n, 3, generator=g, device="cuda") * side
    q = torch.rand(nq, 3, generator=g, device="cuda") * side
    with rtnn_amd.Context(0) as ctx:
        for mode in ("radius", "knn"):
            d2 = torch.empty((nq, 8), dtype=torch.float32, device="cuda")
            torch.cuda.synchronize()  # the context works on a stream of its own
            idx, d2 = ctx.search_noalloc(p, q, mode=mode, radius=1.2, k=8, d2=d2)
            ctx.set_points(p)
            wi, wd, _ = ctx.search(q, mode=mode, radius=1.2, k=8)
            assert torch.equal(idx, wi) and torch.equal(d2, wd)
