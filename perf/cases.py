"""The work a program gives the neighbor search, for timing.

A case is a dict of plain values; `prepare` makes what the program holds before
the call (points, queries, a context with its points or weights, a captured
graph), `run` is one pass through the public entry points and returns its rows.
`listed` are the sizes the repository itself works at (its benchmark's five
workloads, its CLI and tests), `draw` gives others of the same ranges.

Point distributions (all seeded, made on the GPU):
  uniform   a box at a fixed density (0.8 points per unit volume)
  spheres   surfaces of spheres, as scanned objects (radii 5..50, noise 0.05)
  mixture   Gaussian clusters over a uniform background
  levy      a Levy flight (very clustered) with uniform queries
  lattice   jittered cubic lattices, one per cloud (particle blocks)
"""
import math
import random

import numpy as np
import torch

import rtnn_amd

DEV = "cuda"


def listed():
    return [
        # One small frame, e.g. a particle system of a demo or one LiDAR ring:
        # new points every call, so latency and launches are what counts.
        {"name": "range_tiny", "kind": "frame", "dist": "uniform", "n": 1500, "r": 2.0, "k": 50,
         "mode": "radius"},
        # A simulation step: 100,000 particles move, every particle asks for
        # its neighbors (the reference's samepq use).
        {"name": "range_100k", "kind": "frame", "dist": "uniform", "n": 100_000, "r": 2.0,
         "k": 50, "mode": "radius"},
        # Feature extraction on a scan: a fixed cloud, separate key points.
        {"name": "range_scan", "kind": "query", "dist": "spheres", "n": 1_234_567, "nq": 300_001,
         "r": 5.0, "k": 32, "mode": "radius"},
        # The command line's path: host arrays in, host rows out, many neighbors.
        {"name": "range_host", "kind": "host", "dist": "uniform", "n": 60_000, "r": 3.0, "k": 128,
         "mode": "radius"},
        # Plain KNN with a wide radius over clustered points.
        {"name": "knn_clusters", "kind": "query", "dist": "mixture", "n": 1_000_000,
         "nq": 1_000_000, "r": 20.0, "k": 8, "mode": "knn"},
        # The same with the density partition.
        {"name": "knn_clusters_part", "kind": "partitioned", "dist": "mixture", "n": 1_000_000,
         "nq": 1_000_000, "r": 20.0, "k": 8, "mode": "knn"},
        # Plain KNN on scanned surfaces.
        {"name": "knn_surface", "kind": "query", "dist": "spheres", "n": 4_000_000,
         "nq": 4_000_000, "r": 10.0, "k": 16, "mode": "knn"},
        # The benchmark's headline: learned radius, the options its tuner keeps.
        {"name": "knn_learned", "kind": "learned", "dist": "spheres", "n": 10_000_000,
         "nq": 10_000_000, "r": 10.0, "k": 16, "mode": "knn"},
        # Extremely uneven points and queries in mostly empty space.
        {"name": "knn_levy", "kind": "levy", "dist": "levy", "n": 2_000_000, "nq": 2_000_000,
         "r": 100.0, "k": 32, "mode": "knn"},
        # A data set of clouds in one launch (a quarter of the benchmark's).
        {"name": "batched_1024", "kind": "batched", "dist": "lattice", "clouds": 1024,
         "nmin": 1000, "nmax": 200_000, "r": 0.2, "k": 64, "mode": "radius"},
        # A training loop's mini-batch of small clouds, replayed from a graph.
        {"name": "graph_small", "kind": "graph", "dist": "lattice", "clouds": 48, "nmin": 500,
         "nmax": 8000, "r": 0.2, "k": 32, "mode": "radius"},
        # Training of the radius proposal on a new point set (forward and
        # backward of its network).
        {"name": "mlp_train", "kind": "train", "dist": "spheres", "n": 1_000_000, "r": 10.0,
         "k": 16, "samples": 262_144, "steps": 200, "batch": 4096, "mode": "knn"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["frame", "frame", "query", "query", "host", "partitioned", "learned",
                       "levy", "batched", "graph", "train"])
    c = {"kind": kind}
    if kind in ("frame", "host"):
        mode = rng.choice(["radius", "radius", "knn"])
        hi = 1_500_000 if kind == "frame" else 100_000
        c.update(dist="uniform", n=_log(rng, 300, hi), r=round(rng.uniform(1.2, 2.4), 3),
                 k=_log(rng, 4, 64) if mode == "knn" else _log(rng, 8, 160), mode=mode)
    elif kind == "query":
        dist = rng.choice(["spheres", "mixture", "uniform"])
        mode = rng.choice(["radius", "knn", "knn"])
        n = _log(rng, 20_000, 3_000_000)
        c.update(dist=dist, n=n, nq=_log(rng, 1000, 3_000_000),
                 r={"spheres": round(rng.uniform(4.0, 10.0), 2),
                    "mixture": round(rng.uniform(5.0, 20.0), 2) if n <= 1_000_000 else 5.0,
                    "uniform": round(rng.uniform(1.2, 2.4), 2)}[dist],
                 k=_log(rng, 4, 64), mode=mode)
        if dist == "mixture":  # a query's sphere covers a whole cluster
            c.update(nq=min(c["nq"], 1_000_000), k=min(c["k"], 16))
    elif kind == "partitioned":
        c.update(dist=rng.choice(["spheres", "mixture"]), n=_log(rng, 50_000, 3_000_000),
                 nq=_log(rng, 10_000, 3_000_000), r=10.0, k=_log(rng, 4, 40), mode="knn")
    elif kind == "learned":
        c.update(dist="spheres", n=_log(rng, 200_000, 8_000_000),
                 nq=_log(rng, 100_000, 8_000_000), r=10.0, k=rng.randint(4, 16), mode="knn")
    elif kind == "levy":
        c.update(dist="levy", n=_log(rng, 100_000, 2_000_000), nq=_log(rng, 100_000, 1_500_000),
                 r=100.0, k=rng.randint(8, 32), mode="knn")
    elif kind == "batched":
        c.update(dist="lattice", clouds=_log(rng, 16, 900), nmin=1000, nmax=200_000, r=0.2,
                 k=rng.randint(24, 64), mode=rng.choice(["radius", "radius", "knn"]))
    elif kind == "graph":
        c.update(dist="lattice", clouds=_log(rng, 1, 200), nmin=500, nmax=8000, r=0.2,
                 k=rng.randint(16, 48), mode=rng.choice(["radius", "knn"]))
    else:
        c.update(dist="spheres", n=_log(rng, 100_000, 2_000_000), r=10.0, k=rng.randint(4, 32),
                 samples=_log(rng, 30_000, 500_000), steps=rng.randint(50, 250),
                 batch=rng.choice([1000, 2048, 4096, 6000]), mode="knn")
    return c


# ------------------------------------------------------------------ inputs

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _sizes(case):
    """Cloud offsets of a batch: part of the case, the same for every seed."""
    g = random.Random(case["clouds"])
    a, b = math.log(case["nmin"]), math.log(case["nmax"])
    s = [int(round(math.exp(g.uniform(a, b)))) for _ in range(case["clouds"])]
    return np.concatenate([[0], np.cumsum(s)]).astype(np.uint64)


def _unit(g, n):
    v = torch.randn(n, 3, generator=g, device=DEV)
    return v / v.norm(dim=1, keepdim=True).clamp_min(1e-20)


def _uniform(case, g, n):
    side = (case["n"] / 0.8) ** (1 / 3)
    return torch.rand(n, 3, generator=g, device=DEV) * side


def _spheres(case, dist, g, n):
    """Points on sphere surfaces; the spheres come from `dist`, the sample from g."""
    ns = max(8, case["n"] // 5000)
    box = 2000.0 * (ns / 2000) ** (1 / 3)
    c = torch.rand(ns, 3, generator=dist, device=DEV) * box
    rad = 5.0 + 45.0 * torch.rand(ns, generator=dist, device=DEV)
    cum = torch.cumsum((rad * rad).double(), 0)
    u = torch.rand(n, generator=g, device=DEV, dtype=torch.float64) * cum[-1]
    s = torch.searchsorted(cum, u).clamp_max(ns - 1)
    rr = rad[s] + 0.05 * torch.randn(n, generator=g, device=DEV)
    return c[s] + rr[:, None] * _unit(g, n)


def _mixture(case, dist, g, n):
    ncomp = max(4, case["n"] // 15625)
    box = 1000.0 * (ncomp / 64) ** (1 / 3)
    c = torch.rand(ncomp, 3, generator=dist, device=DEV) * box
    s = torch.randint(ncomp, (n,), generator=g, device=DEV)
    p = c[s] + 5.0 * torch.randn(n, 3, generator=g, device=DEV)
    bg = torch.rand(n, generator=g, device=DEV) < 0.2
    return torch.where(bg[:, None], torch.rand(n, 3, generator=g, device=DEV) * box, p)


def _levy(g, n, box=1000.0):
    u = 1.0 - torch.rand(n, generator=g, device=DEV, dtype=torch.float64)
    step = 0.01 * u.clamp_min(1e-15) ** (-1 / 1.5)
    p = torch.cumsum(step[:, None] * _unit(g, n).double(), 0) + box / 2
    return torch.remainder(p, box).float()


def _lattice(offs, g):
    h, jit = 0.1, 0.02
    cnt = torch.from_numpy(np.diff(offs.astype(np.int64))).to(DEV)
    base = torch.from_numpy(offs[:-1].astype(np.int64)).to(DEV)
    n = int(offs[-1])
    cloud = torch.repeat_interleave(torch.arange(len(cnt), device=DEV), cnt)
    i = torch.arange(n, device=DEV) - base[cloud]
    side = torch.ceil(cnt.double() ** (1 / 3) - 1e-9).long()[cloud]
    ijk = torch.stack([i % side, (i // side) % side, i // (side * side)], 1).float()
    return h * (ijk + jit * (2 * torch.rand(n, 3, generator=g, device=DEV) - 1))


def _points(case, seed):
    """(points, queries or None), device float32."""
    d = case["dist"]
    gp, gq, gd = _gen(3 * seed), _gen(3 * seed + 1), _gen(3 * seed + 2)
    if d == "uniform":
        p = _uniform(case, gp, case["n"])
        return p, (_uniform(case, gq, case["nq"]) if "nq" in case else None)
    if d == "levy":
        return _levy(gp, case["n"]), torch.rand(case["nq"], 3, generator=gq, device=DEV) * 1000.0
    make = _spheres if d == "spheres" else _mixture
    p = make(case, gd, gp, case["n"])
    q = make(case, _gen(3 * seed + 2), gq, case["nq"]) if "nq" in case else None
    return p, q


# The options a tuned program keeps for the headline workload, the Levy flight
# and the batches (what the benchmark uses); everything else runs the defaults.
LEARNED = {"cell_factor": 2.0, "queries_per_wave": 32, "grid_levels": 1, "group_buffer": 2}
LEVY = {"grid_levels": 6, "tree_leaf": 65536, "tree_lanes": 2}
BATCHED = {"cell_factor": 1.0, "queries_per_wave": 16, "group_buffer": 1}


def _rows(nq, k):
    return (torch.empty((nq, k), dtype=torch.int32, device=DEV),
            torch.empty((nq, k), dtype=torch.float32, device=DEV))


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case, "ctx": rtnn_amd.Context(0)}
    ctx = s["ctx"]
    if kind in ("batched", "graph"):
        s["offs"] = _sizes(case)
        s["xyz"] = _lattice(s["offs"], _gen(seed))
        torch.cuda.synchronize()  # the context works on a stream of its own
        if kind == "batched":
            ctx.set_options(**BATCHED)
        else:
            s["graph"] = ctx.graph_batched(s["xyz"], s["offs"], mode=case["mode"],
                                           radius=case["r"], k=case["k"])
        return s
    s["p"], s["q"] = _points(case, seed)
    torch.cuda.synchronize()
    if kind == "host":
        s["p"] = s["p"].cpu().numpy()
        s["out"] = (np.zeros((case["n"], case["k"]), np.int32),
                    np.zeros((case["n"], case["k"]), np.float32))
        return s
    if kind == "frame":
        s["out"] = _rows(case["n"], case["k"])
        return s
    ctx.set_points(s["p"])
    if kind == "train":
        return s
    s["out"] = _rows(case["nq"], case["k"])
    if kind == "learned":
        ctx.mlp_train(case["r"], case["k"], n_samples=1 << 18, steps=300, batch=4096, seed=1)
        ctx.set_options(**LEARNED)
    elif kind == "levy":
        ctx.set_options(**LEVY)
    return s


def run(s):
    c, ctx = s["case"], s["ctx"]
    kind, r, k = c["kind"], c["r"], c["k"]
    if kind in ("frame", "host"):  # new points, every point a query
        ctx.set_points(s["p"])
        idx, d2, _ = ctx.search(None, mode=c["mode"], radius=r, k=k, out=s["out"])
    elif kind == "query":
        idx, d2, _ = ctx.search(s["q"], mode=c["mode"], radius=r, k=k, out=s["out"])
    elif kind in ("partitioned", "levy"):
        idx, d2, _ = ctx.search_partitioned(s["q"], radius=r, k=k, out=s["out"])
    elif kind == "learned":
        idx, d2, _ = ctx.search_learned(s["q"], radius=r, k=k, out=s["out"])
    elif kind == "batched":
        idx, _, _ = ctx.search_batched(s["xyz"], s["offs"], mode=c["mode"], radius=r, k=k,
                                       with_d2=False)
        return [idx]
    elif kind == "graph":
        s["graph"].launch()
        idx, d2 = s["graph"].idx, s["graph"].d2
    else:
        loss = ctx.mlp_train(r, k, n_samples=c["samples"], steps=c["steps"], batch=c["batch"],
                             seed=7)
        return [ctx.mlp_weights(), loss]
    return [idx, d2]


def work(case):
    """Inputs read once, rows written once; the tests of the neighbors found."""
    if case["kind"] == "train":
        per = 2 * (30 * 64 + 64 * 64 + 64)
        return {"bytes": 12.0 * case["n"] + case["steps"] * case["batch"] * 4.0 * 31,
                "flops": 3.0 * per * case["steps"] * case["batch"]}
    if "clouds" in case:
        n = nq = int(_sizes(case)[-1])
        own = True
    else:
        n, nq, own = case["n"], case.get("nq", case["n"]), "nq" not in case
    row = case["k"] * (4 if case["kind"] == "batched" else 8)
    return {"bytes": 12.0 * n + (0 if own else 12.0 * nq) + float(nq) * row,
            "flops": 8.0 * nq * case["k"]}


def _brute(p, q, case):
    """d2 in 64 bits of the rows that the inclusion rule (FP32, strict) and the
    order (d2, index) select; empty slots +inf."""
    nq, k = len(q), case["k"]
    r2 = torch.tensor(case["r"], dtype=torch.float32, device=DEV) ** 2
    out = torch.full((nq, k), math.inf, dtype=torch.float64, device=DEV)
    step = max(1, min(4096, (1 << 25) // len(p)))
    idx = torch.arange(len(p), device=DEV)
    none = torch.iinfo(torch.int64).max
    for a in range(0, nq, step):
        b = q[a:a + step]
        e = [b[:, i, None] - p[None, :, i] for i in range(3)]
        d = (e[0] * e[0] + e[1] * e[1]) + e[2] * e[2]
        ok = d < r2
        if case["mode"] == "knn":
            ok &= d > 0
        key = torch.where(ok, (d.view(torch.int32).long() << 32) | idx, none)
        kk = min(k, len(p))
        got = torch.topk(key, kk, largest=False, sorted=True).values
        j = (got & 0xffffffff).clamp_max(len(p) - 1)
        f = b.double()[:, None, :] - p.double()[j]
        out[a:a + step, :kk] = torch.where(got == none, math.inf, (f * f).sum(2))
    return out


def exact(case, seed):
    if case["kind"] in ("train", "batched"):
        return None
    if case["kind"] == "graph":
        offs = _sizes(case)
        xyz = _lattice(offs, _gen(seed))
        if int(offs[-1]) > 400_000:
            return None
        rows = [_brute(xyz[int(a):int(b)], xyz[int(a):int(b)], case)
                for a, b in zip(offs[:-1], offs[1:])]
        return [None, torch.cat(rows)]
    if case["n"] * case.get("nq", case["n"]) > 12_000_000_000:
        return None
    p, q = _points(case, seed)
    return [None, _brute(p, p if q is None else q, case)]
