"""The work users of this framework have it do, as measurable cases.

Every case goes through a public entry point of ``geogram_amd`` on a context
that a program keeps (``default_context()``), with the inputs a program has in
hand: seeds resident on the GPU, except where the path takes host arrays by
its nature (the primal tetrahedra are handed to host mesh code).

Ranges (``draw`` spreads sizes over their logarithm, odd sizes included):

====== ==================================================================
cells  500 .. 2,000,000 Voronoi seeds (uniform, half uniform + 8-Gaussian,
       16-Gaussian), Laguerre up to 500,000, periodic up to 300,000; with
       and without the neighbour CSR
lloyd  1,000 .. 200,000 seeds, 1 .. 10 iterations, one instance; or 2 .. 64
       instances of 500 .. 50,000 seeds
cvt    energy and gradient, 500 .. 500,000 seeds
ot     transport to 1e-4, 2,000 .. 200,000 uniform seeds (equal or
       log-normal masses), clustered seeds up to 60,000
knn    1,000 .. 500,000 points, k 1 .. 32, of the points themselves or of
       query points
surf   5,120 .. 81,920 triangles, 1,000 .. 100,000 seeds near the surface
rdt    1,000 .. 200,000 seeds, host arrays in and out
====== ==================================================================
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

import geogram_amd as ga
from geogram_amd import configs

BOX = np.array([0.0, 0.0, 0.0, 1.0, 1.0, 1.0])
MAX_NBRS, MAX_TETS = 18, 8  # per seed, over a whole diagram


# ------------------------------------------------------------------- cases

def listed():
    return [
        # the smallest instance of the batched workload: launches, copies and
        # synchronisations count
        dict(name="cells_small", op="cells", n=2000, kind=0, weighted=False, periodic=False,
             neighbors=True),
        # an ordinary odd-sized diagram, as RVD / mesh optimisation codes ask for
        dict(name="cells_uniform", op="cells", n=100_003, kind=0, weighted=False, periodic=False,
             neighbors=True),
        # the headline workload: half uniform, half clustered
        dict(name="cells_mixture", op="cells", n=2_000_000, kind=1, weighted=False, periodic=False,
             neighbors=True),
        # Laguerre cells at transport-like weights: what each step of a
        # transport or fluid solver evaluates
        dict(name="cells_laguerre", op="cells", n=300_007, kind=0, weighted=True, periodic=False,
             neighbors=True),
        # cosmology / homogenisation: the 3-torus
        dict(name="cells_periodic", op="cells", n=150_001, kind=0, weighted=False, periodic=True,
             neighbors=False),
        # CVT by Lloyd, the reference's own CVT example size
        dict(name="lloyd", op="lloyd", sizes="100000", kind=0, iters=5),
        # many small independent problems in one launch
        dict(name="lloyd_batch", op="lloyd", sizes="2003,2950,4321,6277,9001,13337,19999,29501,"
             "43210,2048,3333,5551", kind=2, iters=5),
        # one evaluation of a quasi-Newton CVT
        dict(name="cvt_func_grad", op="cvt", n=40_009, kind=1),
        # a whole transport solve from w = 0
        dict(name="transport", op="ot", n=120_000, kind=0, equal=True),
        # exact neighbour lists of a point cloud
        dict(name="knn_self", op="knn", n=100_003, nq=0, k=16, kind=0),
        # centroids restricted to a surface (remeshing)
        dict(name="surface", op="surf", level=6, n=50_021),
        # primal tetrahedra for host mesh code
        dict(name="rdt", op="rdt", n=60_000, kind=0),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["cells", "cells", "cells", "cells", "lloyd", "lloyd", "cvt", "ot", "knn",
                     "knn", "surf", "rdt"])
    if op == "cells":
        mode = rng.choice(["voronoi", "voronoi", "laguerre", "periodic"])
        hi = {"voronoi": 2_000_000, "laguerre": 500_000, "periodic": 300_000}[mode]
        return dict(op=op, n=_log(rng, 500, hi),
                    kind=rng.choice([0, 1, 2]) if mode == "voronoi" else 0,
                    weighted=mode == "laguerre", periodic=mode == "periodic",
                    neighbors=rng.random() < 0.7)
    if op == "lloyd":
        if rng.random() < 0.5:
            sizes = [_log(rng, 1000, 200_000)]
        else:
            sizes = [_log(rng, 500, 50_000) for _ in range(_log(rng, 2, 64))]
        return dict(op=op, sizes=",".join(map(str, sizes)), kind=rng.choice([0, 1, 2]),
                    iters=rng.randint(1, 10))
    if op == "cvt":
        return dict(op=op, n=_log(rng, 500, 500_000), kind=rng.choice([0, 1, 2]))
    if op == "ot":
        kind = rng.choice([0, 0, 2])
        return dict(op=op, n=_log(rng, 2000, 200_000 if kind == 0 else 60_000), kind=kind,
                    equal=rng.random() < 0.5)
    if op == "knn":
        return dict(op=op, n=_log(rng, 1000, 500_000),
                    nq=_log(rng, 100, 500_000) if rng.random() < 0.5 else 0,
                    k=_log(rng, 1, 32), kind=rng.choice([0, 1, 2]))
    if op == "surf":
        return dict(op=op, level=rng.choice([4, 5, 6]), n=_log(rng, 1000, 100_000))
    return dict(op=op, n=_log(rng, 1000, 200_000), kind=rng.choice([0, 1, 2]))


# ------------------------------------------------------------------ inputs

def _seeds(rng, n, kind):
    """Seeds in the unit cube: 0 uniform, 1 half uniform + 8-Gaussian
    mixture, 2 16-Gaussian mixture (the families of vgc_sample_points;
    Gaussian points beyond a face are mirrored back inside)."""
    if kind == 0:
        return rng.random((n, 3))
    nu = n // 2 if kind == 1 else 0
    c = 8 if kind == 1 else 16
    mean = rng.uniform(0.2, 0.8, (c, 3))
    sig = rng.uniform(0.01, 0.1, c) if kind == 1 else rng.uniform(0.02, 0.15, c)
    which = rng.integers(0, c, n - nu)
    g = mean[which] + sig[which, None] * rng.standard_normal((n - nu, 3))
    g = np.abs(g)
    g = 1.0 - np.abs(1.0 - g)
    g = np.clip(g, 1e-9, 1.0 - 1e-9)
    return np.concatenate([rng.random((nu, 3)), g])


def _weights(rng, x):
    """Laguerre weights |p|^2 - Phi(p) of a strictly convex Phi (cells moved
    away from their seeds as in a transport plan, none empty) plus noise of a
    tenth of the squared spacing."""
    n = x.shape[0]
    s = rng.uniform(0.92, 0.99, 3)
    h2 = n ** (-2.0 / 3.0)
    y = x - 0.5
    phi = (s * y * y).sum(1) + y.sum(1) + 0.02 * np.logaddexp(8.0 * y[:, 0], -8.0 * y[:, 1]) / 8.0
    return (x * x).sum(1) - phi + 0.1 * h2 * (rng.random(n) - 0.5)


@functools.lru_cache(maxsize=8)
def _sphere(level):
    return configs.icosphere(level)


def _inputs(case, seed):
    """Host inputs of a case, from the seed alone."""
    rng = np.random.default_rng([seed, 20])
    op = case["op"]
    if op in ("cells", "cvt", "rdt"):
        x = _seeds(rng, case["n"], case["kind"])
        return dict(x=x, w=_weights(rng, x) if case.get("weighted") else None)
    if op == "lloyd":
        sizes = [int(s) for s in case["sizes"].split(",")]
        return dict(x=np.concatenate([_seeds(rng, n, case["kind"]) for n in sizes]), sizes=sizes)
    if op == "ot":
        n = case["n"]
        x = _seeds(rng, n, case["kind"])
        nu = np.full(n, 1.0 / n) if case["equal"] else np.exp(rng.normal(0.0, 0.5, n))
        return dict(x=x, nu=nu / nu.sum())
    if op == "knn":
        x = _seeds(rng, case["n"], case["kind"])
        return dict(x=x, q=_seeds(rng, case["nq"], case["kind"]) if case["nq"] else None,
                    k=min(case["k"], case["n"] - 1))
    V, F = _sphere(case["level"])
    return dict(x=configs.sphere_seeds(case["n"], seed), V=V, F=F)


def prepare(case, seed):
    st = _inputs(case, seed)
    if case["op"] != "rdt":
        st = {k: torch.from_numpy(v).cuda() if isinstance(v, np.ndarray) else v
              for k, v in st.items()}
    if case["op"] == "lloyd":
        st["boxes"] = np.tile(BOX, (len(st["sizes"]), 1))
    # neighbour lists and tetrahedra vary in length with the seeds; the program
    # keeps them in arrays of its own, sized for the longest
    n = case.get("n", 0)
    if case["op"] == "cells" and case["neighbors"]:
        st["nbr"] = torch.full((MAX_NBRS * n,), -1, dtype=torch.int32, device="cuda")
        st["farea"] = torch.zeros(MAX_NBRS * n, dtype=torch.float64, device="cuda")
    if case["op"] == "rdt":
        st["tets"] = np.full((MAX_TETS * n, 4), -1, dtype=np.int32)
    st["case"] = case
    st["ctx"] = ga.default_context()
    return st


# -------------------------------------------------------------------- pass

def run(st):
    case, ctx = st["case"], st["ctx"]
    op = case["op"]
    if op == "cells":
        r = ctx.cells(st["x"], st["w"], BOX, neighbors=case["neighbors"],
                      periodic=case["periodic"])
        if not case["neighbors"]:
            return r.vol, r.mg
        m = r.nbr.shape[0]
        st["nbr"][:m] = r.nbr
        st["farea"][:m] = r.farea
        return r.vol, r.mg, r.nbr_ptr, st["nbr"], st["farea"]
    if op == "lloyd":
        if len(st["sizes"]) == 1:
            return ctx.lloyd(st["x"], case["iters"], BOX)[0]
        return ctx.lloyd(st["x"], case["iters"], inst_n=st["sizes"], boxes=st["boxes"])[0]
    if op == "cvt":
        return ctx.cvt_func_grad(st["x"], BOX)
    if op == "ot":
        return ctx.ot_solve(st["x"], st["nu"], None, BOX, 1e-4)[0]
    if op == "knn":
        if st["q"] is None:
            return ctx.knn(st["x"], st["k"])
        return ctx.knn_search(st["x"], st["q"], st["k"])
    if op == "surf":
        return ctx.surface_centroids(st["x"], st["V"], st["F"])[:2]
    t = ctx.rdt(st["x"], None, BOX)
    st["tets"][:t.shape[0]] = t
    return st["tets"]


# -------------------------------------------------------------------- work

# A cell of a random diagram has about 15.5 facets, 27 corners and 50
# integration tetrahedra; each facet's plane has to be tested against the
# corners alive at that time (about 20, 7 flops each) and each corner formed
# (66), each tetrahedron integrated (34).
CELL_FLOPS = 15.5 * 20 * 7 + 27 * 66 + 50 * 34
CELL_NBRS = 15.5


def work(case):
    op = case["op"]
    if op == "cells":
        n = case["n"]
        b = n * (24 + (8 if case["weighted"] else 0) + 32)
        if case["neighbors"]:
            b += n * (8 + 12 * CELL_NBRS)
        return dict(bytes=b, flops=n * CELL_FLOPS)
    if op == "lloyd":
        n = sum(int(s) for s in case["sizes"].split(",")) * case["iters"]
        return dict(bytes=48 * n, flops=n * CELL_FLOPS)
    if op == "cvt":
        n = case["n"]
        return dict(bytes=48 * n, flops=n * (CELL_FLOPS + 50 * 20))
    if op == "ot":
        # about 5 Newton steps (15 from clustered seeds) of one cell pass and
        # 4.2 n^(1/3) conjugate-gradient products each
        n, steps = case["n"], 5 if case["kind"] == 0 else 15
        its = steps * 4.2 * n ** (1.0 / 3.0)
        return dict(bytes=steps * n * (56 + 12 * CELL_NBRS) + its * n * (12 * CELL_NBRS + 120),
                    flops=steps * n * CELL_FLOPS + its * n * (2 * CELL_NBRS + 12))
    if op == "knn":
        n, q = case["n"], case["nq"] or case["n"]
        return dict(bytes=24 * n + (24 * q if case["nq"] else 0) + 12 * q * case["k"],
                    flops=q * 8 * 3 * case["k"])
    if op == "surf":
        t = 20 * 4 ** case["level"]
        # every triangle meets a few restricted cells, each clipped by about
        # eight bisectors
        return dict(bytes=t * 12 + t * 12 + case["n"] * 56, flops=t * 3 * 8 * 60)
    n = case["n"]
    return dict(bytes=24 * n + 6.7 * 16 * n, flops=n * (CELL_FLOPS - 50 * 34))


def tolerance(case):
    op = case["op"]
    if op in ("cells", "cvt"):
        # FP64 planes, corners and fans: against the polyhedra of `exact`,
        # volumes and moments differ by up to 3e-15 of the result's norm and
        # 1.5e-14 of its root mean square; small facets of large cells more
        return {"rel": 1e-13, "max": 1e-11}
    if op == "lloyd":
        # an iteration moves every seed by its cell's rounding, which the
        # next iterations carry on
        return {"rel": 1e-13}
    if op == "ot":
        # seeds moved by one unit in the last place (another order of every
        # sum) move the weights by up to 4e-9, through the stopping points of
        # conjugate gradients (relative residual 1e-7)
        return {"rel": 2e-8}
    if op == "surf":
        return {"rel": 1e-12, "max": 1e-9}
    return "exact"


# ------------------------------------------------------------------- exact

def _clip_cell(planes_e, planes_h, box):
    """Polyhedron {y : e_j . y <= h_j} in the box (seed-relative), clipped
    plane by plane in order of |plane distance|; returns (vol, first moment,
    second moment, neighbours) about the seed."""
    lo, hi = box
    X = [[lo[0], hi[0]], [lo[1], hi[1]], [lo[2], hi[2]]]

    def v(i, j, k):
        return (X[0][i], X[1][j], X[2][k])

    faces = [(-1, [v(0, 0, 0), v(0, 0, 1), v(0, 1, 1), v(0, 1, 0)]),
             (-1, [v(1, 0, 0), v(1, 1, 0), v(1, 1, 1), v(1, 0, 1)]),
             (-1, [v(0, 0, 0), v(1, 0, 0), v(1, 0, 1), v(0, 0, 1)]),
             (-1, [v(0, 1, 0), v(0, 1, 1), v(1, 1, 1), v(1, 1, 0)]),
             (-1, [v(0, 0, 0), v(0, 1, 0), v(1, 1, 0), v(1, 0, 0)]),
             (-1, [v(0, 0, 1), v(1, 0, 1), v(1, 1, 1), v(0, 1, 1)])]
    norm = np.sqrt((planes_e ** 2).sum(1))
    dist = planes_h / norm
    order = np.argsort(dist)
    R = math.sqrt(max(p[0] ** 2 + p[1] ** 2 + p[2] ** 2 for _, f in faces for p in f))
    for j in order:
        if dist[j] >= R * (1.0 + 1e-12):
            break
        ex, ey, ez = planes_e[j].tolist()
        h = float(planes_h[j])
        out, cut, touched = [], [], False
        for fid, poly in faces:
            s = [ex * p[0] + ey * p[1] + ez * p[2] - h for p in poly]
            if max(s) <= 0.0:
                out.append((fid, poly))
                continue
            touched = True
            if min(s) > 0.0:
                continue
            q = []
            for i in range(len(poly)):
                a, b, sa, sb = poly[i - 1], poly[i], s[i - 1], s[i]
                if (sa > 0.0) != (sb > 0.0):
                    # from the kept end, so both faces of an edge form the same point
                    if sa > 0.0:
                        a, b, sa, sb = b, a, sb, sa
                    t = sa / (sa - sb)
                    p = (a[0] + t * (b[0] - a[0]), a[1] + t * (b[1] - a[1]), a[2] + t * (b[2] - a[2]))
                    q.append(p)
                    cut.append(p)
                if s[i] <= 0.0:
                    q.append(poly[i])
            if len(q) >= 3:
                out.append((fid, q))
        if not touched:
            continue
        pts = list(dict.fromkeys(cut))
        if len(pts) >= 3:
            c = np.array(pts)
            m = c.mean(0)
            nrm = np.array([ex, ey, ez]) / norm[j]
            u = np.cross(nrm, [1.0, 0.0, 0.0] if abs(nrm[0]) < 0.7 else [0.0, 1.0, 0.0])
            w = np.cross(nrm, u)
            ang = np.arctan2((c - m) @ w, (c - m) @ u)
            out.append((int(j), [pts[i] for i in np.argsort(ang)]))
        faces = out
        if not faces:
            return 0.0, (0.0, 0.0, 0.0), 0.0, []
        R = math.sqrt(max(p[0] ** 2 + p[1] ** 2 + p[2] ** 2 for _, f in faces for p in f))
    o = np.mean([np.mean(f, axis=0) for _, f in faces], axis=0)
    tet = np.array([(f[0], f[i], f[i + 1]) for _, f in faces for i in range(1, len(f) - 1)])
    d = tet - o
    tv = np.abs(np.einsum("ij,ij->i", np.cross(d[:, 0], d[:, 1]), d[:, 2])) / 6.0
    s = tet.sum(1) + o
    mom = (tv[:, None] * s).sum(0) / 4.0
    e2 = float((tv * ((tet ** 2).sum((1, 2)) + (o ** 2).sum() + (s ** 2).sum(1))).sum() / 20.0)
    return float(tv.sum()), tuple(mom), e2, [f for f, _ in faces if f >= 0]


def _exact_cells(x, w, periodic):
    """Cells of x in the unit box: volumes, moments, second moments, facet
    counts."""
    n = x.shape[0]
    src = np.arange(n)
    xa, wa = x, np.zeros(n) if w is None else w
    lo, hi = BOX[:3], BOX[3:]
    if periodic:
        sh = np.array([(a, b, c) for a in (-1, 0, 1) for b in (-1, 0, 1) for c in (-1, 0, 1)], float)
        xa = np.concatenate([x + s for s in sh])
        wa = np.tile(wa, 27)
        src = np.tile(src, 27)
        near = np.all((xa > -0.5) & (xa < 1.5), axis=1)
        xa, wa, src = xa[near], wa[near], src[near]
        lo, hi = lo - 0.5, hi + 0.5
    vol, mg, e2, cnt = np.empty(n), np.empty((n, 3)), np.empty(n), np.empty(n, np.int64)
    for i in range(n):
        e = xa - x[i]
        d2 = (e * e).sum(1)
        keep = d2 > 0.0
        h = 0.5 * (d2 + (0.0 if w is None else w[i]) - wa)
        v, m, q, nb = _clip_cell(e[keep], h[keep], (lo - x[i], hi - x[i]))
        vol[i], mg[i], e2[i], cnt[i] = v, np.array(m) + v * x[i], q, len(nb)
    return vol, mg, e2, cnt


EXACT_CELLS = 2200  # cells that the loop above does in about 15 seconds


def exact(case, seed):
    op = case["op"]
    if op == "cells" and case["n"] <= (EXACT_CELLS if not case["periodic"] else 600):
        I = _inputs(case, seed)
        vol, mg, _, cnt = _exact_cells(I["x"], I["w"], case["periodic"])
        if not case["neighbors"]:
            return vol, mg
        return vol, mg, np.concatenate([[0], np.cumsum(cnt)]), None, None
    if op == "cvt" and case["n"] <= EXACT_CELLS:
        x = _inputs(case, seed)["x"]
        vol, mg, e2, _ = _exact_cells(x, None, False)
        return float(e2.sum()), 2.0 * (vol[:, None] * x - mg)
    if op == "lloyd":
        sizes = [int(s) for s in case["sizes"].split(",")]
        if len(sizes) == 1 and sizes[0] * case["iters"] <= EXACT_CELLS:
            x = _inputs(case, seed)["x"]
            for _ in range(case["iters"]):
                vol, mg, _, _ = _exact_cells(x, None, False)
                x = mg / vol[:, None]
            return x
    if op == "knn" and case["n"] * (case["nq"] or case["n"]) <= 1.1e10:
        I = _inputs(case, seed)
        x = torch.from_numpy(I["x"]).cuda()
        q = x if I["q"] is None else torch.from_numpy(I["q"]).cuda()
        k, step = I["k"], max(1, int(2e8 // x.shape[0]))
        idx, d2 = [], []
        for a in range(0, q.shape[0], step):
            b = min(q.shape[0], a + step)
            d = torch.zeros((b - a, x.shape[0]), dtype=torch.float64, device=x.device)
            for c in range(3):
                d += (x[None, :, c] - q[a:b, None, c]) ** 2
            if I["q"] is None:
                d[torch.arange(b - a), torch.arange(a, b)] = math.inf
            v, i = torch.topk(d, k, dim=1, largest=False, sorted=True)
            idx.append(i.to(torch.int32))
            d2.append(v)
        return torch.cat(idx), torch.cat(d2)
    return None
