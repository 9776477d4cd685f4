"""The framework's performance cases: what its users have it do, through its public entry points.

A case is a plain dict; `listed()` names the standing ones, `draw(rng)` gives another of the same
ranges, `prepare(case, seed)` makes the inputs and handles a program has in hand, `run(state)` is
one pass, `work(case)` the bytes and operations a pass cannot do without, and `exact(case, seed)`
the same outputs from plain torch in 64 bits (a brute-force walk over all generators), where
that is feasible.

Kinds:
  rays       one ray per (vertex, dropped generator): hv_raycast_batch_noalloc on device buffers
             (a caller's own walk in a loop that may not allocate), or Context.raycast_batch on
             host arrays
  nearest    half-space nearest-generator queries of host points
  inrange    range queries of host points
  mesh       the whole vertex table: build_mesh and its export
  volumes    cell volumes, neighbours and interface areas: build_mesh and the exact integrator
  geometry   the user-facing class: VoronoiGeometry from points to vertex table and integrals
  batch      independent meshes in one call, every vertex table exported
  montecarlo / points   the two Monte-Carlo integrators on a mesh the program keeps
  refine     new points into a kept mesh, the refined vertex table exported
"""
import itertools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "highvoronoi.jl_amd"))

from hvgpu import synth  # noqa: E402
from hvgpu._lib import PRECISIONS, Context, build_mesh_batch, lib  # noqa: E402
from hvgpu.geometry import (VI_FAST_POLYGON, VI_MONTECARLO, VI_POLYGON, VoronoiGeometry, cuboid)  # noqa: E402

INTEGRATORS = {"polygon": VI_POLYGON, "fast_polygon": VI_FAST_POLYGON, "montecarlo": VI_MONTECARLO}
# vertices and neighbours per generator of uniform points in a box
VERTICES = {2: 2.0, 3: 6.8, 4: 28.0, 5: 160.0, 6: 780.0}
PERIODIC_VERTICES = {2: 2.3, 3: 7.3, 4: 40.0, 5: 330.0, 6: 2850.0}
NEIGHBOURS = {2: 6, 3: 15, 4: 37, 5: 85, 6: 190}


def listed():
    return [
        # a serving loop's ray batch on device buffers: launches and latency count
        {"name": "rays-device-4d", "kind": "rays", "device": True, "d": 4, "n": 20000, "nrays": 256, "precision": "bf16"},
        # a host walk's rays of one level, through the host entry point
        {"name": "rays-host-5d", "kind": "rays", "device": False, "d": 5, "n": 30000, "nrays": 100000, "precision": "fp64"},
        # a few hundred point queries against a fixed set of generators
        {"name": "nearest-3d", "kind": "nearest", "d": 3, "n": 100000, "nq": 1000, "half": True},
        # ragged sizes: neither generators nor queries fill their last leaf or block
        {"name": "inrange-4d-ragged", "kind": "inrange", "d": 4, "n": 30011, "nq": 5003, "mean": 40},
        # the smallest configuration: 2D N=1000, points to volumes through the user-facing class
        {"name": "geometry-2d", "kind": "geometry", "d": 2, "n": 1000, "integrator": "polygon", "integrand": False,
         "periodic": False, "precision": "bf16"},
        # an ordinary 3D mesh, plain FP64 scan, with its vertex table on the host
        {"name": "mesh-3d-fp64", "kind": "mesh", "d": 3, "n": 50001, "points": "uniform", "precision": "fp64"},
        # the 4D configuration, N=20000: mesh and exact volumes
        {"name": "volumes-4d", "kind": "volumes", "d": 4, "n": 20000, "points": "uniform", "periodic": False,
         "precision": "bf16"},
        # the headline configuration: the 5D mixture of 100000 generators, mesh and exact volumes
        {"name": "volumes-5d-mixture", "kind": "volumes", "d": 5, "n": 100000, "points": "mixture", "periodic": False,
         "precision": "bf16"},
        # many independent small meshes of 3 to 6 dimensions
        {"name": "batch-16", "kind": "batch", "count": 16, "nmin": 200, "nmax": 800, "dmin": 3, "dmax": 6,
         "precision": "bf16"},
        # directional Monte Carlo with the default number of directions on the 4D configuration
        {"name": "montecarlo-4d", "kind": "montecarlo", "d": 4, "n": 20000, "ndir": 1000, "precision": "bf16"},
        # point samples in the periodic 6D cube
        {"name": "points-6d-periodic", "kind": "points", "d": 6, "n": 10000, "nsamples": 10000000, "periodic": True,
         "precision": "bf16"},
        # one per cent of new points into a 3D mesh
        {"name": "refine-3d-fp32", "kind": "refine", "d": 3, "n": 50000, "m": 500, "precision": "fp32"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["rays", "rays", "nearest", "inrange", "geometry", "mesh", "volumes", "volumes", "batch",
                       "montecarlo", "points", "refine"])
    precision = rng.choice(["bf16", "fp64", "fp32"])
    if kind == "rays":
        d, device = rng.randint(2, 6), rng.random() < 0.5
        return {"kind": kind, "device": device, "d": d, "precision": precision,
                "n": _log(rng, 500, {2: 200000, 3: 200000, 4: 50000, 5: 30000, 6: 5000}[d]),
                "nrays": _log(rng, 64, 32768 if device else 200000)}
    if kind == "nearest":
        return {"kind": kind, "d": rng.randint(2, 6), "n": _log(rng, 1000, 500000), "nq": _log(rng, 64, 50000),
                "half": rng.random() < 0.5}
    if kind == "inrange":
        return {"kind": kind, "d": rng.randint(2, 6), "n": _log(rng, 1000, 200000), "nq": _log(rng, 64, 20000),
                "mean": rng.randint(5, 60)}
    if kind == "geometry":
        d, periodic = rng.randint(2, 4), rng.random() < 0.4
        integrator = rng.choice(["polygon", "fast_polygon", "montecarlo"])
        return {"kind": kind, "d": d, "n": _log(rng, 200, {2: 20000, 3: 8000, 4: 1500}[d]), "integrator": integrator,
                "integrand": integrator != "montecarlo" and rng.random() < 0.4, "periodic": periodic,
                "precision": precision}
    if kind == "mesh":
        d = rng.randint(2, 6)
        return {"kind": kind, "d": d, "n": _log(rng, 200, {2: 150000, 3: 50000, 4: 12000, 5: 2200, 6: 500}[d]),
                "points": rng.choice(["uniform", "mixture"]), "precision": precision}
    if kind == "volumes":
        d, periodic = rng.randint(2, 6), rng.random() < 0.3
        top = {2: 500000, 3: 200000, 4: 80000, 5: 50000, 6: 5000}[d]
        return {"kind": kind, "d": d, "n": _log(rng, 300, top // 4 if periodic else top), "periodic": periodic,
                "points": "uniform" if periodic else rng.choice(["uniform", "mixture"]), "precision": precision}
    if kind == "batch":
        dmin = rng.randint(2, 4)
        return {"kind": kind, "count": rng.randint(3, 24), "nmin": 200, "nmax": rng.randint(300, 800), "dmin": dmin,
                "dmax": rng.randint(dmin, 6 if dmin > 2 else 5), "precision": precision}
    if kind == "montecarlo":
        d = rng.randint(2, 6)
        return {"kind": kind, "d": d, "n": _log(rng, 300, {2: 100000, 3: 50000, 4: 20000, 5: 10000, 6: 3000}[d]),
                "ndir": _log(rng, 50, 2000), "precision": "bf16"}
    if kind == "points":
        d, periodic = rng.randint(2, 6), rng.random() < 0.5
        return {"kind": kind, "d": d, "n": _log(rng, 500, {2: 50000, 3: 50000, 4: 20000, 5: 10000, 6: 5000}[d]),
                "nsamples": _log(rng, 100000, 10000000), "periodic": periodic, "precision": "bf16"}
    d = rng.randint(2, 5)
    n = _log(rng, 500, {2: 100000, 3: 50000, 4: 10000, 5: 2000}[d])
    return {"kind": kind, "d": d, "n": n, "m": max(1, int(n * math.exp(rng.uniform(math.log(0.001), math.log(0.05))))),
            "precision": precision}


# ---------------------------------------------------------------------------------------------
# inputs

class _Placement:
    """A seed's placement of a point set in the unit cube: one of the cube's symmetries (axes
    permuted, some reflected) and another numbering.  How many vertices, neighbours or hits a
    call returns follows from the set alone, which belongs to the case: every seed is other
    input and gives other values in outputs of one shape."""

    def __init__(self, d, seed):
        self.rng = np.random.default_rng(seed)
        self.axes, self.flip = self.rng.permutation(d), self.rng.random(d) < 0.5

    def points(self, x):
        x = x[:, self.axes]
        return np.where(self.flip, 1.0 - x, x)

    def directions(self, u):
        u = u[:, self.axes]
        return np.where(self.flip, -u, u)

    def shuffled(self, *arrays):
        order = self.rng.permutation(len(arrays[0]))
        return tuple(np.ascontiguousarray(a[order]) for a in arrays)


def _set(case, extra=0):
    d, n = case["d"], case["n"]
    if case.get("points") == "mixture":
        return synth.gaussian_mixture_5d(n, seed=2, d=d)
    return np.random.default_rng([d, n, extra]).random((n, d))


def _points(case, seed):
    place = _Placement(case["d"], seed)
    return place.shuffled(place.points(_set(case)))[0]


def _new_points(case, seed):
    place = _Placement(case["d"], seed)
    return place.shuffled(place.points(_set({"d": case["d"], "n": case["m"]}, 1)))[0]


def _batch_points(case, seed):
    rng = np.random.default_rng([case["count"], case["nmin"], case["nmax"], case["dmin"], case["dmax"]])
    out = []
    for k in range(case["count"]):
        d = case["dmin"] + k % (case["dmax"] - case["dmin"] + 1)
        n = int(math.exp(rng.uniform(math.log(case["nmin"]), math.log(case["nmax"]))))
        place = _Placement(d, [seed, k])
        out.append(place.shuffled(place.points(rng.random((n, d))))[0])
    return out


def _queries(case, seed):
    d, nq = case["d"], case["nq"]
    place, rng = _Placement(d, seed), np.random.default_rng([d, case["n"], nq])
    q = rng.random((nq, d))
    if case["kind"] == "inrange":
        ball = math.pi ** (d / 2) / math.gamma(d / 2 + 1)
        r = (case["mean"] / (ball * case["n"])) ** (1.0 / d) * rng.uniform(0.7, 1.2, nq)
        return place.shuffled(place.points(q), r)
    u = rng.standard_normal((nq, d))
    u /= np.linalg.norm(u, axis=1, keepdims=True)
    q, u = place.shuffled(place.points(q), place.directions(u))
    return q, u, (u * q).sum(1) if case["half"] else np.full(nq, -np.inf)


def _context(x, periodic=False):
    d = x.shape[1]
    ctx = Context(0)
    ctx.set_points(x)
    ctx.set_boundary(*cuboid(d, periodic=None if periodic else []).arrays())
    return ctx


def _rays(case, ctx, seed):
    """nrays walkable (vertex, dropped position) pairs of the mesh, as a walk meets them."""
    d, n, nrays = case["d"], case["n"], case["nrays"]
    rng = np.random.default_rng(seed + 2)
    cells = rng.permutation(n)[:min(n, int(nrays / VERTICES[d]) + 8)] + 1
    m = ctx.build_mesh_cells(np.sort(cells), precision=case["precision"])
    keys, coords = m.export()
    m.free()
    v, p = np.divmod(rng.permutation(len(keys) * (d + 1)), d + 1)
    first = np.where(p == 0, keys[v, 1], keys[v, 0])   # the edge left has to hold a generator
    v, p = v[first <= n], p[first <= n]
    v, p = np.resize(v, nrays), np.resize(p, nrays)
    return keys[v].astype(np.int64), p.astype(np.int32), coords[v]


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case}
    if kind == "geometry":
        s["x"], s["boundary"] = _points(case, seed), cuboid(case["d"], periodic=None if case["periodic"] else [])
        return s
    if kind == "batch":
        s["x"] = _batch_points(case, seed)
        s["planes"] = [synth.cube_planes(x.shape[1]) for x in s["x"]]
        return s
    x = _points(case, seed)
    s["ctx"] = ctx = _context(x, case.get("periodic", False))
    if kind in ("nearest", "inrange"):
        s["q"] = _queries(case, seed)
    elif kind == "rays":
        s["rays"] = sig, drop, r = _rays(case, ctx, seed)
        if case["device"]:
            ctx.raycast_batch(sig, drop, r, precision=case["precision"])   # the tree the device calls run on
            s["in"] = [torch.from_numpy(a).cuda() for a in (sig, drop, r)]
            s["out"] = [torch.empty_like(s["in"][0]), torch.empty_like(s["in"][2]),
                        torch.empty(len(sig), dtype=torch.float64, device="cuda"), torch.empty_like(s["in"][1])]
    elif kind in ("montecarlo", "points", "refine"):
        s["mesh"] = ctx.build_mesh(precision=case["precision"])
        s["seed"] = seed & 0xffff
        if kind == "refine":
            s["new"] = _new_points(case, seed)
    return s


# ---------------------------------------------------------------------------------------------
# one pass

def _integrand(p):
    return np.stack([p[:, 0], p[:, 1] ** 2], axis=1)


def _integrals(r):
    return {k: r[k] for k in ("volumes", "nbr_ptr", "neighbors", "areas", "bulk", "interface") if k in r}


def _table(mesh):
    keys, coords = mesh.export()
    mesh.free()
    return {"keys": keys, "coords": coords}


def run(s):
    case = s["case"]
    kind, ctx = case["kind"], s.get("ctx")
    if kind == "rays":
        if not case["device"]:
            sig, drop, r = s["rays"]
            return ctx.raycast_batch(sig, drop, r, precision=case["precision"])
        rc = lib().hv_raycast_batch_noalloc(ctx._h, PRECISIONS[case["precision"]], case["nrays"],
                                            *[t.data_ptr() for t in s["in"] + s["out"]])
        if rc:
            raise RuntimeError(f"hv_raycast_batch_noalloc: {rc}")
        return s["out"]
    if kind == "nearest":
        return ctx.nn_halfspace(*s["q"])
    if kind == "inrange":
        return ctx.inrange(*s["q"])
    if kind == "mesh":
        return _table(ctx.build_mesh(precision=case["precision"]))
    if kind == "volumes":
        mesh = ctx.build_mesh(precision=case["precision"])
        r = ctx.integrate(mesh, "polytope")
        mesh.free()
        return _integrals(r)
    if kind == "geometry":
        VG = VoronoiGeometry(s["x"], s["boundary"], integrator=INTEGRATORS[case["integrator"]],
                             search_settings={"precision": case["precision"]},
                             integrand=_integrand if case["integrand"] else None)
        keys, coords = VG.vertex_table()
        return {"keys": keys, "coords": coords, **_integrals(VG.integral)}
    if kind == "batch":
        meshes, status = build_mesh_batch(s["x"], s["planes"], precision=case["precision"])
        if status.any():
            raise RuntimeError(f"hv_build_mesh_batch: {sorted(set(status.tolist()))}")
        return [_table(m) for m in meshes]
    if kind == "montecarlo":
        return _integrals(ctx.integrate(s["mesh"], "montecarlo", ndir=case["ndir"], seed=s["seed"]))
    if kind == "points":
        return _integrals(ctx.integrate(s["mesh"], "points", nsamples=case["nsamples"], seed=s["seed"]))
    mesh, _ = ctx.refine(s["mesh"], s["new"], precision=case["precision"])
    return _table(mesh)


# ---------------------------------------------------------------------------------------------
# the least a pass moves and computes

def work(case):
    kind = case["kind"]
    if kind == "batch":
        sizes = [x.shape for x in _batch_points(case, 0)]
        per = [work({"kind": "mesh", "d": d, "n": n}) for n, d in sizes]
        return {k: sum(w[k] for w in per) for k in ("bytes", "flops")}
    d, n = case["d"], case["n"]
    if kind == "refine":
        n += case["m"]
    nv = n * (PERIODIC_VERTICES if case.get("periodic") else VERTICES)[d]
    rows = n * NEIGHBOURS[d]
    points, table, areas = 8 * d * n, 8 * (2 * d + 1) * nv, 16 * rows + 16 * n
    solve = 2 * d ** 3 / 3 + 4 * d * d                  # a vertex from its d + 1 generators
    faces = 2 * d * (d + 1) * 2 ** (d - 1)              # one height per (face, sub-face) of a vertex
    if kind == "rays":
        m = case["nrays"]
        return {"bytes": m * (16 * (d + 1) + 16 * d + 16), "flops": m * (solve + 4 * d * d)}
    if kind == "nearest":
        m = case["nq"]
        return {"bytes": points + m * (16 * d + 24), "flops": m * 4 * d}
    if kind == "inrange":
        m = case["nq"]
        return {"bytes": points + m * (8 * d + 16 + 8 * case["mean"]), "flops": 2 * d * m * case["mean"]}
    if kind in ("mesh", "refine"):
        return {"bytes": points + table, "flops": nv * (solve + 2 * d * (d + 1))}
    if kind == "volumes":
        return {"bytes": points + areas, "flops": nv * (solve + 2 * d * (d + 1) + faces)}
    if kind == "geometry":
        return {"bytes": points + areas + table, "flops": nv * (solve + 2 * d * (d + 1) + faces)}
    keys = (4 * (d + 1) + 8 * d) * nv                   # the kept mesh, read once
    if kind == "montecarlo":
        return {"bytes": points + areas + keys, "flops": 4.0 * d * rows * case["ndir"]}
    return {"bytes": points + areas + keys, "flops": 4.0 * d * case["nsamples"]}


# ---------------------------------------------------------------------------------------------
# the same outputs in plain torch, 64 bits

PAIRS = 4e10      # (ray, generator) pairs a brute-force walk may evaluate


class _Box:
    """Generators 0 .. n-1 and the unit box's planes n + 2k (x_k = 1) and n + 2k + 1 (x_k = 0)."""

    def __init__(self, x):
        self.x = torch.as_tensor(np.ascontiguousarray(x), dtype=torch.float64)
        if torch.cuda.is_available():
            self.x = self.x.cuda()
        self.n, self.d = self.x.shape
        eye = torch.eye(self.d, dtype=torch.float64, device=self.x.device)
        self.normal = torch.stack([eye, -eye], dim=1).reshape(2 * self.d, self.d)
        self.h = torch.tensor([1.0, 0.0] * self.d, dtype=torch.float64, device=self.x.device)
        self.xx = (self.x * self.x).sum(1)

    def rows(self, ids, x0):
        """Row and right-hand side of {y : equidistant to x0 and ids} relative to x0."""
        gen = (ids < self.n)[:, None]
        v = self.x[ids.clamp(max=self.n - 1)] - x0
        nrm = self.normal[(ids - self.n).clamp(min=0)]
        plane = self.h[(ids - self.n).clamp(min=0)] - (nrm * x0).sum(1)
        return torch.where(gen, 2 * v, nrm), torch.where(gen[:, 0], (v * v).sum(1), plane)

    def step(self, a, b, q, beta):
        """Gram-Schmidt of row a (right-hand side b) against the unit rows q with sides beta."""
        for _ in range(2):
            for qi, bi in zip(q, beta):
                c = (a * qi).sum(1)
                a = a - c[:, None] * qi
                b = b - c * bi
        s = a.norm(dim=1)
        return a / s[:, None], b / s

    def centre(self, keys):
        """The vertex of each sorted key (d + 1 ids), with one refinement."""
        x0 = self.x[keys[:, 0]]
        rows = [self.rows(keys[:, j], x0) for j in range(1, self.d + 1)]
        y = torch.zeros_like(x0)
        for _ in range(2):
            q, beta = [], []
            for a, b in rows:
                qa, bb = self.step(a, b - (a * y).sum(1), q, beta)
                q.append(qa)
                beta.append(bb)
            y = y + sum(qa * bb[:, None] for qa, bb in zip(q, beta))
        return x0 + y

    def cast(self, edge, drop, r):
        """The first generator or plane met from r along the edge, away from drop; and its t."""
        n, d = self.n, self.d
        x0 = self.x[edge[:, 0]]
        zero = torch.zeros(len(edge), dtype=torch.float64, device=x0.device)
        q = []
        for j in range(d - 1, 0, -1):
            q.append(self.step(self.rows(edge[:, j], x0)[0], zero, q, [zero] * len(q))[0])
        u = -self.step(self.rows(drop, x0)[0], zero, q, [zero] * len(q))[0]
        win, t = [], []
        size = max(1, int(1.5e8 / n))
        for a in range(0, len(edge), size):
            s = slice(a, a + size)
            ux0, rx0 = (u[s] * x0[s]).sum(1), (r[s] * x0[s]).sum(1)
            den = 2 * (u[s] @ self.x.T - ux0[:, None])
            tg = (self.xx[None] - 2 * (r[s] @ self.x.T) + (2 * rx0 - (x0[s] ** 2).sum(1))[:, None]) / den
            tg[den <= 1e-13] = math.inf
            nu = u[s] @ self.normal.T
            tp = (self.h[None] - r[s] @ self.normal.T) / nu
            tp[nu <= 1e-14] = math.inf
            tt = torch.cat([tg, tp], dim=1)
            tt.scatter_(1, torch.cat([edge[s], drop[s][:, None]], dim=1), math.inf)
            best = tt.min(dim=1)
            win.append(best.indices)
            t.append(best.values)
        return torch.cat(win), torch.cat(t)

    @staticmethod
    def hashed(ids):
        h = torch.full((len(ids),), 0x1234567, dtype=torch.int64, device=ids.device)
        for j in range(ids.shape[1]):
            h = (h ^ ids[:, j]) * -7046029254386353131
            h = h ^ (h >> 29)
        return h

    def walk(self):
        """Every vertex: (keys, coordinates) in lexicographic key order, from the box's corners."""
        n, d, dev = self.n, self.d, self.x.device
        corner = torch.tensor(list(itertools.product([0.0, 1.0], repeat=d)), dtype=torch.float64, device=dev)
        near = torch.stack([((self.x - c) ** 2).sum(1).argmin() for c in corner])
        planes = n + 2 * torch.arange(d, device=dev)[None] + (corner == 0).long()
        new, at = torch.cat([near[:, None], planes], dim=1), corner
        keys, coords = [new], [at]
        before = torch.zeros(0, dtype=torch.int64, device=dev)
        while len(new):
            cols = torch.arange(d + 1, device=dev)
            edge = torch.cat([new[:, cols != p] for p in range(d + 1)])
            drop = new.T.reshape(-1)
            r = at.repeat(d + 1, 1)
            h = self.hashed(edge)
            _, inv, cnt = torch.unique(h, return_inverse=True, return_counts=True)
            left = (edge[:, 0] < n) & (cnt[inv] == 1) & ~torch.isin(h, before)
            edge, drop, r, before = edge[left], drop[left], r[left], h[left]
            if not len(edge):
                break
            win, _ = self.cast(edge, drop, r)
            found = torch.cat([edge, win[:, None]], dim=1).sort(dim=1).values
            hk, order = self.hashed(found).sort()
            first = torch.ones_like(hk, dtype=torch.bool)
            first[1:] = hk[1:] != hk[:-1]
            new = found[order[first]]
            at = self.centre(new)
            keys.append(new)
            coords.append(at)
        keys, coords = torch.cat(keys), torch.cat(coords)
        for j in range(d, -1, -1):   # stable sorts, the last column first
            order = keys[:, j].argsort(stable=True)
            keys, coords = keys[order], coords[order]
        return keys, coords

    def pairs(self, keys):
        """Neighbour rows (cell * (n + 2d) + neighbour), sorted."""
        out = [keys[:, a] * (self.n + 2 * self.d) + keys[:, b]
               for a in range(self.d + 1) for b in range(self.d + 1) if a != b]
        rows = torch.unique(torch.cat(out))
        return rows[rows < self.n * (self.n + 2 * self.d)]

    def integrals(self, keys):
        """Volumes and areas as signed sums over the flags (cell, facet, .., vertex): the foot
        points of the cell's generator on the nested faces are at the Gram-Schmidt sides beta."""
        n, d = self.n, self.d
        wide = n + 2 * d
        rows = self.pairs(keys)
        area = torch.zeros(len(rows), dtype=torch.float64, device=self.x.device)
        vol = torch.zeros(n, dtype=torch.float64, device=self.x.device)
        for a in range(d + 1):
            k = keys[keys[:, a] < n]
            i = k[:, a]
            x0 = self.x[i]
            con = {j: self.rows(k[:, j], x0) for j in range(d + 1) if j != a}

            def below(used, q, beta, product):
                if len(used) == d:
                    return product
                total = 0.0
                for j in con:
                    if j not in used:
                        qa, b = self.step(*con[j], q, beta)
                        total = total + below(used + [j], q + [qa], beta + [b], product * b)
                return total

            for j in con:
                qa, b = self.step(*con[j], [], [])
                f = below([j], [qa], [b], torch.ones_like(b)) / math.factorial(d - 1)
                area.index_add_(0, torch.searchsorted(rows, i * wide + k[:, j]), f)
                vol.index_add_(0, i, f * b / d)
        return rows, vol, area

    def directions(self, keys, ndir, seed):
        """The directional Monte-Carlo estimate with the stream's directions (splitmix64,
        Box-Muller), each interface averaged over its two sides."""
        n, d, dev = self.n, self.d, self.x.device
        wide = n + 2 * d
        rows = self.pairs(keys)
        cell, nb = rows // wide, rows % wide
        ptr = torch.searchsorted(rows, torch.arange(n + 1, device=dev) * wide)
        x0 = self.x[cell]
        nrm = self.normal[(nb - n).clamp(min=0)]
        mirror = x0 + 2 * (self.h[(nb - n).clamp(min=0)] - (nrm * x0).sum(1))[:, None] * nrm
        e = torch.where((nb < n)[:, None], self.x[nb.clamp(max=n - 1)], mirror) - x0
        width = int((ptr[1:] - ptr[:-1]).max())
        at = ptr[:-1, None] + torch.arange(width, device=dev)[None]
        has = at < ptr[1:, None]
        at = at.clamp(max=len(rows) - 1)
        ee = e[at]                                         # n x width x d
        num = (ee * ee).sum(2)

        def unif(i):
            z = seed + (i + 1) * -7046029254386353131
            for shift, mul in ((30, -4658895280553007687), (27, -7723592293110705685)):
                z = (z ^ ((z >> shift) & ((1 << (64 - shift)) - 1))) * mul
            z = z ^ ((z >> 31) & ((1 << 33) - 1))
            return ((z >> 11) & ((1 << 53) - 1)).double() / 9007199254740992.0

        vol = torch.zeros(n, dtype=torch.float64, device=dev)
        area = torch.zeros(len(rows), dtype=torch.float64, device=dev)
        even = (d + 1) // 2 * 2
        size = max(1, int(4e7 / (n * width)))
        for q0 in range(0, ndir, size):
            q = torch.arange(q0, min(ndir, q0 + size), device=dev)
            base = (torch.arange(n, device=dev)[:, None] * ndir + q[None]) * even
            u = []
            for c in range(0, d, 2):
                p = (base + c) >> 1
                rad, ang = torch.sqrt(-2 * torch.log(unif(2 * p).clamp(min=1e-300))), 2 * math.pi * unif(2 * p + 1)
                u += [rad * torch.cos(ang), rad * torch.sin(ang)]
            u = torch.stack(u[:d], dim=2)
            u = u / u.norm(dim=2, keepdim=True)            # n x chunk x d
            den = sum(u[:, :, None, c] * ee[:, None, :, c] for c in range(d))
            t = torch.where((den > 0) & has[:, None], num[:, None] / (2 * den), math.inf)
            t, w = t.min(dim=2)
            vol += (t ** d).sum(1)
            cos = den.gather(2, w[..., None])[..., 0] / num.gather(1, w).sqrt()
            area.index_add_(0, at.gather(1, w).reshape(-1), (t ** (d - 1) / cos).reshape(-1))
        ball = math.pi ** (d / 2) / math.gamma(d / 2 + 1)
        vol, area = vol * ball / ndir, area * ball * d / ndir
        lower = (nb < cell).nonzero()[:, 0]                # (i, k), k < i: the two sides of an interface
        i, k = cell[lower], nb[lower]
        back = torch.searchsorted(rows, k * wide + i)
        old, other = area[lower], area[back]
        mean = torch.where(other < old * 1e-10, old, 0.5 * (old + other))
        f = 0.5 * (self.x[i] - self.x[k]).norm(dim=1) / d
        vol.index_add_(0, k, (mean - other) * f)
        vol.index_add_(0, i, (mean - old) * f)
        area[lower] = mean
        area[back] = mean
        return rows, vol, area

    def rows_out(self, rows, vol, area):
        wide = self.n + 2 * self.d
        ptr = torch.searchsorted(rows, torch.arange(self.n + 1, device=rows.device) * wide)
        return {"volumes": vol.cpu(), "nbr_ptr": ptr.cpu(), "neighbors": (rows % wide + 1).cpu(), "areas": area.cpu()}


def _walkable(n, d):
    return n * VERTICES[d] * (d + 1) / 2 * n <= PAIRS


def exact(case, seed):
    kind = case["kind"]
    if kind in ("points", "inrange"):   # sample counts by position in the program's own strata; whole numbers
        return None
    if kind == "batch":
        points = _batch_points(case, seed)
        if sum(x.shape[0] * VERTICES[x.shape[1]] for x in points) > 2e6:
            return None
        tables = [_Box(x).walk() for x in points]
        return [{"keys": (k + 1).cpu(), "coords": c.cpu()} for k, c in tables]
    x = _points(case, seed)
    d, n = case["d"], case["n"]
    if kind == "nearest":
        q, u, c = (torch.as_tensor(a) for a in _queries(case, seed))
        if case["nq"] * n > PAIRS:
            return None
        box = _Box(x)
        q, u, c = (a.to(box.x.device) for a in (q, u, c))
        idx, dist = [], []
        size = max(1, int(1e8 / n))
        for a in range(0, len(q), size):
            s = slice(a, a + size)
            d2 = sum((box.x[None, :, k] - q[s, k][:, None]) ** 2 for k in range(d))
            d2[u[s] @ box.x.T <= c[s][:, None]] = math.inf
            best = d2.min(dim=1)
            idx.append(torch.where(best.values < math.inf, best.indices + 1, 0))
            dist.append(best.values.sqrt())
        return torch.cat(idx).cpu(), torch.cat(dist).cpu()
    if kind == "rays":
        if case["nrays"] * n > PAIRS:
            return None
        box = _Box(x)
        sig, drop, r = (torch.as_tensor(a).to(box.x.device) for a in _rays(case, _context(x), seed))
        sig, pos = sig - 1, drop.long()
        cols = torch.arange(d + 1, device=sig.device)
        edge = sig[cols[None] != pos[:, None]].reshape(-1, d)
        win, t = box.cast(edge, sig.gather(1, pos[:, None])[:, 0], r)
        key = torch.cat([edge, win[:, None]], dim=1).sort(dim=1).values
        return (key + 1).cpu(), box.centre(key).cpu(), t.cpu(), torch.zeros_like(drop).cpu()
    if case.get("periodic") or case.get("integrand"):
        return None
    if kind == "refine":
        x = np.concatenate([x, _new_points(case, seed)])
        n = len(x)
    if not _walkable(n, d):
        return None
    box = _Box(x)
    keys, coords = box.walk()
    out = {}
    if kind in ("mesh", "refine", "geometry"):
        out = {"keys": (keys + 1).cpu(), "coords": coords.cpu()}
    if kind == "montecarlo":
        out.update(box.rows_out(*box.directions(keys, case["ndir"], seed & 0xffff)))
    elif kind == "geometry" and case["integrator"] == "montecarlo":
        out.update(box.rows_out(*box.directions(keys, 1000, 0)))
    elif kind in ("volumes", "geometry"):
        out.update(box.rows_out(*box.integrals(keys)))
    return out
