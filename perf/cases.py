"""The work this library is used for, as cases that can be timed.

A case is a dict of plain values; ``prepare`` makes what a program holds
before the call (inputs in GPU or host memory, a server, resident meshes),
``run`` is one pass through the public entry points and returns what they
wrote, ``work`` the bytes and operations one pass cannot do without, and
``exact`` the value of computed numbers in 64 bits.

Kinds of work:

* ``rcb``    one partition of points in GPU memory (``Rcb.partition``)
* ``host``   the same from host memory, through coupe's own C entry point
* ``rib``    one inertial partition of points in GPU memory
* ``batch``  many independent instances of both dimensions in one call
* ``serve``  a burst of requests to a running server: new meshes from host
             memory and repartitions of meshes resident in HBM
* ``grid``   ``Grid.rcb`` on a cartesian grid of weights in GPU memory
* ``loads``  per-part loads and imbalance of a partition in GPU memory
"""
import math
import random

import numpy as np
import torch

import coupe_amd
from coupe_amd import imbalance

DEV = "cuda:0"
_WBYTES = {"unit": 8, "int32": 4, "int64": 8, "whole": 8, "lognormal": 8, "real": 8}


def listed():
    return [
        # a coarse mesh or one block of a small one: all latency and launches
        dict(name="rcb_2d_1k", kind="rcb", n=1021, dim=2, points="uniform", weights="unit", levels=3, tol=0.05),
        # a small request of the served range (10^4 points)
        dict(name="rcb_3d_10k", kind="rcb", n=10007, dim=3, points="uniform", weights="int32", levels=6, tol=0.01),
        # 2^20 uniform points in the plane, 8 parts, unit weights
        dict(name="rcb_2d_1m", kind="rcb", n=1 << 20, dim=2, points="uniform", weights="unit", levels=3, tol=0.05),
        # an ordinary mesh whose element costs are measured times (not whole numbers)
        dict(name="rcb_3d_real", kind="rcb", n=300007, dim=3, points="uniform", weights="real", levels=8, tol=0.02),
        # 2^24 points around 8 centres into 1024 parts: splits far from the boxes' middles
        dict(name="rcb_3d_gauss", kind="rcb", n=1 << 24, dim=3, points="gauss", weights="whole", levels=10, tol=0.01),
        # the largest mesh: 512^3 jittered cell centres into 4096 parts
        dict(name="rcb_3d_grid", kind="rcb", n=1 << 27, dim=3, points="jgrid", weights="lognormal", levels=12,
             tol=0.01),
        # a program that keeps its mesh in host memory and calls coupe's interface
        dict(name="host_3d", kind="host", n=3000017, dim=3, points="uniform", weights="int64", levels=10, tol=0.01),
        # an elongated cloud cut along its inertia axes
        dict(name="rib_3d", kind="rib", n=(1 << 21) - 5, dim=3, points="gauss", weights="int64", levels=9, tol=0.02),
        # 4096 instances of 10^3..10^6 points, 16 to 256 parts each, in one call
        dict(name="batch_mixed", kind="batch", count=4096, sizes_seed=3, lg_lo=3.0, lg_hi=6.0, tol=0.02),
        # a burst of requests, three in ten repartitions of resident meshes
        dict(name="serve_burst", kind="serve", count=20, sizes_seed=4, lg_lo=4.0, lg_hi=6.5, tol=0.01),
        # the reference's own cartesian benchmark: 10000 x 10000 cells, 4096 parts
        dict(name="grid_2d", kind="grid", nx=10000, ny=10000, nz=0, weights="whole", levels=12),
        # the check after a partition: loads and imbalance over 1024 parts
        dict(name="loads_1k", kind="loads", n=(1 << 24) + 77, parts=1024, weights="real"),
    ]


def _lg(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random):
    kind = rng.choice(["rcb", "rcb", "rcb", "rcb", "host", "rib", "batch", "serve", "grid", "loads"])
    weights = rng.choice(["unit", "int32", "int64", "whole", "lognormal", "real"])
    if kind in ("rcb", "host", "rib"):
        n = _lg(rng, 1000, {"rcb": 6e7, "host": 6e6, "rib": 1e7}[kind])
        points = rng.choice(["uniform", "gauss", "graded"])
        dim = 3 if points == "graded" else rng.choice([2, 3])
        if points == "graded":   # whole cells: the nearest cube
            n = max(10, round(n ** (1 / 3))) ** 3
        most = min(12, max(3, int(math.log2(n)) - 6))
        return dict(kind=kind, n=n, dim=dim, points=points, weights=weights, levels=rng.randint(3, most),
                    tol=rng.choice([0.01, 0.02, 0.05]))
    if kind == "batch":
        return dict(kind=kind, count=_lg(rng, 16, 2000), sizes_seed=rng.randrange(1 << 20), lg_lo=3.0,
                    lg_hi=round(rng.uniform(4.0, 6.0), 2), tol=0.02)
    if kind == "serve":
        return dict(kind=kind, count=rng.randint(4, 24), sizes_seed=rng.randrange(1 << 20), lg_lo=4.0,
                    lg_hi=round(rng.uniform(4.5, 6.5), 2), tol=0.01)
    if kind == "grid":
        cells = _lg(rng, 1e4, 6e7)
        if rng.random() < 0.5:
            nx = _lg(rng, 50, cells / 50)
            return dict(kind=kind, nx=nx, ny=max(2, cells // nx), nz=0, weights=weights, levels=rng.randint(4, 12))
        side = max(8, round(cells ** (1 / 3)))
        nx, ny = _lg(rng, side / 2, side * 2), _lg(rng, side / 2, side * 2)
        return dict(kind=kind, nx=nx, ny=ny, nz=max(2, cells // (nx * ny)), weights=weights,
                    levels=rng.randint(4, 12))
    return dict(kind=kind, n=_lg(rng, 1e4, 6e7), parts=_lg(rng, 2, 4096), weights=weights)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _rand(shape, g):
    return torch.rand(shape, generator=g, device=DEV, dtype=torch.float64)


def _weights(kind, n, g):
    if kind == "unit":
        return torch.ones(n, device=DEV, dtype=torch.float64)
    if kind == "int32":
        return torch.randint(1, 101, (n,), generator=g, device=DEV, dtype=torch.int32)
    if kind == "int64":
        return torch.randint(1, 101, (n,), generator=g, device=DEV, dtype=torch.int64)
    if kind == "whole":
        return torch.floor(_rand(n, g).mul_(100.0)).add_(1.0)
    if kind == "lognormal":
        w = torch.randn(n, generator=g, device=DEV, dtype=torch.float64)
        return w.exp_().mul_(10.0).round_().add_(1.0)
    return _rand(n, g).mul_(9.5).add_(0.5)


def _points(kind, n, dim, g):
    if kind == "uniform":
        return _rand((n, dim), g)
    if kind == "gauss":
        centres = _rand((8, dim), g)
        which = torch.randint(0, 8, (n,), generator=g, device=DEV)
        p = torch.randn((n, dim), generator=g, device=DEV, dtype=torch.float64).mul_(0.05)
        return p.add_(centres[which])
    m = round(n ** (1 / 3))   # jittered centres of an m^3 grid, x fastest
    p = _rand((n, dim), g).sub_(0.5).mul_(0.5).add_(0.5)
    i = torch.arange(n, device=DEV, dtype=torch.int64)
    p[:, 0].add_(i % m)
    p[:, 1].add_((i // m) % m)
    p[:, 2].add_(i // (m * m))
    p.div_(m)
    if kind == "graded":   # cells that grow away from three faces, as in a boundary layer
        p.pow_(1.0 + 0.5 * _rand((1, dim), g))
    return p


def _instances(case):
    """(n, dimension, iter_count, tolerance) of a batch's instances."""
    r = random.Random(case["sizes_seed"])
    return [(round(10 ** r.uniform(case["lg_lo"], case["lg_hi"])), r.choice([2, 3]), r.randint(4, 8), case["tol"])
            for _ in range(case["count"])]


def _requests(case):
    """(n, iter_count, resident) of a burst's requests."""
    r = random.Random(case["sizes_seed"])
    return [(round(10 ** r.uniform(case["lg_lo"], case["lg_hi"])), r.randint(6, 12), k % 10 in (2, 5, 8))
            for k in range(case["count"])]


_SERVER = None


def _server():
    global _SERVER
    if _SERVER is None:
        _SERVER = coupe_amd.Server(device=0, slots=4, memory_budget=64 << 30, max_batch_points=1 << 26,
                                   max_batch_requests=64)
    return _SERVER


class _Resident:
    """A mesh resident on the server, given back with its last user."""

    def __init__(self, points, weights):
        self.mesh = _server().create_mesh(points, weights)

    def __del__(self):
        self.mesh.destroy()


def prepare(case, seed):
    kind = case["kind"]
    g = _gen(seed)
    if kind in ("rcb", "rib", "host"):
        pts = _points(case["points"], case["n"], case["dim"], g)
        if kind == "rib":
            pts[:, 0].mul_(3.0).add_(pts[:, 1], alpha=0.7)
        w = _weights(case["weights"], case["n"], g)
        algo = (coupe_amd.Rib if kind == "rib" else coupe_amd.Rcb)(case["levels"], case["tol"])
        if kind == "host":
            return dict(kind=kind, algo=algo, points=pts.cpu().numpy(), weights=w.cpu().numpy(),
                        ids=np.zeros(case["n"], dtype=np.uint64))
        return dict(kind=kind, algo=algo, points=pts, weights=w,
                    ids=torch.zeros(case["n"], device=DEV, dtype=torch.int64))
    if kind == "batch":
        inst = _instances(case)
        total = sum(i[0] for i in inst)
        pts = _rand(sum(i[0] * i[1] for i in inst), g)
        box = _rand((len(inst), 6), g)   # each instance in a box of its own
        at = 0
        for q, (n, d, _, _) in enumerate(inst):
            p = pts[at: at + n * d].view(n, d)
            p.mul_(box[q, 3: 3 + d].add(0.1)).add_(box[q, :d])
            at += n * d
        w = torch.floor(_rand(total, g).mul_(16.0)).add_(1.0)
        return dict(kind=kind, instances=inst, points=pts, weights=w,
                    ids=torch.zeros(total, device=DEV, dtype=torch.int64))
    if kind == "serve":
        reqs = []
        for n, levels, resident in _requests(case):
            p, w = _rand((n, 3), g), _weights("whole", n, g)
            if resident:   # moved, and partly re-weighted, since it was stored
                mesh = _Resident(p, w)
                p = p + 0.01 * torch.randn((n, 3), generator=g, device=DEV, dtype=torch.float64)
                w = torch.where(_rand(n, g) < 0.05, _weights("whole", n, g), w)
                reqs.append((levels, mesh, p, w, torch.zeros(n, device=DEV, dtype=torch.int64)))
            else:
                reqs.append((levels, None, p.cpu().pin_memory().numpy(), w.cpu().pin_memory().numpy(),
                             torch.zeros(n, dtype=torch.int64).pin_memory().numpy()))
        return dict(kind=kind, requests=reqs, tol=case["tol"])
    if kind == "grid":
        size = tuple(s for s in (case["nx"], case["ny"], case["nz"]) if s)
        grid = coupe_amd.Grid(size)
        w = _weights(case["weights"], len(grid), g).view(*reversed(size))
        lo = (_rand(len(size), g) * 0.5).tolist()   # cells that cost more, in one region
        w[tuple(slice(int(f * s), int((f + 0.3) * s) + 1) for f, s in zip(lo, w.shape))] *= 4
        return dict(kind=kind, grid=grid, levels=case["levels"], weights=w.view(-1),
                    ids=torch.zeros(len(grid), device=DEV, dtype=torch.int64))
    ids = torch.randint(0, case["parts"], (case["n"],), generator=g, device=DEV, dtype=torch.int64)
    return dict(kind=kind, parts=case["parts"], ids=ids, weights=_weights(case["weights"], case["n"], g))


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(state):
    kind = state["kind"]
    if kind in ("rcb", "rib", "host"):
        state["algo"].partition(state["ids"], (state["points"], state["weights"]))
        return state["ids"]
    if kind == "batch":
        coupe_amd.partition_batch_mixed(state["ids"], state["points"], state["weights"], state["instances"])
        return state["ids"]
    if kind == "serve":
        srv, tickets = _server(), []
        for levels, mesh, p, w, ids in state["requests"]:
            if mesh is None:
                tickets.append(srv.submit(ids, p, w, levels, state["tol"]))
            else:
                mesh.mesh.update(points=p, weights=w)
                tickets.append(srv.submit_mesh(mesh.mesh, ids, levels, state["tol"]))
        for t in tickets:
            srv.wait(t)
        return [r[4] for r in state["requests"]]
    if kind == "grid":
        state["grid"].rcb(state["ids"], state["weights"], state["levels"], threads=16)
        return state["ids"]
    return [imbalance.compute_parts_load(state["ids"], state["parts"], state["weights"]),
            imbalance.imbalance(state["parts"], state["ids"], state["weights"])]


def work(case):
    """Each input read once, each id or load written once; no operations to speak of."""
    kind = case["kind"]
    if kind in ("rcb", "rib", "host"):
        return {"bytes": case["n"] * (8 * case["dim"] + _WBYTES[case["weights"]] + 8), "flops": 0}
    if kind == "batch":
        return {"bytes": sum(n * (8 * d + 16) for n, d, _, _ in _instances(case)), "flops": 0}
    if kind == "serve":
        return {"bytes": sum(n * 40 for n, _, _ in _requests(case)), "flops": 0}
    if kind == "grid":
        cells = case["nx"] * case["ny"] * max(1, case["nz"])
        return {"bytes": cells * (_WBYTES[case["weights"]] + 8), "flops": 0}
    # two calls, each reads the ids and the weights
    return {"bytes": 2 * case["n"] * (8 + _WBYTES[case["weights"]]), "flops": 0}


def exact(case, seed):
    """Loads and imbalance of the same inputs by numpy; ids are whole numbers
    and have no 64-bit value of their own."""
    if case["kind"] != "loads":
        return None
    s = prepare(case, seed)
    ids, w = s["ids"].cpu().numpy(), s["weights"].cpu().numpy()
    # (whole weights: sums far below 2^53, exact in float64)
    loads = np.bincount(ids, weights=w, minlength=case["parts"]).astype(w.dtype)
    total = float(loads.sum(dtype=loads.dtype))   # in the weight type, as the reference sums it
    ideal = total / case["parts"]
    return [loads, float(((loads.astype(np.float64) - ideal) / ideal).max()) if total else 0.0]
