"""Calls whose levels come from one sweep over the tree of box midpoints: ids
against the oracle, on clouds that leave no node open, a few, most, or the
root; sizes at the edges of tiles and of the classes of open nodes; every
weight kind and width; box magnitudes and duplicates that put points on the
midpoints; first and later calls of a shape.  With COUPE_HIP_MID=0 the
frontier takes the single problems (test_gpu_paths.py checks which path runs)."""
import numpy as np
import pytest

import coupe_amd
from coupe_amd import workloads
from tests import cases

pytestmark = pytest.mark.gpu


def _cloud(rng, name, n, dim):
    if name == "uniform":
        return rng.random((n, dim))
    if name == "far":        # few bits of the coordinate left across the box
        return rng.random((n, dim)) * 1e-3 + 1000.0
    if name == "lattice":    # points on the midpoints
        return rng.integers(0, 65, (n, dim)) / 64.0
    if name == "dense":      # half of the points in a small corner: large open nodes
        return np.concatenate([rng.random((n // 2, dim)), rng.random((n - n // 2, dim)) * 0.4])
    return rng.normal(0, 1, (n, dim)) ** 5


def _weights(rng, kind, n):
    if kind == "u16":
        return rng.integers(1, 100, n).astype(np.float64)
    if kind == "int32":
        return rng.integers(1, 1 << 20, n).astype(np.int32)
    if kind == "wrap":
        return rng.integers(2 ** 20, 2 ** 22, n).astype(np.int32)   # sums pass 2^31
    if kind == "int64":
        return rng.integers(2 ** 33, 2 ** 34, n).astype(np.int64)
    if kind == "wide":
        return rng.integers(2 ** 33, 2 ** 34, n).astype(np.float64)
    if kind == "negative":
        return rng.integers(-5, 100, n).astype(np.int64)
    return rng.random(n) * 3.0 + 0.1


def _same(got, exp, w, label):
    if cases.integral(w):
        assert np.array_equal(got, exp), f"{label}: {int(np.count_nonzero(got != exp))} ids differ"
    elif not np.array_equal(got, exp):
        a = np.bincount(got.astype(np.int64), weights=w)
        b = np.bincount(exp.astype(np.int64), weights=w)
        assert a.shape == b.shape, label
        np.testing.assert_allclose(a, b, rtol=1e-12, atol=0, err_msg=label)


CASES = [  # n, cloud, weights, levels, tolerance
    (16385, "uniform", "u16", 12, 0.02), (18432, "uniform", "real", 1, 0.05), (40000, "lattice", "int32", 7, 0.05),
    (65536, "far", "u16", 9, 0.02), (100_003, "uniform", "wide", 8, 0.02), (131_072, "lattice", "negative", 12, 0.3),
    (200_001, "dense", "u16", 6, 0.2), (262_145, "uniform", "int64", 11, 0.01), (300_007, "uniform", "real", 8, 0.02),
    (524_289, "uniform", "wrap", 10, 0.01), (400_000, "cluster", "u16", 9, 0.01), (700_001, "dense", "real", 5, 0.5),
    (1_000_003, "uniform", "u16", 12, 0.005), (50_000, "uniform", "u16", 5, 0.0), (33_000, "far", "int64", 3, 1.5),
]


@pytest.mark.parametrize("mid", ["1", "0"])
@pytest.mark.parametrize("dim", [2, 3])
def test_midpoint_tree_alone(oracle_mod, monkeypatch, dim, mid):
    torch = pytest.importorskip("torch")
    monkeypatch.setenv("COUPE_HIP_MID", mid)
    ctx = coupe_amd.DeviceContext(0)
    try:
        for q, (n, cloud, kind, iters, tol) in enumerate(CASES):
            rng = np.random.default_rng(7000 + 10 * q + dim)
            for call in range(2):   # the second call of a shape: other points
                label = f"n={n} d={dim} {cloud} {kind} L={iters} tol={tol} call {call}"
                print(f"[gpu] mid {mid}: {label}", flush=True)
                pts, w = _cloud(rng, cloud, n, dim), _weights(rng, kind, n)
                out = torch.full((n,), -1, dtype=torch.int64, device="cuda")
                coupe_amd.Rcb(iters, tol).partition(
                    out, (torch.from_numpy(pts).cuda(), torch.from_numpy(w).cuda()), context=ctx)
                err, exp, _ = oracle_mod.rcb(pts, w, iters, tol, parallel=True, nthreads=8)
                assert err == 0
                _same(out.cpu().numpy().astype(np.uint64), exp, w, label)
    finally:
        ctx.close()


@pytest.mark.parametrize("dim", [2, 3])
def test_midpoint_tree_in_a_batch(oracle_mod, dim):
    torch = pytest.importorskip("torch")
    rng = np.random.default_rng(50 + dim)
    specs = [(int(n), int(rng.integers(0, 13)), float(rng.choice([0.01, 0.02, 0.05])))
             for n in rng.permutation([16385, 20000, 300, 0, 100_001, 70_000, 2048, 30_000, 45_001, 250_000, 1, 17_000])]
    pts = np.concatenate([_cloud(rng, ["uniform", "lattice", "far", "uniform"][q % 4], n, dim) * (q + 1)
                          for q, (n, _, _) in enumerate(specs)])
    w = rng.integers(1, 50, pts.shape[0]).astype(np.float64)
    out = torch.full((pts.shape[0],), -1, dtype=torch.int64, device="cuda")
    for call in range(2):
        print(f"[gpu] midpoint tree, batch, dim {dim}, call {call}", flush=True)
        out.fill_(-1)
        coupe_amd.partition_batch(out, torch.from_numpy(pts).cuda(), torch.from_numpy(w).cuda(), specs)
        got, off = out.cpu().numpy().astype(np.uint64), 0
        for q, (n, iters, tol) in enumerate(specs):
            _, exp, _ = oracle_mod.rcb(pts[off:off + n], w[off:off + n], iters, tol)
            _same(got[off:off + n], exp, w[off:off + n], f"call {call} problem {q}: n={n} L={iters} tol={tol}")
            off += n


def test_grids_and_other_points_of_a_shape(oracle_mod):
    """A shape's calls alternate between points the tree settles, points that
    leave nodes open and points whose root search goes on (frontier)."""
    torch = pytest.importorskip("torch")
    pts, w = workloads.jgrid(48, 2, True)
    n = len(w)
    rng = np.random.default_rng(8)
    ctx = coupe_amd.DeviceContext(0)
    try:
        for call, p in enumerate([pts, pts, rng.random((n, 3)), pts, rng.normal(0, 1, (n, 3)) ** 5, pts, pts]):
            print(f"[gpu] alternating points, call {call}", flush=True)
            ww = np.ones(n) if call == 1 else w
            out = torch.full((n,), -1, dtype=torch.int64, device="cuda")
            coupe_amd.Rcb(9, 0.02).partition(out, (torch.from_numpy(p).cuda(), torch.from_numpy(ww).cuda()), context=ctx)
            _, exp, _ = oracle_mod.rcb(p, ww, 9, 0.02)
            _same(out.cpu().numpy().astype(np.uint64), exp, ww, f"call {call}")
    finally:
        ctx.close()
