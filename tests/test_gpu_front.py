"""Calls of one instance whose searches run on the frontier (points not moved):
ids against the oracle, on clouds whose splits lie away from the middle of
their box, with few and many points per part, duplicates, coordinates over many
magnitudes (long searches: the rounds queued ahead run out), every weight kind,
first and later calls of a shape; with COUPE_HIP_FRONT=0 the general path takes
what the midpoint tree, tried first, leaves."""
import numpy as np
import pytest

import coupe_amd
from tests import cases
from tests.test_gpu_mid import _same, _weights

pytestmark = pytest.mark.gpu


def _cloud(rng, name, n, dim):
    if name == "cluster":
        return rng.normal(0, 1, (n, dim)) ** 5
    if name == "graded":
        return rng.random((n, dim)) ** 3
    if name == "dup":
        return rng.integers(0, 40, (n, dim)) ** 3.0
    if name == "wide":
        return rng.normal(0, 1, (n, dim)) * 10.0 ** rng.integers(-30, 30, (n, dim))
    return np.concatenate([np.tile(rng.random(dim), (n // 2, 1)), rng.random((n - n // 2, dim)) ** 2])   # half equal


CASES = [  # n, cloud, weights, levels, tolerance
    (40_001, "cluster", "u16", 9, 0.01), (65_536, "graded", "real", 12, 0.0), (100_003, "dup", "int32", 10, 0.01),
    (131_073, "wide", "u16", 8, 0.01), (262_144, "half", "int64", 7, 0.02), (300_000, "graded", "wrap", 1, 0.01),
    (524_287, "cluster", "negative", 11, 0.05), (700_000, "graded", "u16", 12, 0.001), (90_000, "wide", "real", 5, 0.0),
    (1_200_001, "cluster", "wide", 8, 0.01), (9_000_000, "graded", "u16", 12, 0.01),
]


@pytest.mark.parametrize("front", ["1", "0"])
@pytest.mark.parametrize("dim", [2, 3])
def test_frontier_alone(oracle_mod, monkeypatch, dim, front):
    torch = pytest.importorskip("torch")
    monkeypatch.setenv("COUPE_HIP_FRONT", front)
    ctx = coupe_amd.DeviceContext(0)
    try:
        for q, (n, cloud, kind, iters, tol) in enumerate(CASES):
            rng = np.random.default_rng(9000 + 10 * q + dim)
            for call in range(2 if n < 1_000_000 else 1):   # the second call of a shape: other points
                label = f"n={n} d={dim} {cloud} {kind} L={iters} tol={tol} call {call}"
                print(f"[gpu] front {front}: {label}", flush=True)
                pts, w = _cloud(rng, cloud, n, dim), _weights(rng, kind, n)
                out = torch.full((n,), -1, dtype=torch.int64, device="cuda")
                coupe_amd.Rcb(iters, tol).partition(
                    out, (torch.from_numpy(pts).cuda(), torch.from_numpy(w).cuda()), context=ctx)
                err, exp, _ = oracle_mod.rcb(pts, w, iters, tol, parallel=True, nthreads=8)
                assert err == 0
                _same(out.cpu().numpy().astype(np.uint64), exp, w, label)
    finally:
        ctx.close()


def test_easy_and_hard_points_of_a_shape(oracle_mod):
    """A shape's calls alternate: the midpoint tree, long searches (more rounds
    than the last call took), the frontier again."""
    torch = pytest.importorskip("torch")
    n = 120_000
    rng = np.random.default_rng(12)
    ctx = coupe_amd.DeviceContext(0)
    try:
        w = rng.integers(1, 50, n).astype(np.float64)
        kinds = ["graded", "wide", "graded", "uniform", "uniform", "half", "wide"]
        for call, kind in enumerate(kinds):
            print(f"[gpu] easy and hard points, call {call}: {kind}", flush=True)
            p = rng.random((n, 3)) if kind == "uniform" else _cloud(rng, kind, n, 3)
            out = torch.full((n,), -1, dtype=torch.int64, device="cuda")
            coupe_amd.Rcb(6, 0.01).partition(out, (torch.from_numpy(p).cuda(), torch.from_numpy(w).cuda()), context=ctx)
            _, exp, _ = oracle_mod.rcb(p, w, 6, 0.01)
            _same(out.cpu().numpy().astype(np.uint64), exp, w, f"call {call}")
    finally:
        ctx.close()
