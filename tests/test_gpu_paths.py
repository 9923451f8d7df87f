"""Which path a call takes: switches of the general path count where they differ
from their defaults (those of its parts wherever they are set), and each path
gives the oracle's ids where it is the one that runs."""
import numpy as np
import pytest

import coupe_amd
from tests import cases
from tests.test_gpu_hints import path_of
from tests.test_gpu_mid import _same

pytestmark = pytest.mark.gpu

PARTS = ("PAIRS", "FORWARD", "FULL_FIRST")
DEFAULTS = {"PAIRS": "1", "FORWARD": "1", "FULL_FIRST": "1", "BIN_COPIES": "256", "MOVE_NT_BYTES": "2.5e9",
            "SEARCH_CHUNK": "2", "GRAPHS": "0", "BINS": "256", "WG_PER_CU": "0", "SCAN_DIRECT": "2048",
            "SEARCH_PASSES": "3"}
OTHERS = {"PAIRS": "0", "FORWARD": "0", "FULL_FIRST": "0", "BIN_COPIES": "0", "MOVE_NT_BYTES": "0", "SEARCH_CHUNK": "1",
          "GRAPHS": "1", "BINS": "64", "WG_PER_CU": "2", "SCAN_DIRECT": "64", "SEARCH_PASSES": "2"}


def _call(oracle_mod, ctx, pts, w, iters, tol, label):
    import torch

    print(f"[gpu] {label}", flush=True)
    out = torch.full((len(w),), -1, dtype=torch.int64, device="cuda")
    coupe_amd.Rcb(iters, tol).partition(out, (torch.from_numpy(pts).cuda(), torch.from_numpy(w).cuda()), context=ctx)
    err, exp, _ = oracle_mod.rcb(pts, w, iters, tol, parallel=True, nthreads=8)
    assert err == 0
    _same(out.cpu().numpy().astype(np.uint64), exp, w, label)
    return path_of(ctx)


@pytest.mark.parametrize("name", sorted(DEFAULTS))
def test_switches_at_and_off_their_defaults(oracle_mod, monkeypatch, name):
    pytest.importorskip("torch")
    rng = np.random.default_rng(2)
    in_place, general = ("small", "mid"), ("general", "general")
    for value, expect in ((DEFAULTS[name], general if name in PARTS else in_place), ("", in_place),
                          (OTHERS[name], general)):
        monkeypatch.setenv(f"COUPE_HIP_{name}", value)
        ctx = coupe_amd.DeviceContext(0)
        try:
            ctx.set_profiling(True)
            for n, path in zip((5000, 60_000), expect):
                got = _call(oracle_mod, ctx, rng.random((n, 3)), rng.integers(1, 50, n).astype(np.float64), 6, 0.2,
                            f"{name}={value!r} n={n}")
                assert got == path, f"{name}={value!r} n={n}: {got}"
        finally:
            ctx.close()


@pytest.mark.parametrize("path", ["default", "front", "general"])
@pytest.mark.parametrize("seed", range(3))
def test_each_path_where_it_runs(oracle_mod, monkeypatch, path, seed):
    """Clouds for every path; with the tree off the frontier takes them, with
    both (and the small problems) off the general path."""
    pytest.importorskip("torch")
    if path != "default":
        for name in ("SMALL", "MID") + (("FRONT",) if path == "general" else ()):
            monkeypatch.setenv(f"COUPE_HIP_{name}", "0")
    rng = np.random.default_rng(seed)
    ctx = coupe_amd.DeviceContext(0)
    try:
        ctx.set_profiling(True)
        for n, dim, expect in ((3000, 3, "small"), (70_001, 2, "mid"), (300_000, 3, "mid"), (120_000, 3, "front")):
            even = expect != "front"
            pts = rng.random((n, dim)) if even else rng.normal(0, 1, (n, dim)) ** 5
            w = rng.integers(1, 50, n).astype([np.float64, np.int32, np.int64][seed])
            for call in range(2):
                got = _call(oracle_mod, ctx, pts, w, 7, 0.05 if even else 0.01, f"{path} n={n} d={dim} call {call}")
                assert got == (expect if path == "default" else path), got
    finally:
        ctx.close()


@pytest.mark.parametrize("seed", range(40))
def test_general_path_on_small_cases(oracle_mod, monkeypatch, seed):
    """The general path on inputs the one-workgroup kernel takes by default."""
    pytest.importorskip("torch")
    for name in ("SMALL", "MID", "FRONT"):
        monkeypatch.setenv(f"COUPE_HIP_{name}", "0")
    pts, w, iters, tol = cases.random_case(700 + seed, 3000)
    ctx = coupe_amd.DeviceContext(0)
    try:
        _call(oracle_mod, ctx, pts, w, iters, tol, f"seed {seed}")
    finally:
        ctx.close()


def test_new_shapes_after_misses_of_the_midpoint_tree(oracle_mod):
    """Batches of another shape each call whose roots do not split at the
    midpoints: after three the tree is passed by for 2, then 4 new shapes; a
    batch that splits there brings it back."""
    torch = pytest.importorskip("torch")
    rng = np.random.default_rng(14)
    pieces, tol = 4, 0.25
    ctx = coupe_amd.DeviceContext(0)
    try:
        ctx.set_profiling(True)
        # (cloud, path, whether the tree was tried and left the call)
        calls = [("skew", "general", t) for t in (1, 1, 1, 0, 0, 1, 0, 0)]
        calls += [("even", "general", 0), ("even", "mid", 0), ("skew", "general", 1), ("even", "mid", 0)]
        for k, (cloud, path, tried) in enumerate(calls):
            n = 100_000 + k
            print(f"[gpu] new shapes, call {k}: {cloud}", flush=True)
            pts = rng.random((n * pieces, 3))
            if cloud == "skew":
                pts = pts ** 3
            w = rng.integers(1, 50, n * pieces).astype(np.float64)
            out = torch.zeros(n * pieces, dtype=torch.int64, device="cuda")
            coupe_amd.partition_batch(out, torch.from_numpy(pts).cuda(), torch.from_numpy(w).cuda(),
                                      [(n, 8, tol)] * pieces, context=ctx)
            got = out.cpu().numpy().astype(np.uint64)
            for q in range(pieces):
                s = slice(q * n, (q + 1) * n)
                err, exp, _ = oracle_mod.rcb(pts[s], w[s], 8, tol, parallel=True, nthreads=8)
                assert err == 0 and np.array_equal(got[s], exp), f"call {k} piece {q}"
            assert path_of(ctx) == path, f"call {k}: {ctx.kernel_times()}"
            assert ctx.stats()["reruns"] == tried, f"call {k}: {ctx.stats()}"
    finally:
        ctx.close()


def test_autotuner_leaves_what_the_call_does_not_read(oracle_mod):
    """A batch that the midpoint tree and the one-workgroup kernel take whole
    does not read the general path's bins, first pass and chunks: the tuner
    keeps them (graphs, which would take that path, must win to be chosen)."""
    torch = pytest.importorskip("torch")
    rng = np.random.default_rng(31)
    specs = [(n, 3, 6, 0.2) for n in (30_000, 60_000, 5000, 90_000)]
    total = sum(s[0] for s in specs)
    pts, w = rng.random(total * 3), rng.integers(1, 50, total).astype(np.float64)
    out = torch.full((total,), -1, dtype=torch.int64, device="cuda")
    ctx = coupe_amd.DeviceContext(0)
    try:
        print("[gpu] autotune of a batch in place", flush=True)
        for trial in range(3):
            chosen = coupe_amd.autotune(out, torch.from_numpy(pts).cuda(), torch.from_numpy(w).cuda(), specs, trials=1,
                                        context=ctx)
            if not chosen["graphs"]:
                assert (chosen["bins"], chosen["full_first"], chosen["search_chunk"]) == (256, 1, 2), chosen
        got, off = out.cpu().numpy().astype(np.uint64), 0
        for n, d, iters, tol in specs:
            err, exp, _ = oracle_mod.rcb(pts[off * 3:(off + n) * 3].reshape(n, 3), w[off:off + n], iters, tol)
            assert err == 0 and np.array_equal(got[off:off + n], exp)
            off += n
    finally:
        ctx.close()


@pytest.mark.parametrize("cloud", ["lognormal", "clusters", "changing"])
def test_long_searches_of_large_calls(oracle_mod, cloud):
    """More than 2^22 points off the midpoints: a shape whose frontier took many
    rounds goes to the general path, unless its searches run out there twice;
    other shapes stay on the frontier."""
    torch = pytest.importorskip("torch")
    n, iters, tol = (1 << 22) + 5, 8, 0.01
    rng = np.random.default_rng(21)
    w = rng.integers(1, 50, n).astype(np.float64)
    ctx = coupe_amd.DeviceContext(0)
    try:
        ctx.set_profiling(True)
        paths, reruns = [], []
        for call in range(3 if cloud != "changing" else 5):
            if cloud == "clusters":
                pts = rng.random((8, 3))[rng.integers(0, 8, n)] + 0.05 * rng.normal(0, 1, (n, 3))
            elif cloud == "lognormal":
                pts = np.exp(2.0 * np.random.default_rng(5).normal(0, 1, (n, 3)))
            else:   # windows of other extents each call
                pts = np.tan(np.pi * (rng.random((n, 3)) - 0.5)) * 10.0 ** (3 * call)
            label = f"{cloud} call {call}"
            paths.append(_call(oracle_mod, ctx, pts, w, iters, tol, label))
            st = ctx.stats()
            reruns.append(st["reruns"])
            print(f"[gpu] {label}: {paths[-1]}, {st['passes']} passes, reruns {reruns[-1]}", flush=True)
        if cloud == "clusters":
            assert paths == ["front"] * 3
        elif cloud == "lognormal":
            assert paths == ["front", "general", "general"]
        else:
            assert paths[:2] == ["front", "general"]
            for k in range(2, len(paths)):
                assert paths[k] == ("front" if sum(reruns[1:k]) >= 2 else "general"), (paths, reruns)
    finally:
        ctx.close()
