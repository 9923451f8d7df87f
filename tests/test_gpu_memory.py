"""Device memory that has room for the general path's buffers but not for those
of the paths in place beside them: the call runs on the general path, and what
the general path alone cannot have is refused.  The bound is the context's
(COUPE_HIP_MEMORY_LIMIT); ids against the oracle."""
import numpy as np
import pytest

import coupe_amd
from coupe_amd import _native
from tests.test_gpu_hints import path_of

pytestmark = pytest.mark.gpu

N, PIECES, TOL = 1 << 20, 4, 0.01


def _points(rng, cloud):
    return rng.random((N, 3)) if cloud == "uniform" else rng.normal(0, 1, (N, 3)) ** 5


def _call(ctx, pts, w, iters, batch):
    import torch

    out = torch.full((N,), -1, dtype=torch.int64, device="cuda")
    p, ww = torch.from_numpy(pts).cuda(), torch.from_numpy(w).cuda()
    if batch:
        coupe_amd.partition_batch(out, p, ww, [(N // PIECES, iters, TOL)] * PIECES, context=ctx)
    else:
        coupe_amd.Rcb(iters, TOL).partition(out, (p, ww), context=ctx)
    return out.cpu().numpy().astype(np.uint64)


def _check(oracle_mod, got, pts, w, iters, batch, label):
    for q in range(PIECES if batch else 1):
        m = N // PIECES if batch else N
        s = slice(q * m, (q + 1) * m)
        err, exp, _ = oracle_mod.rcb(pts[s], w[s], iters, TOL, parallel=True, nthreads=8)
        assert err == 0
        assert np.array_equal(got[s], exp), f"{label}: piece {q}"


def _general_bytes(monkeypatch, pts, w, calls):
    """What a context holds after the calls on the general path."""
    for name in ("SMALL", "MID", "FRONT"):
        monkeypatch.setenv(f"COUPE_HIP_{name}", "0")
    ctx = coupe_amd.DeviceContext(0)
    for iters, batch in calls:
        _call(ctx, pts, w, iters, batch)
    held = ctx.stats()["device_bytes"]
    ctx.close()
    for name in ("SMALL", "MID", "FRONT"):
        monkeypatch.delenv(f"COUPE_HIP_{name}")
    return held


@pytest.mark.parametrize("cloud", ["uniform", "cluster"])
@pytest.mark.parametrize("calls", [[(8, False)], [(8, True)], [(13, False), (8, False)], [(13, False), (8, True)]],
                         ids=["alone", "batch", "after deep", "batch after deep"])
def test_room_for_the_general_path_only(oracle_mod, monkeypatch, cloud, calls):
    pytest.importorskip("torch")
    rng = np.random.default_rng(len(calls))
    pts, w = _points(rng, cloud), rng.integers(1, 100, N).astype(np.float64)
    limit = _general_bytes(monkeypatch, pts, w, calls) + (1 << 20)
    monkeypatch.setenv("COUPE_HIP_MEMORY_LIMIT", str(limit))
    ctx = coupe_amd.DeviceContext(0)
    try:
        ctx.set_profiling(True)
        for k, (iters, batch) in enumerate(calls + calls[-1:]):
            label = f"{cloud} call {k}: L={iters} batch={batch} limit={limit}"
            print(f"[gpu] {label}", flush=True)
            got = _call(ctx, pts, w, iters, batch)
            _check(oracle_mod, got, pts, w, iters, batch, label)
            st = ctx.stats()
            assert st["device_bytes"] <= limit, st
        if len(calls) == 2 or (cloud == "cluster" and calls[0][1]):   # no room beside the general path's buffers
            assert path_of(ctx) == "general"
            assert st["reruns"] == 0, "a shape that had no room goes there at once"
    finally:
        ctx.close()


def test_no_room_at_all(monkeypatch):
    pytest.importorskip("torch")
    rng = np.random.default_rng(9)
    pts, w = _points(rng, "uniform"), rng.integers(1, 100, N).astype(np.float64)
    monkeypatch.setenv("COUPE_HIP_MEMORY_LIMIT", str(16 << 20))
    ctx = coupe_amd.DeviceContext(0)
    try:
        for batch in (False, True, False):
            print(f"[gpu] no room, batch={batch}", flush=True)
            with pytest.raises(coupe_amd.CoupeError) as e:
                _call(ctx, pts, w, 8, batch)
            assert e.value.code == _native.ALLOC
    finally:
        ctx.close()


def test_what_a_call_that_leaves_the_tree_holds(oracle_mod, monkeypatch):
    """A large call that the midpoint tree gives up holds no gathered points
    beside the general path's buffers; one that it takes gives the oracle's ids
    on the first call, and its gathered points go when other points end elsewhere."""
    torch = pytest.importorskip("torch")
    n, pieces = 1 << 20, 5   # a batch: no frontier
    rng = np.random.default_rng(4)
    held = {}
    clouds = {"cluster": rng.normal(0, 1, (n * pieces, 3)) ** 5, "uniform": rng.random((n * pieces, 3))}
    w = rng.integers(1, 50, n * pieces).astype(np.float64)
    out = torch.zeros(n * pieces, dtype=torch.int64, device="cuda")
    for path in ("general", "default"):
        if path == "general":
            for name in ("SMALL", "MID", "FRONT"):
                monkeypatch.setenv(f"COUPE_HIP_{name}", "0")
        else:
            for name in ("SMALL", "MID", "FRONT"):
                monkeypatch.delenv(f"COUPE_HIP_{name}")
        ctx = coupe_amd.DeviceContext(0)
        ctx.set_profiling(True)
        order = ["cluster", "uniform", "uniform", "cluster"] if path == "default" else ["cluster"]
        for k, cloud in enumerate(order):
            print(f"[gpu] {path} call {k}: {cloud}", flush=True)
            iters = 8 if k == 0 else 7   # another shape after the first call
            out.fill_(-1)
            coupe_amd.partition_batch(out, torch.from_numpy(clouds[cloud]).cuda(), torch.from_numpy(w).cuda(),
                                      [(n, iters, TOL)] * pieces, context=ctx)
            got = out.cpu().numpy().astype(np.uint64)
            for q in range(pieces):
                s = slice(q * n, (q + 1) * n)
                err, exp, _ = oracle_mod.rcb(clouds[cloud][s], w[s], iters, TOL, parallel=True, nthreads=8)
                assert err == 0 and np.array_equal(got[s], exp), f"{path} call {k} {cloud} piece {q}"
            st = ctx.stats()
            held[path, k] = st["device_bytes"] / (n * pieces)
            if path == "default" and cloud == "uniform":
                assert path_of(ctx) == "mid" and st["reruns"] == 0, st
        ctx.close()
    for k in (0, 3):   # cells and tables: 2 bytes a point and a few more
        assert held["default", k] < held["general", 0] + 4, held
