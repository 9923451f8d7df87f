"""Coordinates near the ends of f32's range, where a window's extent, the sum of
its ends or the reciprocal of its extent leaves f32, and infinite ones: ids
against the oracle on every path (one workgroup, midpoint tree, frontier).
NaN coordinates go left at every split: ids as on the general path."""
import numpy as np
import pytest

import coupe_amd
from tests.test_gpu_mid import _same, _weights

pytestmark = pytest.mark.gpu


def _cloud(rng, name, n, dim):
    kind, _, size = name.partition(" ")
    s = float(size or 0)
    r = rng.random((n, dim))
    if kind == "both":       # from -s to s
        return (2.0 * r - 1.0) * s
    if kind == "positive":   # from 0 to s
        return r * s
    if kind == "high":       # from s / 2 to s: sums of two leave f32 first
        return (1.0 + r) * (0.5 * s)
    if kind == "outliers":   # a cloud of size 1, a few points at s
        return np.where(rng.random((n, dim)) < 0.01, s * np.sign(r - 0.5), r)
    value = {"inf": np.inf, "-inf": -np.inf, "nan": np.nan}.get(kind)
    if value is None:        # "infs": both infinities
        value = np.where(r < 0.5, -np.inf, np.inf)
    return np.where(rng.random((n, dim)) < 0.01, value, rng.normal(0, 1, (n, dim)) ** 3)


CLOUDS = [f"{kind} {s}" for kind in ("both", "positive", "high", "outliers") for s in ("2e37", "5e37", "1e38", "3e38")]
CLOUDS += ["both 1.6e38", "both 1.8e38", "inf", "-inf", "infs"]
KINDS = ["u16", "real", "int32", "int64", "negative", "wide"]


def _partition(ctx, pts, w, iters, tol):
    import torch

    out = torch.full((len(w),), -1, dtype=torch.int64, device="cuda")
    coupe_amd.Rcb(iters, tol).partition(out, (torch.from_numpy(pts).cuda(), torch.from_numpy(w).cuda()), context=ctx)
    return out.cpu().numpy().astype(np.uint64)


@pytest.mark.parametrize("mid", ["1", "0"])
@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("n", [1000, 12_000, 50_001, 200_000, 2_000_000])
def test_wide_boxes(oracle_mod, monkeypatch, n, dim, mid):
    pytest.importorskip("torch")
    monkeypatch.setenv("COUPE_HIP_MID", mid)
    if n <= 16384 and mid == "0":
        pytest.skip("one workgroup either way")
    clouds = CLOUDS if n < 1_000_000 else ["both 5e37", "both 3e38", "positive 1e38", "high 3e38", "infs"]
    ctx = coupe_amd.DeviceContext(0)
    try:
        for q, cloud in enumerate(clouds):
            rng = np.random.default_rng(100 * q + dim)
            pts, w = _cloud(rng, cloud, n, dim), _weights(rng, KINDS[(q + dim) % len(KINDS)], n)
            iters, tol = [4, 7, 9][q % 3], [0.01, 0.05][q % 2]
            label = f"n={n} d={dim} mid {mid} {cloud} {KINDS[(q + dim) % len(KINDS)]} L={iters} tol={tol}"
            print(f"[gpu] {label}", flush=True)
            got = _partition(ctx, pts, w, iters, tol)
            err, exp, _ = oracle_mod.rcb(pts, w, iters, tol, parallel=True, nthreads=8)
            assert err == 0
            _same(got, exp, w, label)
    finally:
        ctx.close()


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("n", [1000, 12_000, 50_001, 200_000])
def test_nan_coordinates(monkeypatch, n, dim):
    pytest.importorskip("torch")
    rng = np.random.default_rng(n + dim)
    pts, w = _cloud(rng, "nan", n, dim), _weights(rng, "u16", n)
    ids = {}
    for path in ("default", "general"):
        if path == "general":
            for name in ("COUPE_HIP_SMALL", "COUPE_HIP_MID", "COUPE_HIP_FRONT"):
                monkeypatch.setenv(name, "0")
        ctx = coupe_amd.DeviceContext(0)
        try:
            print(f"[gpu] nan n={n} d={dim} {path}", flush=True)
            ids[path] = _partition(ctx, pts, w, 7, 0.02)
        finally:
            ctx.close()
    assert np.array_equal(ids["default"], ids["general"])
