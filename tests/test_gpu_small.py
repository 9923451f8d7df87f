"""Problems of few points, one workgroup each: ids against the oracle where
the kernel can go wrong -- the edges of its three shapes (2048, 8192 and
16384 points), the largest depth it takes and the next one, duplicated
points, clusters, empty leftmost parts, every weight kind -- alone and in
batches beside problems of the general path.  Integer and integer-valued
weights: ids bit for bit; others by per-part weights to 1e-12 relative."""
import numpy as np
import pytest

import coupe_amd
from tests import cases

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 63, 64, 65, 255, 257, 2047, 2048, 2049, 8191, 8192, 8193, 16383, 16384, 16385]
CLOUDS = ["uniform", "cluster", "dup", "wide", "equal"]
KINDS = ["u16", "int32", "negative", "wide", "real", "zero"]


def _cloud(rng, name, n, dim):
    if name == "uniform":
        return rng.random((n, dim))
    if name == "cluster":
        return rng.normal(0, 1, (n, dim)) ** 5
    if name == "dup":
        return rng.integers(0, 6, (n, dim)).astype(np.float64)
    if name == "wide":
        return rng.normal(0, 1, (n, dim)) * 10.0 ** rng.integers(-30, 30, (n, dim))
    return np.tile(rng.random(dim), (n, 1))


def _weights(rng, kind, n):
    if kind == "u16":
        return rng.integers(0, 65536, n).astype(np.float64)
    if kind == "int32":
        return rng.integers(2 ** 28, 2 ** 31 - 1, n).astype(np.int32)   # their sums wrap
    if kind == "negative":
        return rng.integers(-50, 50, n).astype(np.int64)
    if kind == "wide":
        return rng.integers(2 ** 40, 2 ** 41, n).astype(np.int64)
    if kind == "real":
        return rng.random(n) * 3.0 + 0.1
    return np.zeros(n)


def _same(got, exp, w, label):
    if cases.integral(w):
        assert np.array_equal(got, exp), f"{label}: {int(np.count_nonzero(got != exp))} ids differ"
    elif not np.array_equal(got, exp):
        a = np.bincount(got.astype(np.int64), weights=w)
        b = np.bincount(exp.astype(np.int64), weights=w)
        assert a.shape == b.shape, label
        np.testing.assert_allclose(a, b, rtol=1e-12, atol=0, err_msg=label)


@pytest.mark.parametrize("small", ["1", "0"])
@pytest.mark.parametrize("dim", [2, 3])
def test_small_problems_alone(oracle_mod, monkeypatch, dim, small):
    torch = pytest.importorskip("torch")
    monkeypatch.setenv("COUPE_HIP_SMALL", small)
    ctx = coupe_amd.DeviceContext(0)
    try:
        for q, n in enumerate(SIZES):
            for r, cloud in enumerate(CLOUDS):
                rng = np.random.default_rng(1000 * dim + 10 * q + r)
                kind = KINDS[(q + r) % len(KINDS)]
                iters = [3, 8, 11, 12, 13, 0, 1][(q + 2 * r) % 7]
                tol = [0.0, 0.01, 0.05, -1.0][(q + r) % 4]
                label = f"n={n} d={dim} {cloud} {kind} L={iters} tol={tol}"
                print(f"[gpu] small {small}: {label}", flush=True)
                pts, w = _cloud(rng, cloud, n, dim), _weights(rng, kind, n)
                out = torch.full((n,), -1, dtype=torch.int64, device="cuda")
                coupe_amd.Rcb(iters, tol).partition(
                    out, (torch.from_numpy(pts).cuda(), torch.from_numpy(w).cuda()), context=ctx)
                err, exp, _ = oracle_mod.rcb(pts, w, iters, tol)
                assert err == 0
                _same(out.cpu().numpy().astype(np.uint64), exp, w, label)
    finally:
        ctx.close()


@pytest.mark.parametrize("dim", [2, 3])
def test_small_problems_in_a_batch(oracle_mod, dim):
    torch = pytest.importorskip("torch")
    rng = np.random.default_rng(40 + dim)
    sizes = rng.permutation(np.array(SIZES + [0, 30000, 50001, 700, 5000, 12000, 0]))
    specs = [(int(n), int(rng.integers(0, 14)), float(rng.choice([0.0, 0.02]))) for n in sizes]
    pts = np.concatenate([_cloud(rng, CLOUDS[q % 3], n, dim) for q, (n, _, _) in enumerate(specs)])
    w = rng.integers(1, 50, pts.shape[0]).astype(np.float64)
    out = torch.full((pts.shape[0],), -1, dtype=torch.int64, device="cuda")
    print(f"[gpu] batch of {len(specs)} problems, dim {dim}", flush=True)
    for call in range(2):
        out.fill_(-1)
        coupe_amd.partition_batch(out, torch.from_numpy(pts).cuda(), torch.from_numpy(w).cuda(), specs)
        got, off = out.cpu().numpy().astype(np.uint64), 0
        for q, (n, iters, tol) in enumerate(specs):
            _, exp, _ = oracle_mod.rcb(pts[off:off + n], w[off:off + n], iters, tol)
            _same(got[off:off + n], exp, w[off:off + n], f"call {call} problem {q}: n={n} L={iters} tol={tol}")
            off += n
