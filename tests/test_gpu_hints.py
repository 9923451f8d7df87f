"""What a context keeps of a shape's last call must not show in the next one's
ids: weights of another type or kind on the same points, with calls of other
shapes between.  Ids against the oracle."""
import numpy as np
import pytest

import coupe_amd
from tests.test_gpu_mid import _same

pytestmark = pytest.mark.gpu


def _weights(rng, kind, n):
    if kind == "unit":
        return np.ones(n)
    if kind == "real":
        return rng.random(n) * 3.0 + 0.1
    if kind == "whole":
        return rng.integers(1, 100, n).astype(np.float64)
    if kind == "int32":
        return rng.integers(1, 1 << 20, n).astype(np.int32)
    return rng.integers(2 ** 33, 2 ** 34, n).astype(np.int64)


def _call(oracle_mod, ctx, pts, w, iters, tol, label):
    import torch

    print(f"[gpu] {label}", flush=True)
    out = torch.full((len(w),), -1, dtype=torch.int64, device="cuda")
    coupe_amd.Rcb(iters, tol).partition(out, (torch.from_numpy(pts).cuda(), torch.from_numpy(w).cuda()), context=ctx)
    err, exp, _ = oracle_mod.rcb(pts, w, iters, tol, parallel=True, nthreads=8)
    assert err == 0
    _same(out.cpu().numpy().astype(np.uint64), exp, w, label)


# (shape, weights) in call order; shape A takes the paths that leave the points
# in place, B another size of them, S one workgroup, G the general path
ORDERS = [
    "A real, B whole, A int64, A int32, A real, B int64, A int32",
    "A real, S whole, A int64, B real, G real, A int32",
    "A real, G int64, A int64, G real, B int32, G int64, A whole",
    "G real, A unit, G int32, G real, S real, G int64",
]


@pytest.mark.parametrize("graphs", ["0", "1"])
@pytest.mark.parametrize("order", ORDERS)
def test_weights_of_another_type_between_other_shapes(oracle_mod, monkeypatch, order, graphs):
    pytest.importorskip("torch")
    monkeypatch.setenv("COUPE_HIP_GRAPHS", graphs)
    sizes = {"A": (40_000, 6), "B": (65_537, 7), "S": (5000, 5), "G": (30_000, 13)}
    rng = np.random.default_rng(3)
    ctx = coupe_amd.DeviceContext(0)
    try:
        for k, call in enumerate(order.split(", ")):
            shape, kind = call.split()
            n, iters = sizes[shape]
            _call(oracle_mod, ctx, rng.random((n, 3)), _weights(rng, kind, n), iters, 0.02,
                  f"graphs {graphs}, {order}: call {k} {call}")
    finally:
        ctx.close()


def path_of(ctx):
    """The path of the context's last call (profiling enabled)."""
    t = ctx.kernel_times()
    if t["prologue"]["launches"] == 0:
        return "small"
    if t["partition"]["algo_bytes"] > 0:
        return "general"
    return "mid" if t["decide"]["launches"] == 1 else "front"


@pytest.mark.parametrize("n", [50_000, 400_000])
@pytest.mark.parametrize("kinds", ["unit real real", "whole real real", "real whole real", "unit int64 real", "int64 real unit"])
def test_a_change_of_weights_leaves_the_shape_its_path(oracle_mod, n, kinds):
    """Points that split at the midpoints: a call whose expected weight mode
    does not hold runs again, and neither it nor the next one ends on another path."""
    pytest.importorskip("torch")
    rng = np.random.default_rng(n)
    iters, tol = 8, 0.25
    ctx = coupe_amd.DeviceContext(0)
    try:
        ctx.set_profiling(True)
        for k, kind in enumerate(kinds.split()):
            for again in range(2):
                _call(oracle_mod, ctx, rng.random((n, 3)), _weights(rng, kind, n), iters, tol,
                      f"n={n} {kinds}: call {k}.{again} {kind}")
                st = ctx.stats()
                assert st["passes"] == iters, st
                if again:
                    assert path_of(ctx) == "mid", ctx.kernel_times()
    finally:
        ctx.close()
