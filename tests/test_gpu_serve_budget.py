"""A server's device memory stays within its budget whichever paths its batches
take: ids against the oracle, the accounted peak against the budget."""
import numpy as np
import pytest

import coupe_amd

pytestmark = pytest.mark.gpu


def _same(oracle_mod, out, pts, w, iters, tol, label):
    err, exp, _ = oracle_mod.rcb(pts, w, iters, tol)
    assert err == 0
    assert np.array_equal(out, exp), f"{label}: {int(np.count_nonzero(out != exp))} ids differ"


def test_one_larger_request_among_small_ones(oracle_mod):
    """The small requests of a batch run as one workgroup each; the larger one
    is then alone, and the frontier's bins are more than this budget has."""
    torch = pytest.importorskip("torch")
    rng = np.random.default_rng(5)
    budget = 28 << 20
    srv = coupe_amd.Server(slots=1, memory_budget=budget, max_batch_requests=16)
    sizes = (5000, 3000, 100_000, 700, 12_000, 16_000)
    data = [(np.zeros(n, dtype=np.uint64), rng.normal(0, 1, (n, 3)) ** 5, rng.integers(1, 50, n).astype(np.float64))
            for n in sizes]
    try:
        # a request whose points are ready late, so that the others queue up
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            torch.cuda._sleep(400_000_000)
            pts = torch.rand((1000, 3), device="cuda", dtype=torch.float64)
            first = srv.submit(torch.zeros(1000, dtype=torch.int64, device="cuda"), pts,
                               torch.ones(1000, device="cuda", dtype=torch.float64), 3, 0.05)
        reqs = [(srv.submit(out, p, w, 8, 0.01), out, p, w) for out, p, w in data]
        srv.wait(first)
        for t, out, p, w in reqs:
            st = srv.wait(t)
            assert st["batch_requests"] == len(reqs), st
            _same(oracle_mod, out, p, w, 8, 0.01, f"n={len(w)}")
        st = srv.stats()
        assert st["peak_device_bytes"] <= budget, st
    finally:
        srv.close()


def test_buffers_of_both_kinds_of_paths(oracle_mod):
    """A batch in place, then, with a mesh created meanwhile, one for which
    only the general path's buffers have room: those of the first are given back."""
    rng = np.random.default_rng(6)
    budget, n, iters = 420_000_000, 2_000_000, 10
    srv = coupe_amd.Server(slots=1, memory_budget=budget)
    try:
        # (the frontier: its bins are held too)
        pts, w, out = rng.normal(0, 1, (n, 3)) ** 5, rng.integers(1, 100, n).astype(np.float64), np.zeros(n, dtype=np.uint64)
        for call in range(3):
            srv.wait(srv.submit(out, pts, w, iters, 0.05))
            _same(oracle_mod, out, pts, w, iters, 0.05, f"call {call}")
            st = srv.stats()
            assert st["peak_device_bytes"] <= budget, st
            if call == 0:   # 28 bytes a point
                mesh = srv.create_mesh(rng.random((6_857_000, 3)), np.ones(6_857_000))
        mesh.destroy()
        srv.wait(srv.submit(out, pts, w, iters, 0.05))
        _same(oracle_mod, out, pts, w, iters, 0.05, "after the mesh")
        assert srv.stats()["peak_device_bytes"] <= budget
    finally:
        srv.close()
