"""2D grids by strips (COUPE_HIP_GRID_STRIPS=1 sends every 2D call of up to 20
levels there) against the oracle, id for id: sizes around a band of rows and
a group of columns (16), their partial scans (64 rows, 512 columns) and the
workgroup's step along an axis (256 cross-sections); subgrids of a few cells and
empty ones; more subgrids than CUs; weights at one cell, zero, negative.  Axes
of more than one step a chunk: test_gpu_strips_long.py."""
import numpy as np
import pytest

from tests.test_gpu_grid import gpu_grid, say

pytestmark = pytest.mark.gpu

SIZES = [([1, 1], 3), ([15, 17], 6), ([16, 16], 8), ([17, 31], 9), ([33, 48], 12), ([511, 9], 7), ([513, 40], 10),
         ([2048, 24], 9), ([24, 2049], 9), ([4097, 65], 11), ([70, 8193], 12), ([9001, 130], 10), ([1, 4100], 6),
         ([5000, 1], 6), ([700, 640], 14)]


@pytest.mark.parametrize("size,iters", SIZES)
@pytest.mark.parametrize("kind", ["i32", "i64", "f64int"])
def test_strips(oracle_mod, monkeypatch, size, iters, kind):
    monkeypatch.setenv("COUPE_HIP_GRID_STRIPS", "1")
    rng = np.random.default_rng(size[0] * 7 + size[1] + iters)
    n = size[0] * size[1]
    if kind == "i32":
        w = rng.integers(-5, 1000, n).astype(np.int32)
    elif kind == "i64":
        w = rng.integers(0, 1 << 40, n).astype(np.int64)
    else:
        w = rng.integers(0, 100, n).astype(np.float64)
    threads = 3 + size[0] % 40
    say(f"strips {size} {kind} L={iters} threads={threads}")
    assert np.array_equal(gpu_grid(size, w, iters, threads), oracle_mod.grid_rcb(size, w, iters, threads=threads))


@pytest.mark.parametrize("where", ["corner", "middle", "none", "quarter", "wrap"])
def test_strips_odd_weights(oracle_mod, monkeypatch, where):
    """One heavy cell, no weight at all, quarter weights (handed to the
    per-level path), sums that wrap in i32."""
    monkeypatch.setenv("COUPE_HIP_GRID_STRIPS", "1")
    size, iters = [300, 210], 10
    n = size[0] * size[1]
    w = np.zeros(n)
    if where == "corner":
        w[-1] = 1e6
    elif where == "middle":
        w += 1.0
        w[n // 2 + 150] = 1e9
    elif where == "quarter":
        w = np.random.default_rng(5).integers(0, 400, n) / 4.0
    elif where == "wrap":
        w = np.full(n, 1 << 20, dtype=np.int32)
    say(f"strips {where}")
    assert np.array_equal(gpu_grid(size, w, iters, 16), oracle_mod.grid_rcb(size, w, iters, threads=16))


def test_strips_by_size(oracle_mod, monkeypatch):
    """A grid that the rule sends to the strips, and the same one by the table."""
    rng = np.random.default_rng(8)
    size, iters = [5003, 4999], 9
    w = rng.integers(1, 50, size[0] * size[1]).astype(np.int64)
    say("strips by size")
    got = gpu_grid(size, w, iters, 16)
    monkeypatch.setenv("COUPE_HIP_GRID_STRIPS", "0")
    assert np.array_equal(got, gpu_grid(size, w, iters, 16))
    assert np.array_equal(got, oracle_mod.grid_rcb(size, w, iters, threads=16))
