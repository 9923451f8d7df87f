"""2D grids by strips with an axis longer than 64 steps of a workgroup (16384
cross-sections): a chunk of an axis' prefix is then several steps, which carry
the prefix on, and the medians look their chunk up by its length.  Ids against
the oracle and against the table's."""
import numpy as np
import pytest

from tests.test_gpu_grid import gpu_grid, say

pytestmark = pytest.mark.gpu

SIZES = [([16383, 21], 8), ([16384, 40], 9), ([16385, 40], 10), ([21, 16383], 8), ([40, 16384], 9), ([40, 16385], 10),
         ([33000, 70], 12), ([70, 33000], 12), ([40961, 17], 11), ([17, 40961], 11), ([100_003, 3], 9), ([3, 100_003], 9)]


@pytest.mark.parametrize("size,iters", SIZES)
@pytest.mark.parametrize("kind", ["i32", "f64int", "one end"])
def test_long_axes(oracle_mod, monkeypatch, size, iters, kind):
    rng = np.random.default_rng(size[0] + 3 * size[1] + iters)
    n = size[0] * size[1]
    if kind == "i32":
        w = rng.integers(-5, 1000, n).astype(np.int32)
    elif kind == "f64int":
        w = rng.integers(0, 100, n).astype(np.float64)
    else:   # nearly all of the weight in the last tenth of the cells: splits far along the axis
        w = rng.integers(0, 2, n).astype(np.float64)
        w[n - n // 10:] += 1000.0
    threads = 2 + size[1] % 30
    say(f"long strips {size} {kind} L={iters} threads={threads}")
    monkeypatch.setenv("COUPE_HIP_GRID_STRIPS", "1")
    got = gpu_grid(size, w, iters, threads)
    assert np.array_equal(got, oracle_mod.grid_rcb(size, w, iters, threads=threads))
    monkeypatch.setenv("COUPE_HIP_GRID_STRIPS", "0")
    assert np.array_equal(got, gpu_grid(size, w, iters, threads))
