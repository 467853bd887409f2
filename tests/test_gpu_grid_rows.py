"""The grid search's stencil rows: bodies before, in and past the last 16-entry
wave, grids of 4 to 64 cells an axis wrapped over larger domains, one to four
levels, sparse and so dense that a wave's pairs exceed the kept ones.  Every
overlapping pair is found once, as brute force has it."""
import numpy as np
import pytest

import oracle as O
from experiments_amd import _lib as L
from test_gpu_grid import run_grid

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 63, 65, 1000, 4001])
@pytest.mark.parametrize("dims,box", [((4, 4, 4), 9.0), ((4, 8, 16), 30.0), ((64, 4, 8), 14.0),
                                      ((32, 32, 32), 40.0)])
@pytest.mark.parametrize("levels", [1, 2, 4])
def test_rows_equal_brute_force(n, dims, box, levels):
    rng = np.random.default_rng(n + 7 * levels + dims[0])
    top = 0.5 * 2 ** (levels - 1)
    half = np.exp(rng.uniform(np.log(0.1), np.log(top), (n, 3))) * 0.999
    c = rng.uniform(-0.5, 0.5, (n, 3)) * box
    c[: n // 3] = np.round(c[: n // 3])  # centres on cell edges
    half[: n // 6] = 0.5                 # boxes of a whole cell, touching
    mn, mx = np.zeros((n, 4), np.float32), np.zeros((n, 4), np.float32)
    mn[:, :3], mx[:, :3] = c - half, c + half
    got, flags, _ = run_grid(mn, mx, 1.0, dims, levels, 1 << 22)
    assert flags == 0
    assert np.array_equal(got, O.find_pairs_brute(mn, mx))


def test_far_and_unbounded_boxes():
    """Boxes at large coordinates, an unbounded one (reported) and NaN ones,
    which overlap nothing."""
    n = 300
    rng = np.random.default_rng(2)
    c = np.round(rng.uniform(-4, 4, (n, 3)))
    c[100:] += 4096.0
    c[200:] -= 3.0e6
    mn, mx = np.zeros((n, 4), np.float32), np.zeros((n, 4), np.float32)
    mn[:, :3], mx[:, :3] = c - 0.5, c + 0.5
    mx[7, 1] = np.inf
    mn[150, 0] = mx[151, 2] = np.nan
    got, flags, _ = run_grid(mn, mx, 1.0, (16, 16, 16), 2, 1 << 16)
    assert flags == L.OVERFLOW_LEVEL
    ref = O.find_pairs_brute(mn, mx)
    ref = ref[(ref != 7).all(1)]
    assert len(ref) > 100
    assert np.array_equal(got, ref)
