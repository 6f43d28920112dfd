"""Each kx column of the Poisson solve is transformed by itself: a right-hand
side that does not depend on x has exact zeros in every column but kx = 0, so
its solution does not depend on x either, to the bit, whatever the grid's
transforms (whole planes, or x and y apart)."""
import numpy as np
import pytest

from fen_amd import Solver
from fen_amd._lib import BC_PERIODIC, BC_WALL, FP32_REFINE

pytestmark = pytest.mark.gpu

GRIDS = [(16, 64, 32), (16, 128, 16), (32, 32, 32), (32, 64, 16), (32, 128, 16), (64, 16, 16), (64, 32, 16), (64, 64, 64),
         (64, 128, 128), (128, 16, 32), (128, 32, 16), (128, 64, 128), (16, 16, 16), (128, 128, 16), (256, 32, 16)]


@pytest.mark.parametrize("precision", [0, FP32_REFINE])
@pytest.mark.parametrize("wall_z", [0, 1])
@pytest.mark.parametrize("n", GRIDS)
def test_columns_do_not_mix(n, wall_z, precision):
    print("columns", n, wall_z, precision, flush=True)
    bc = [BC_PERIODIC] * 4 + [BC_WALL if wall_z else BC_PERIODIC] * 2
    f = np.random.default_rng(n[1]).standard_normal((1,) + n[1:])
    f = np.asfortranarray(np.broadcast_to(f - f.mean(), n))
    with Solver(3, n, tuple(m / 8.0 for m in n), bc=bc, precision=precision) as s:
        a = s.solve_poisson(f, 0)
    assert np.abs(a).max() > 0.0
    assert np.array_equal(a, np.broadcast_to(a[:1], n)), float(np.abs(a - a[:1]).max() / np.abs(a).max())
