"""The tridiagonal direction's solve at the lengths where its chunks begin and
end (and past the longest the chunked kernel takes): direct Poisson solves
against the oracle.  Each sweep rounds once per row, so the bar is 8 roundings
per row (and 8 rows' worth for the transforms) of the largest value."""
import numpy as np
import pytest

from fen_amd import Solver
from fen_amd._lib import BC_PERIODIC, BC_WALL, FP32_REFINE
from oracle import oracle as O

pytestmark = pytest.mark.gpu

EPS = {0: 2.0 ** -53, FP32_REFINE: 2.0 ** -24}


def _solve(dim, n, walls, precision, seed):
    bc = []
    for w in walls:
        bc += [BC_WALL if w else BC_PERIODIC] * 2
    L = tuple(m / 8.0 for m in n)
    rng = np.random.default_rng(seed)
    f = np.asfortranarray(rng.standard_normal(n))
    f -= f.mean()
    with Solver(dim, n, L, bc=bc, precision=precision) as g:
        a = g.solve_poisson(f, 0)
    o = O.Oracle(dim, n, L, bc=bc)
    b = o.poisson_solve(f.copy(order="F"), 0)
    return float(np.abs(a - b).max() / np.abs(b).max())


@pytest.mark.parametrize("nz", [2, 7, 8, 9, 16, 17, 33, 100, 129, 511, 513, 1024, 1025])
@pytest.mark.parametrize("walls", [(0, 0, 1), (1, 0, 1), (1, 1, 1)])
def test_columns_along_z(walls, nz):
    print("tridiag z", walls, nz, flush=True)
    err = _solve(3, (8, 16, nz), walls, 0, nz)
    assert err <= 8 * (nz + 8) * EPS[0], err


@pytest.mark.parametrize("nz", [2, 9, 16, 100, 513, 1025])
def test_columns_fp32(nz):
    """FP32 storage, FP64 elimination: only the transforms round in FP32."""
    print("tridiag fp32", nz, flush=True)
    err = _solve(3, (16, 8, nz), (0, 0, 1), FP32_REFINE, nz)
    assert err <= 64 * EPS[FP32_REFINE], err


@pytest.mark.parametrize("solver,ny", [("pn", 8), ("pn", 64), ("pn", 512), ("pn", 1024), ("nn", 2), ("nn", 7), ("nn", 8),
                                       ("nn", 9), ("nn", 65), ("nn", 200), ("nn", 4095), ("nn", 4097)])
def test_columns_along_y(solver, ny):
    print("tridiag y", solver, ny, flush=True)
    err = _solve(2, (16, ny, 1), (solver == "nn", 1, 0), 0, ny)
    assert err <= 8 * (ny + 8) * EPS[0], err


@pytest.mark.parametrize("solver", ["ppn", "ppp"])
def test_ghosts_of_an_fp32_solve(solver):
    """With ghosts: ppn leaves them minus the mean it subtracts, ppp as they
    came; the interior is the ghostless solve's."""
    n = (16, 8, 32)
    bc = [BC_PERIODIC] * 4 + ([BC_WALL] * 2 if solver == "ppn" else [BC_PERIODIC] * 2)
    rng = np.random.default_rng(3)
    f = np.asfortranarray(rng.standard_normal(tuple(m + 2 for m in n)))
    inner = np.asfortranarray(f[1:-1, 1:-1, 1:-1])
    with Solver(3, n, (2.0, 1.0, 4.0), bc=bc, precision=FP32_REFINE) as g:
        a, b = g.solve_poisson(f, 1), g.solve_poisson(inner, 0)
    assert np.array_equal(a[1:-1, 1:-1, 1:-1], b)
    ghost = np.ones(a.shape, bool)
    ghost[1:-1, 1:-1, 1:-1] = False
    if solver == "ppp":
        assert np.array_equal(a[ghost], f[ghost].astype(np.float32).astype(np.float64))
    else:
        assert np.unique(a[ghost]).size == 1
