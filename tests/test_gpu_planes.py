"""The x and y transforms of whole z planes at every plane shape they take, and
just outside: direct solves and steps against the oracle.

Bars: the transforms round O(log n) times per value (64 roundings of the
largest value), the tridiagonal sweeps once per row (8 rows' worth per row);
a step adds its stencil sums (512 roundings over two steps)."""
import numpy as np
import pytest

from fen_amd import Solver
from fen_amd._lib import BC_PERIODIC, BC_WALL, FP32_REFINE, U, V, W
from oracle import oracle as O
from tests.test_gpu_adjoint import test_gpu_adjoint_matches_oracle_adjoint as adjoint_matches_oracle

pytestmark = pytest.mark.gpu

EPS = {0: 2.0 ** -53, FP32_REFINE: 2.0 ** -24}
CASES = [(nx, ny, 8) for nx, ny in [(16, 32), (16, 64), (16, 128), (32, 16), (32, 32), (32, 64), (32, 128), (64, 16),
                                    (64, 32), (64, 64), (128, 8), (128, 16), (128, 32), (256, 16)]]
CASES += [(64, 128, 64), (64, 128, 128), (128, 64, 128), (16, 64, 1024)]


def _bc(wall_z):
    return [BC_PERIODIC] * 4 + [BC_WALL if wall_z else BC_PERIODIC] * 2


@pytest.mark.parametrize("precision", [0, FP32_REFINE])
@pytest.mark.parametrize("wall_z", [0, 1])
@pytest.mark.parametrize("n", CASES)
def test_plane_solves(n, wall_z, precision):
    if wall_z:
        n = (n[0], n[1], n[2] + 1)   # the tridiagonal direction takes any length
    print("plane", n, wall_z, precision, flush=True)
    L = tuple(m / 8.0 for m in n)
    rng = np.random.default_rng(n[0] + n[1])
    f = np.asfortranarray(rng.standard_normal(n))
    f -= f.mean()
    with Solver(3, n, L, bc=_bc(wall_z), precision=precision) as g:
        a = g.solve_poisson(f, 0)
        if precision == 0:
            assert np.array_equal(g.solve_poisson_noalloc(f, 0), a)
    o = O.Oracle(3, n, L, bc=_bc(wall_z))
    b = o.poisson_solve(f.copy(order="F"), 0)
    bar = 8 * (n[2] + 8) if wall_z and precision == 0 else 64
    assert np.abs(a - b).max() <= bar * EPS[precision] * np.abs(b).max()


def test_long_grid_without_allocation():
    """More planes than the allocation-free solve's scratch holds sums: the separate passes."""
    n = (32, 32, 32770)
    print("plane", n, flush=True)
    f = np.asfortranarray(np.random.default_rng(1).standard_normal(n))
    with Solver(3, n, tuple(m / 8.0 for m in n), bc=_bc(1)) as g:
        assert np.array_equal(g.solve_poisson_noalloc(f, 0), g.solve_poisson(f, 0))


@pytest.mark.parametrize("wall_z", [0, 1])
@pytest.mark.parametrize("n", [(16, 64, 8), (32, 32, 8), (64, 16, 8), (128, 32, 8), (128, 64, 128)])
def test_plane_steps(n, wall_z):
    print("plane steps", n, wall_z, flush=True)
    L = tuple(m / 8.0 for m in n)
    rng = np.random.default_rng(n[1])
    shape = tuple(m + 2 for m in n)
    o = O.Oracle(3, n, L, bc=_bc(wall_z))
    with Solver(3, n, L, bc=_bc(wall_z)) as g:
        for s in (g, o):
            s.set_params(density=1.3, viscosity=0.01, cfl=0.2)
        dt = g.set_timestep(4.0)
        o.set_timestep(4.0)
        for f in (U, V, W):
            a = np.asfortranarray(rng.standard_normal(shape))
            g.upload(f, a)
            o.field(f)[...] = a
            g.update_ghost_nodes(f)
            o.update_ghost_nodes(f)
        for step in (1, 2):
            g.navier_stokes_solver(step, dt)
            o.step(step, dt)
        for f in (U, V, W):
            a, b = g.download(f), np.asarray(o.field(f))
            assert np.abs(a - b).max() <= 512 * EPS[0] * np.abs(b).max(), f


@pytest.mark.parametrize("n", [(64, 32, 128), (128, 64, 256)])
def test_plane_adjoint(n, monkeypatch):
    """The transposed projection's right-hand side, formed as the planes load;
    the transposed step's march in its shortest and longest cuts."""
    print("plane adjoint", n, flush=True)
    adjoint_matches_oracle(n, monkeypatch)
