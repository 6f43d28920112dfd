"""The cosine transforms' lengths, each way and with both row starts (16-byte
aligned lines and ghosted rows at 8), through direct solves and a step against
the oracle.  Bar: 1e-12 of the largest value, as for every Neumann solve."""
import numpy as np
import pytest

from fen_amd import Solver
from fen_amd._lib import BC_WALL, U, V, W
from oracle import oracle as O

pytestmark = pytest.mark.gpu

TOL = 1e-12
SIZES = [(2, (8, 12, 1)), (2, (16, 9, 1)), (2, (64, 20, 1)), (2, (512, 6, 1)), (2, (1024, 6, 1)),
         (3, (8, 16, 5)), (3, (16, 8, 6)), (3, (64, 512, 3)), (3, (512, 64, 3)), (3, (1024, 8, 2))]


@pytest.mark.parametrize("dim,n", SIZES)
def test_cosine_lengths(dim, n):
    print("dct", n, flush=True)
    L = tuple(m / 8.0 for m in n)
    bc = [BC_WALL] * 6
    rng = np.random.default_rng(n[0] + n[1])
    o = O.Oracle(dim, n, L, bc=bc)
    with Solver(dim, n, L, bc=bc) as g:
        for gl in (0, 1):
            f = np.asfortranarray(rng.standard_normal(tuple(m + 2 * gl for m in n)))
            a, b = g.solve_poisson(f, gl), o.poisson_solve(f.copy(order="F"), gl)
            if gl:
                k = slice(1, -1)
                a, b = a[k, k, k], b[k, k, k]
            assert np.abs(a - b).max() <= TOL * np.abs(b).max()
        for s in (g, o):
            s.set_params(density=1.3, viscosity=0.01, cfl=0.2)
        dt = g.set_timestep(4.0)
        o.set_timestep(4.0)
        for f in (U, V, W)[:dim]:
            a = np.asfortranarray(rng.standard_normal(tuple(m + 2 for m in n)))
            if dim == 2:
                a[:, :, 0] = a[:, :, 2] = 0.0
            g.upload(f, a)
            o.field(f)[...] = a
            g.update_ghost_nodes(f)
            o.update_ghost_nodes(f)
        g.navier_stokes_solver(1, dt)
        o.step(1, dt)
        for f in (U, V, W)[:dim]:
            a, b = g.download(f), np.asarray(o.field(f))
            if dim == 2:
                a, b = a[:, :, 1], b[:, :, 1]
            assert np.abs(a - b).max() <= TOL * np.abs(b).max(), f
