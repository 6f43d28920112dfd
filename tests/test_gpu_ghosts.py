"""The ghost fill and the steps' reading of it under mixed boundary rules: every
field's ghosts bit for bit against the oracle's fill for random types (Dirichlet
or Neumann on wall faces) and boundary planes, and two steps of those
conditions against the oracle (bar: 1024 roundings of the largest value, the
transforms', the tridiagonal sweeps' and the stencils' together)."""
import numpy as np
import pytest

from fen_amd import Solver
from fen_amd._lib import BC_PERIODIC, BC_WALL, P, U, V, W
from oracle import oracle as O

pytestmark = pytest.mark.gpu

WALLS = {"ppn": (0, 0, 1), "npn": (1, 0, 1), "nnn": (1, 1, 1), "pn": (0, 1, 0), "nn": (1, 1, 0)}


@pytest.mark.parametrize("seed", range(4))
@pytest.mark.parametrize("solver", list(WALLS))
def test_mixed_rules(solver, seed):
    print("ghosts", solver, seed, flush=True)
    dim = 3 if len(solver) == 3 else 2
    n = (16, 8, 11 if dim == 3 else 1)
    walls = WALLS[solver]
    bc = []
    for w in walls:
        bc += [BC_WALL if w else BC_PERIODIC] * 2
    L = tuple(m / 8.0 for m in n)
    rng = np.random.default_rng(100 * seed + len(solver))
    o = O.Oracle(dim, n, L, bc=bc)
    fields = (U, V, W, P) if dim == 3 else (U, V, P)
    shape = tuple(m + 2 for m in n)
    with Solver(dim, n, L, bc=bc) as g:
        for s in (g, o):
            s.set_params(density=1.3, viscosity=0.01, cfl=0.2)
        dt = g.set_timestep(4.0)
        o.set_timestep(4.0)
        for f in fields:
            for face in range(2 * dim):
                if not walls[face // 2]:
                    continue
                t = int(rng.integers(1, 3))
                g.set_bc_type(f, face, t)
                o.set_bc_type(f, face, t)
                plane = o.bc_plane(f, face)
                plane[...] = 0.1 * rng.standard_normal(plane.shape)
                g.set_bc_plane(f, face, plane)
            a = np.asfortranarray(rng.standard_normal(shape))
            if dim == 2:
                a[:, :, 0] = a[:, :, 2] = 0.0
            g.upload(f, a)
            o.field(f)[...] = a
            g.update_ghost_nodes(f)
            o.update_ghost_nodes(f)
            x, y = g.download(f), np.asarray(o.field(f))
            if dim == 2:
                x, y = x[:, :, 1], y[:, :, 1]
            assert np.array_equal(x, y), f
        for step in (1, 2):
            g.navier_stokes_solver(step, dt)
            o.step(step, dt)
        for f in fields[:dim]:
            x, y = g.download(f), np.asarray(o.field(f))
            if dim == 2:
                x, y = x[:, :, 1], y[:, :, 1]
            assert np.abs(x - y).max() <= 1024 * 2.0 ** -53 * np.abs(y).max(), f
