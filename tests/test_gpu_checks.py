"""The checks of a pending step against those its projection forms when nothing
is pending: the same numbers, so equal to the bit, at grids that its columns of
64 x 8 cells and 8 planes do not divide, on every kind of wall."""
import numpy as np
import pytest

from fen_amd import Solver
from fen_amd._lib import BC_PERIODIC, BC_WALL, FP32_REFINE, P, U, V, W

pytestmark = pytest.mark.gpu

CASES = [((8, 8, 8), (0, 0, 0), 0), ((16, 8, 8), (0, 0, 0), FP32_REFINE), ((64, 16, 9), (0, 0, 1), 0),
         ((128, 8, 23), (0, 0, 1), FP32_REFINE), ((1024, 8, 700), (0, 0, 1), 0), ((32, 16, 11), (1, 0, 1), 0),
         ((128, 16, 17), (1, 1, 1), 0), ((128, 128, 128), (0, 0, 0), 0), ((256, 64, 64), (0, 0, 0), FP32_REFINE)]


@pytest.mark.parametrize("n,walls,precision", CASES)
def test_pending_checks(n, walls, precision, monkeypatch):
    print("checks", n, walls, precision, flush=True)
    bc = []
    for w in walls:
        bc += [BC_WALL if w else BC_PERIODIC] * 2
    rng = np.random.default_rng(n[2])
    init = {f: np.asfortranarray(rng.standard_normal(tuple(m + 2 for m in n))) for f in (U, V, W, P)}
    res = []
    for fused in ("1", "0"):
        monkeypatch.setenv("FEN_FUSED_RUN", fused)
        with Solver(3, n, tuple(m / 8.0 for m in n), bc=bc, precision=precision) as g:
            g.set_params(density=1.3, viscosity=0.01, cfl=0.2)
            dt = g.set_timestep(4.0)
            for f, a in init.items():
                g.upload(f, a)
                g.update_ghost_nodes(f)
            res.append([g.navier_stokes_solver(step, dt)[1:] for step in (1, 2)])
    assert res[0] == res[1]
