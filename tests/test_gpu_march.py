"""The fused projection + momentum march against single steps (bit for bit)
where its cutting of the grid can go wrong: grids narrower than a tile, on
both sides of the line between its two tile widths, nz that no march length
divides, and densities whose reciprocal is not exact."""
import numpy as np
import pytest

from fen_amd import Solver
from fen_amd._lib import BC_PERIODIC, BC_WALL, FP32_REFINE, P, S_X, S_Y, S_Z, U, V, W
from tests.test_gpu_fused import _state

pytestmark = pytest.mark.gpu

CASES = [
    # n, walls (x, y, z), precision, density, source
    ((8, 8, 8), (0, 0, 0), 0, 1.0, False),
    ((64, 8, 16), (0, 0, 0), 0, 1.3, False),
    ((64, 16, 8), (0, 0, 0), FP32_REFINE, 1.0, False),
    ((128, 32, 16), (0, 0, 0), FP32_REFINE, 0.7, True),
    ((64, 16, 2), (0, 0, 1), 0, 1.0, False),
    ((32, 16, 37), (0, 0, 1), 0, 1.3, True),
    ((128, 8, 19), (0, 0, 1), FP32_REFINE, 1.0, False),
    ((64, 8, 23), (1, 0, 1), 0, 0.5, False),
    ((128, 16, 41), (1, 1, 1), 0, 1.3, True),
    ((128, 64, 641), (0, 0, 1), 0, 1.0, False),     # wide FP64 tiles from 5 * 2^20 cells
    ((128, 64, 639), (0, 0, 1), 0, 1.0, False),
    ((256, 64, 321), (1, 0, 1), 0, 1.3, False),
    ((256, 64, 321), (1, 1, 1), 0, 1.0, True),
    ((256, 256, 128), (0, 0, 0), 0, 1.0, False),
]


@pytest.mark.parametrize("n,walls,precision,density,source", CASES)
def test_march_equals_single_steps(n, walls, precision, density, source, monkeypatch):
    print("march", n, walls, precision, density, source, flush=True)
    bc = []
    for w in walls:
        bc += [BC_WALL if w else BC_PERIODIC] * 2
    rng = np.random.default_rng(n[2])
    shape = tuple(m + 2 for m in n)
    init = {f: np.asfortranarray(rng.standard_normal(shape)) for f in (U, V, W, P)}
    force = {f: np.asfortranarray(rng.standard_normal(n)) for f in (S_X, S_Y, S_Z)} if source else {}
    d = 1.0 / n[0]
    res = {}
    for fused in ("1", "0"):
        monkeypatch.setenv("FEN_FUSED_RUN", fused)
        g = Solver(3, n, tuple(d * m for m in n), bc=bc, precision=precision)
        g.set_params(density=density, viscosity=0.01, cfl=0.2)
        for f, a in {**init, **force}.items():
            g.upload(f, a)
            if f in init:
                g.update_ghost_nodes(f)
        g.run(0, 3, g.set_timestep(8.0))
        res[fused] = _state(g)
        g.close()
    for k, (a, b) in enumerate(zip(res["1"], res["0"])):
        assert np.array_equal(np.asarray(a), np.asarray(b)), k
