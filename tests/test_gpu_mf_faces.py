"""Two-phase runs with unlike faces on an axis (one Periodic, one Wall):
fen_create takes them (solver pn or nn) and the ghosts of the vof, its normals
and curvature, rho, mu and p_hat follow each face's own rule, as the fields'
first fill and the oracle's.

The bars are tests/test_gpu_multiphase.py's: libm of the device and the host
may differ in the last bit, so vof to 1e-10 absolute and the flow to 1e-9
relative.  Two steps without surface tension move by at most 2e-14 for a
1e-15 change of the start (the oracle shows it; with sigma > 0 the curvature
of nearly empty cells takes that to 1e-6)."""
import numpy as np
import pytest

from fen_amd._lib import BC_PERIODIC as PER, BC_WALL as WALL, MU, P, RHO, U, V, VOF
from tests.test_gpu_multiphase import _pair, _rel
from tests.test_oracle_multiphase import vof_from_distance

pytestmark = pytest.mark.gpu

FACES = [(PER, PER, PER, WALL), (PER, PER, WALL, PER), (PER, WALL, WALL, WALL), (WALL, PER, WALL, WALL),
         (PER, WALL, WALL, PER), (WALL, PER, PER, WALL), (WALL, WALL, WALL, WALL)]


def setup(faces):
    """A wavy slanted band cut off at the sides: both fluids meet all four
    faces, no two alike."""
    n, d = (32, 64), 1.0 / 32
    lx, ly = n[0] * d, n[1] * d
    band = lambda x, y: 0.22 * ly - np.abs(y - 0.45 * ly - 0.37 * ly * (2.0 * x / lx - 1.0)
                                           - 0.06 * ly * np.cos(7.3 * x / lx + 0.4))
    vof = vof_from_distance(lambda x, y: np.maximum(band(x, y), 0.13 * lx - np.abs(x - 0.31 * lx)), n, d)
    i, j = np.arange(1, n[0] + 1)[:, None] / n[0], np.arange(1, n[1] + 1)[None, :] / n[1]
    u, v = 0.3 * np.cos(2.0 * i + 1.1 * j + 0.3), 0.4 * np.sin(1.7 * i - 2.1 * j + 0.2)
    return n, (lx, ly), list(faces) + [PER, PER], vof, u, v


@pytest.mark.parametrize("faces", FACES)
def test_two_phase_steps_on_unlike_faces(faces):
    print("two-phase faces", faces, flush=True)
    n, L, bc, vof, u, v = setup(faces)
    o, g = _pair(n, L, bc, (1.0, 3.0, 0.01, 0.03, 0.0), vof, u, v,
                 params=dict(density=1.0, viscosity=0.01, g=(0.0, -1.0, 0.0), cfl=0.1))
    for s in (o, g):
        s.update_material_properties()
    for f in (RHO, MU):   # the whole live plane, ghosts included
        assert np.array_equal(g.download(f)[:, :, 1], o.field(f)[:, :, 1]), f
    dt = o.mf_set_timestep(1.0)
    assert g.set_timestep(1.0) == dt
    for s in range(1, 3):
        o.step(s, dt)
        g.navier_stokes_solver(s, dt)
        a, b = g.download(VOF)[:, :, 1], o.field(VOF)[:, :, 1]
        assert np.abs(a - b).max() < 1e-10, (s, np.abs(a - b).max())
    errs = {f: _rel(g.download(f)[:, :, 1], o.field(f)[:, :, 1]) for f in (RHO, MU, U, V, P)}
    print("two-phase faces", faces, "rel err", errs, flush=True)
    for f, e in errs.items():
        assert e < 1e-9, (f, e)
