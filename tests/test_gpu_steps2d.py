"""2-D steps whose kernels fill the ghosts they produce: every boundary rule
(moving and permeable walls, free-slip overrides, Inflow and Outflow,
periodic), random boundary values, sizes down to the smallest.  The velocity
(and the vof) with its ghosts and corners against the oracle, where four steps
round a few hundred times per value: 1e-12 of the largest.  The pressure, which
starts at the size of its first projection's correction and ends a thousand
times smaller, acts on the velocity through every step; its ghosts, as all the
others, must be left exactly as the ghost fill would leave them."""
import numpy as np
import pytest

from fen_amd import Solver
from fen_amd._lib import (BC_INFLOW, BC_OUTFLOW, BC_PERIODIC, BC_WALL, BOTTOM, DVO_X, DVO_Y, FP32_REFINE, LEFT, P, PHI,
                          RIGHT, S_X, S_Y, TOP, U, V, VOF)
from oracle import oracle as O

pytestmark = pytest.mark.gpu
Pe, Wa, In, Out = BC_PERIODIC, BC_WALL, BC_INFLOW, BC_OUTFLOW

CASES = [
    # nx, ny, faces, {(field, face): type override}
    ((8, 8), [Pe, Pe, Pe, Pe], {}),
    ((128, 64), [Pe, Pe, Pe, Pe], {}),
    ((64, 8), [Pe, Pe, Wa, Wa], {}),
    ((16, 64), [Pe, Pe, Wa, Wa], {(U, TOP): 2, (U, BOTTOM): 2}),
    ((32, 16), [Pe, Pe, In, Out], {}),
    ((8, 2), [Wa, Wa, Wa, Wa], {}),
    ((64, 37), [Wa, Wa, Wa, Wa], {}),
    ((32, 5), [Wa, Wa, Wa, Wa], {(V, LEFT): 2, (V, RIGHT): 2, (U, TOP): 2}),
    ((16, 40), [Wa, Wa, In, Out], {}),
]


def _pair(n, faces, types, seed):
    nx, ny = n
    bc, size, L = faces + [Pe, Pe], (nx, ny, 1), (1.0, ny / nx, 1.0 / nx)
    rng = np.random.default_rng(seed)
    shape = (nx + 2, ny + 2, 3)
    init = {f: np.asfortranarray(0.1 * rng.standard_normal(shape)) for f in (U, V, P)}
    g, o = Solver(2, size, L, bc=bc), O.Oracle(2, size, L, bc=bc)
    for s in (g, o):
        s.set_params(density=1.0, viscosity=0.02, g=(0.3, -0.2, 0.0), cfl=0.2)
    for (f, face), t in types.items():
        g.set_bc_type(f, face, t)
        o.set_bc_type(f, face, t)
    for f in (U, V):
        for face in (LEFT, RIGHT, BOTTOM, TOP):
            plane = 0.05 * rng.standard_normal((ny + 2 if face < 2 else nx + 2, 3))
            g.set_bc_plane(f, face, plane)
            o.bc_plane(f, face)[...] = plane
    for f, a in init.items():
        g.upload(f, a)
        o.field(f)[...] = a
        g.update_ghost_nodes(f)
        o.update_ghost_nodes(f)
    return g, o


def _compare(g, o, fields):
    for f in fields:
        a, b = g.download(f)[:, :, 1], o.field(f)[:, :, 1]
        err = float(np.abs(a - b).max() / np.abs(b).max())
        assert err < 1e-12, (f, err)
    for f in fields + (P, PHI):
        a = g.download(f)[:, :, 1]
        g.update_ghost_nodes(f)
        assert np.array_equal(a, g.download(f)[:, :, 1]), f


@pytest.mark.parametrize("n,faces,types", CASES)
def test_steps_match_oracle(n, faces, types):
    print("steps 2-D", n, faces, types, flush=True)
    g, o = _pair(n, faces, types, n[1])
    dt = 0.02 / n[0]
    for s in (g, o):
        s.set_dt_o(dt)
    for step in (1, 2, 3):
        g.navier_stokes_solver(step, dt, want_checks=False)
        o.step(step, dt)
        if step == 2:
            sc = g.scalars()
    _, mdo, mco = o.step(4, dt)
    _, mdg, mcg = g.navier_stokes_solver(4, dt)
    assert sc["maxcfl"] > 0 and abs(mcg - mco) <= 1e-12 * mco
    _compare(g, o, (U, V))


@pytest.mark.parametrize("n,faces", [((32, 8), [Pe, Pe, Wa, Wa]), ((16, 64), [Pe, Pe, Pe, Pe]), ((32, 21), [Wa] * 4)])
def test_two_phase_steps_match_oracle(n, faces):
    """Non-zero velocities on and beside the walls; the interface crosses them."""
    print("two-phase", n, faces, flush=True)
    g, o = _pair(n, faces, {}, 7)
    x = (np.arange(n[0] + 2) - 0.5)[:, None] / n[0]
    y = (np.arange(n[1] + 2) - 0.5)[None, :] / n[0]
    f = 0.5 * (1.0 + np.tanh(n[0] * (0.31 * x + 0.87 * y - 0.55 * n[1] / n[0])))
    vof = np.asfortranarray(np.repeat(f[:, :, None], 3, axis=2))
    for s in (g, o):
        s.set_multiphase(1.0, 3.0, 0.01, 0.03, 0.2)
    g.upload(VOF, vof)
    o.field(VOF)[...] = vof
    for s in (g, o):
        s.update_ghost_nodes(VOF)
        s.update_material_properties()
    dt = 0.02 / n[0]
    for s in (g, o):
        s.set_dt_o(dt)
    for step in (1, 2, 3, 4):
        g.navier_stokes_solver(step, dt, want_checks=False)
        o.step(step, dt)
    _compare(g, o, (U, V, VOF))


@pytest.mark.parametrize("precision,source", [(0, False), (0, True), (FP32_REFINE, True)])
@pytest.mark.parametrize("n,faces,types", [c for c in CASES if In not in c[1]] + [((64, 256), [Pe] * 4, {}), ((512, 16), [Wa] * 4, {})])
def test_fused_steps_equal_single_steps(n, faces, types, precision, source, monkeypatch):
    """The projection fused with the next step's momentum, bit for bit."""
    if precision and Wa in faces:
        pytest.skip("the FP32 form is periodic in 2-D")
    print("fused 2-D", n, faces, types, precision, source, flush=True)
    rng = np.random.default_rng(5)
    init = {f: np.asfortranarray(0.1 * rng.standard_normal((n[0] + 2, n[1] + 2, 3))) for f in (U, V, P)}
    planes = {(f, face): 0.05 * rng.standard_normal((n[1] + 2 if face < 2 else n[0] + 2, 3))
              for f in (U, V) for face in (LEFT, RIGHT, BOTTOM, TOP)}
    force = {f: np.asfortranarray(rng.standard_normal((n[0], n[1], 1))) for f in (S_X, S_Y)} if source else {}
    res = {}
    for fused in ("1", "0"):
        monkeypatch.setenv("FEN_FUSED_RUN", fused)
        g = Solver(2, (n[0], n[1], 1), (1.0, n[1] / n[0], 1.0), bc=faces + [Pe, Pe], precision=precision)
        g.set_params(density=1.3, viscosity=0.02, g=(0.3, 0.0, 0.0), cfl=0.2)
        for (f, face), t in types.items():
            g.set_bc_type(f, face, t)
        for (f, face), a in planes.items():
            g.set_bc_plane(f, face, a)
        for f, a in {**init, **force}.items():
            g.upload(f, a)
            if f in init:
                g.update_ghost_nodes(f)
        g.set_dt_o(0.02 / n[0])
        out = []
        for step in range(1, 6):
            g.navier_stokes_solver(step, 0.02 / n[0], want_checks=False)
            if step in (2, 3):
                sc = g.scalars()      # the checks of a pending step
                out += [sc["maxdiv"], sc["maxcfl"]]
            if step == 3:
                out += [g.download(f)[:, :, 1] for f in (U, V)]
        out += [g.download(f)[:, :, 1] for f in (U, V, P, PHI)] + [g.download(f) for f in (DVO_X, DVO_Y)]
        res[fused] = out
        g.close()
    for k, (a, b) in enumerate(zip(res["1"], res["0"])):
        assert np.array_equal(np.asarray(a), np.asarray(b)), k
