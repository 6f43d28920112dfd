"""Steps replayed from the captured HIP graph equal eager steps to the bit.

Grids whose steps end pending never reach the graph, so fusion is off in both
arms (FEN_FUSED_RUN=0), but for the 2-D Inflow/Outflow grid, whose steps do not
(phi is fixed at its Outflow face) and which takes the graph as it is.  Between replays the scalars and PHI are read: a read turns the
step's block sums of the mean and its unread checks into numbers, and the next
replay has to leave both pending again."""
import numpy as np
import pytest

from fen_amd import cases
from fen_amd._lib import DVO_X, FP32_REFINE, P, PHI, U, V, W
from tests.common import make_gpu

pytestmark = pytest.mark.gpu

CASES = {
    "pp": lambda: cases.tgv2d(32, steps=1), "pn": lambda: cases.channel2d(32, 16), "nn": lambda: cases.cavity2d(32, 27),
    "ppp": lambda: cases.tgv3d(32, steps=1), "ppn": lambda: cases.channel(32, 16, 16, steps=1),
    "npn": lambda: cases.duct3d(16, 16, 12), "nnn": lambda: cases.cavity3d(16, 16, 12),
    "pn inflow": lambda: cases.channel2d(32, 16, inflow=True), "npn inflow": lambda: cases.duct3d(16, 16, 12, z_io=True),
}
RUNS = [(name, 0) for name in CASES] + [(name, FP32_REFINE) for name in ("pp", "ppp", "ppn")]


@pytest.mark.parametrize("name,precision", RUNS)
def test_replays_between_reads(name, precision, monkeypatch):
    print("step graph", name, precision, flush=True)
    case = CASES[name]()
    if name == "pn inflow":
        monkeypatch.delenv("FEN_FUSED_RUN", raising=False)
    else:
        monkeypatch.setenv("FEN_FUSED_RUN", "0")
    fields = [U, V, P, PHI, DVO_X] + ([W] if case.dim == 3 else [])
    results = []
    for graph in ("0", "1"):
        monkeypatch.setenv("FEN_STEP_GRAPH", graph)
        g = make_gpu(case, precision)
        seen, dt = [], case.dt

        def read(*what):
            for f in what:
                seen.append(list(g.scalars().values()) if f == "scalars" else g.download(f))

        g.navier_stokes_solver(1, dt, want_checks=False)       # captured
        read("scalars", PHI)
        for s, what in enumerate([(PHI,), ("scalars",), (PHI, "scalars"), (), ("scalars", PHI), fields], 2):
            g.navier_stokes_solver(s, dt, want_checks=False)   # replayed
            read(*what)
        seen.append(g.navier_stokes_solver(8, dt))             # with its checks
        g.run(8, 3, dt)
        read(*fields, "scalars")
        g.run(11, 3, 0.5 * dt)                                 # another dt: captured again
        read(PHI)
        g.run(14, 2, 0.5 * dt)
        read("scalars", *fields)
        g.set_params(density=case.density, viscosity=2 * case.viscosity, g=case.g, cfl=case.cfl)
        for s in range(17, 20):                                # other parameters: captured again
            g.navier_stokes_solver(s, 0.5 * dt, want_checks=False)
            read(PHI, "scalars")
        read(*fields)
        results.append(seen)
        g.close()
    assert len(results[0]) == len(results[1])
    for q, (a, b) in enumerate(zip(*results)):
        assert np.array_equal(np.asarray(a), np.asarray(b)), q
