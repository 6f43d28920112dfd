"""FP32 direct solves against the oracle, ghosts and mean included: ppn zeroes
its ghosts and then subtracts the solution's mean from the whole array, ppp
leaves both alone (reference src/poisson.f90:1151-1171).

The oracle's singular column fixes phi at the last cell, so the mean that ppn
subtracts is of the solution's own size, far above the bar: 64 roundings in
FP32 of the largest value before the subtraction, as the transforms' elsewhere."""
import numpy as np
import pytest

from fen_amd import Solver
from fen_amd._lib import BC_PERIODIC, BC_WALL, FP32_REFINE
from oracle import oracle as O

pytestmark = pytest.mark.gpu
U32 = 2.0 ** -24


@pytest.mark.parametrize("solver", ["ppn", "ppp"])
@pytest.mark.parametrize("gl", [0, 1])
@pytest.mark.parametrize("n", [(16, 8, 32), (32, 32, 17), (16, 16, 40)])
def test_whole_array(n, gl, solver):
    if solver == "ppp":
        n = n[:2] + (32,)
    print("fp32 solve", solver, n, gl, flush=True)
    bc = [BC_PERIODIC] * 4 + [BC_WALL if solver == "ppn" else BC_PERIODIC] * 2
    L = tuple(m / 8.0 for m in n)
    rng = np.random.default_rng(5)
    z = (np.arange(n[2]) + 0.5) / n[2]
    inner = rng.standard_normal(n) + 3.0 * np.cos(np.pi * z)[None, None, :]
    inner -= inner.mean()
    f = rng.standard_normal(tuple(m + 2 * gl for m in n))   # the ghosts' values before the solve
    f[tuple(slice(gl, m + gl) for m in n)] = inner
    f = np.asfortranarray(f.astype(np.float32).astype(np.float64))
    o = O.Oracle(3, n, L, bc=bc)
    b = o.poisson_solve(f.copy(order="F"), gl)
    with Solver(3, n, L, bc=bc, precision=FP32_REFINE) as s:
        a = s.solve_poisson(f, gl)
    bar = 64 * U32 * 2.0 * np.abs(b).max()
    if gl and solver == "ppn":   # what was subtracted from the zeroed ghosts
        mean = -b[0, 0, 0]
        print(f"  mean subtracted {mean:.4f}, largest value {np.abs(b).max():.4f}, bar {bar:.2e}")
        assert abs(mean) > 1000 * bar
    assert np.abs(a - b).max() <= bar, (float(np.abs(a - b).max()), bar)
