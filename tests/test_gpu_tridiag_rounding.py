"""Round-off of the 2-D solvers' tridiagonal direction, against 80-bit values.

A right-hand side that does not depend on x excites only the column of kx = 0,
the singular one, whose recurrences are plain sums: each row divides by a pivot
of -1/delta^2, and a quotient taken as a product with the rounded reciprocal is
wrong by the same factor on every row, which sums up with the rows instead of
their square root.

The bar is derived from the rounding model: each of a row's operations (the
product with the off-diagonal, the difference, the quotient) is an independent
error of at most u |value|, uniform, variance u^2/3 of its square; the chunks'
carries add two more.  Row i's error reaches x_0 through the n - i rows above
it (the backward recurrence adds d), so the deviation of x_0 is u sqrt(5/3)
sqrt(sum_i ((n - i) d_i)^2), to which the transforms and the backward sums add
a few roundings of the largest value.  Two and a half deviations are allowed."""
import numpy as np
import pytest

from fen_amd import Solver
from fen_amd._lib import BC_PERIODIC, BC_WALL
from oracle import oracle as O

pytestmark = pytest.mark.gpu
U = 2.0 ** -53
LD = np.longdouble


def problem(solver, ny, delta, seed):
    """The solver's solution in 80 bits (up to its constant) and the bar, for a
    right-hand side of y alone whose sum is zero."""
    rng = np.random.default_rng(seed)
    g = rng.standard_normal(ny)
    g = np.rint((g - g.mean()) * 2.0 ** 30)
    g[-1] -= g.sum()          # whole numbers: the sum is exactly zero
    g *= 2.0 ** -30
    d = np.cumsum(g.astype(LD)) * LD(delta) ** 2           # -d_i of the forward recurrence
    x = np.concatenate([[LD(0)], np.cumsum(d[:-1])])       # x_{j+1} - x_j
    x -= x.mean()
    w = np.arange(ny, 0, -1)
    bar = 2.5 * U * np.sqrt(5.0 / 3.0 * float(np.sum((w * d.astype(float)) ** 2))) + 32 * U * float(np.abs(x).max())
    return g, x, bar


@pytest.mark.parametrize("solver,ny", [("nn", 40), ("nn", 333), ("nn", 1000), ("nn", 4000), ("pn", 64), ("pn", 1024)])
@pytest.mark.parametrize("delta", [0.0137, 1.0 / 3.0, 0.25])
def test_singular_column(solver, ny, delta):
    nx = 16
    print("singular column", solver, ny, delta, flush=True)
    bc = [BC_WALL if solver == "nn" else BC_PERIODIC] * 2 + [BC_WALL] * 2 + [BC_PERIODIC] * 2
    L = (nx * delta, ny * delta, delta)
    with Solver(2, (nx, ny, 1), L, bc=bc) as s:
        for seed in range(3):
            g, x, bar = problem(solver, ny, s.delta, seed)
            f = np.asfortranarray(np.broadcast_to(g[None, :, None], (nx, ny, 1)))
            a = s.solve_poisson(f, 0)[:, :, 0]
            o = O.Oracle(2, (nx, ny, 1), L, bc=bc).poisson_solve(f.copy(order="F"), 0)[:, :, 0]
            errs = []
            for z in (a, o):
                z = z.astype(LD)
                z = z - z.mean()
                errs.append(float(np.abs(z - x[None, :]).max()))
            print(f"  seed {seed}: error {errs[0] / bar:.3f} of the bar (oracle {errs[1] / bar:.3f})", flush=True)
            assert errs[0] <= bar and errs[1] <= bar, (errs, bar)
