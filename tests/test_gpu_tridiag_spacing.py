"""The tridiagonal direction at spacings that are no power of two: the singular
column's last pivot is then round-off instead of zero, its quotient a constant
of any size that the pressure does not depend on.  Solutions are compared with
the oracle's up to that constant.

Each sweep rounds once per row, so the bar is 8 roundings per row (and 8 rows'
worth for the transforms) of the largest value, the constant included."""
import numpy as np
import pytest

from fen_amd import Solver
from fen_amd._lib import BC_PERIODIC, BC_WALL
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nz", [8, 9, 33, 100, 513, 1025])
@pytest.mark.parametrize("walls", [(0, 0, 1), (1, 0, 1), (1, 1, 1)])
@pytest.mark.parametrize("delta", [0.0137, 1.0 / 3.0])
def test_columns_along_z(walls, nz, delta):
    n = (16, 8, nz)
    print("spacing", walls, nz, delta, flush=True)
    bc = []
    for w in walls:
        bc += [BC_WALL if w else BC_PERIODIC] * 2
    L = tuple(m * delta for m in n)
    f = np.asfortranarray(np.random.default_rng(nz).standard_normal(n))
    f -= f.mean()
    with Solver(3, n, L, bc=bc) as g:
        a = g.solve_poisson(f, 0)
    b = O.Oracle(3, n, L, bc=bc).poisson_solve(f.copy(order="F"), 0)
    bar = 8 * (nz + 8) * 2.0 ** -53 * max(np.abs(a).max(), np.abs(b).max())
    a, b = a - a.mean(), b - b.mean()
    err = float(np.abs(a - b).max())
    print(f"  error {err / bar:.3f} of the bar, bar {bar / np.abs(b).max():.1e} of the solution", flush=True)
    assert err <= bar
