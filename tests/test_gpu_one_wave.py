"""Direct solves on both sides of the lines where the z pass and the 2-D cosine
passes change between one-wave and larger workgroups, against the oracle.

Bars: the transforms round O(log n) times per value (64 roundings of the
largest value); the tridiagonal sweeps of nn once per row (8 rows' worth per
row)."""
import numpy as np
import pytest

from fen_amd import Solver
from fen_amd._lib import BC_PERIODIC, BC_WALL, FP32_REFINE
from oracle import oracle as O

pytestmark = pytest.mark.gpu

EPS = {0: 2.0 ** -53, FP32_REFINE: 2.0 ** -24}


def _error(n, wall, precision):
    dim = 2 if n[2] == 1 else 3
    bc = [BC_WALL if wall else BC_PERIODIC] * 4 + [BC_PERIODIC] * 2
    L = tuple(m / 8.0 for m in n)
    f = np.asfortranarray(np.random.default_rng(n[0] + n[1]).standard_normal(n))
    f -= f.mean()
    with Solver(dim, n, L, bc=bc, precision=precision) as g:
        a = g.solve_poisson(f, 0)
    b = O.Oracle(dim, n, L, bc=bc).poisson_solve(f.copy(order="F"), 0)
    return float(np.abs(a - b).max() / np.abs(b).max()) / EPS[precision]


@pytest.mark.parametrize("precision", [0, FP32_REFINE])
@pytest.mark.parametrize("n", [(16, 8, 512), (8, 16, 512), (16, 16, 512), (8, 32, 512), (32, 16, 512), (32, 16, 256),
                               (64, 16, 256), (32, 32, 256), (16, 32, 128), (8, 8, 1024)])
def test_z_pass(n, precision):
    print("z pass", n, precision, flush=True)
    err = _error(n, 0, precision)
    assert err <= 64, err


@pytest.mark.parametrize("n", [(512, 7, 1), (512, 335, 1), (512, 337, 1), (512, 385, 1), (256, 337, 1), (256, 1025, 1)])
def test_cosine_passes(n):
    print("cosine passes", n, flush=True)
    err = _error(n, 1, 0)
    assert err <= 8 * (n[1] + 8), err
