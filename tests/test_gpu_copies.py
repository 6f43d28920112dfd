"""Fields up and down unchanged (FP32: each value rounded once) on both sides
of the size from which copies go in pieces, with a ragged last piece."""
import numpy as np
import pytest

from fen_amd import Solver
from fen_amd._lib import DVO_X, FP32_REFINE, U

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, FP32_REFINE])
@pytest.mark.parametrize("n", [(64, 64, 64), (128, 64, 64), (128, 128, 64), (256, 128, 64), (64, 512, 64)])
def test_round_trip(n, precision):
    print("round trip", n, precision, flush=True)
    rng = np.random.default_rng(n[0])
    with Solver(3, n, (1.0, 1.0, 1.0), precision=precision) as a, Solver(3, n, (1.0, 1.0, 1.0), precision=precision) as b:
        for s in (a, b):
            for f in (U, DVO_X):
                x = np.asfortranarray(rng.standard_normal(s.shape(f)))
                s.upload(f, x)
                want = x if precision == 0 else x.astype(np.float32).astype(np.float64)
                assert np.array_equal(s.download(f), want), f
