"""Downloads into arrays that are pinned already: the same values as into
pageable ones, and straight over the bus.  Pageable arrays of this size go
through the library's own pinned pieces, one more copy on the host (27 GB/s
against 57); a pinned one must not pay for it."""
import time

import numpy as np
import pytest
import torch

from fen_amd import Solver
from fen_amd._lib import P, U
from fen_amd.solver import _dp

pytestmark = pytest.mark.gpu


def _best(s, field, a, n=8):
    best = np.inf
    for _ in range(n):
        t = time.perf_counter()
        s._check(s.lib.fen_download(s.h, field, _dp(a), a.size))
        best = min(best, time.perf_counter() - t)
    return best


def test_download_into_pinned_memory():
    n = (128, 128, 128)
    with Solver(3, n, (1.0, 1.0, 1.0)) as s:
        x = np.asfortranarray(np.random.default_rng(1).standard_normal(s.shape(U)))
        s.upload(U, x)
        plain = np.zeros(x.shape, order="F")
        keep = torch.empty(x.size + 4096, dtype=torch.float64, pin_memory=True)
        whole = keep.numpy()
        pinned = whole[1024:1024 + x.size].reshape(x.shape, order="F")   # inside the allocation
        whole[:] = 7.0
        t_plain, t_pinned = _best(s, U, plain), _best(s, U, pinned)
        assert np.array_equal(plain, x) and np.array_equal(pinned, x)
        assert np.all(whole[:1024] == 7.0) and np.all(whole[1024 + x.size:] == 7.0)
        s.upload(P, 2.0 * x)   # and again after another field's
        s._check(s.lib.fen_download(s.h, P, _dp(pinned), x.size))
        assert np.array_equal(pinned, 2.0 * x)
        print(f"download of {8e-6 * x.size:.1f} MB: pageable {1e3 * t_plain:.2f} ms, pinned {1e3 * t_pinned:.2f} ms")
        # staged, both take the same time; direct, 27/57 of it
        assert t_pinned < 0.75 * t_plain, (t_pinned, t_plain)
