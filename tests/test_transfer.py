"""Staged host copies, kept modules and streams: sizes around the 1 MB chunks
and the per-thread slices, several threads at once, and giving everything idle
back in between."""
import threading

import numpy as np
import pytest

from pypde_amd import _capi, systems, weno_solver
from pypde_amd.solvers import Solver

pytestmark = pytest.mark.gpu

MB = 1 << 20
# bytes of a one-variable state: below and at one chunk, one double past it,
# two slices of unequal length, eight slices with several chunks each
SIZES = [8, MB - 8, MB, MB + 8, 2 * MB + 4096 + 8, 21 * MB + 24]


def _round_trip(n, seed):
    u = np.random.default_rng(seed).standard_normal((n, 1))
    sol = Solver(u, [1.0], systems.source("advect"), order=3)
    back = sol.state()
    sol.close()
    assert np.array_equal(back, u)


@pytest.mark.parametrize("size", SIZES)
def test_state_round_trip(size):
    _round_trip(size // 8, size)


def test_threads_and_release():
    errors = []

    def work(k):
        try:
            for i in range(3):
                _round_trip(SIZES[(k + i) % len(SIZES)] // 8, 10 * k + i)
                _capi.lib().pypde_release_idle()
        except Exception as e:  # reported by the main thread
            errors.append(e)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(6)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors


@pytest.mark.parametrize("shape,order", [((64 + 4, 1 + 4, 1), 3), ((65 + 4,), 3), ((9, 11, 9), 4),
                                         ((130, 3, 2), 2)])
def test_rows_of_the_reconstruction(shape, order):
    """weno_solver's row layout at cell counts off the transposition's 64 and
    plane counts on either side of its slabs of 32: every variable on its own
    gives the same rows."""
    u = np.random.default_rng(1).standard_normal(shape if len(shape) > 1 else shape + (3,))
    full = weno_solver(u, order)
    for v in range(u.shape[-1]):
        one = weno_solver(np.ascontiguousarray(u[..., v:v + 1]), order)
        assert np.array_equal(full[..., v:v + 1], one)
