"""The face flux with a point's eigenvalue problems split over wavefronts
equals the one-thread-per-point kernels bit for bit, for every flux and term,
on grids whose faces leave the last workgroups ragged."""
import os

import numpy as np
import pytest

from pypde_amd import systems
from pypde_amd.solvers import Solver


def _run(variant, u0, L, **kw):
    os.environ["PYPDE_TUNE_FORCE"] = f"0,{variant},1,0"
    try:
        sol = Solver(u0, L, order=3, boundaryTypes="periodic", **kw)
        sol.run(1.0, max_steps=4)
        u = sol.state()
        sol.close()
    finally:
        del os.environ["PYPDE_TUNE_FORCE"]
    return u


@pytest.mark.gpu
@pytest.mark.parametrize("system,flux,ndim", [
    ("euler2d", "rusanov", 2), ("euler2d", "roe", 2), ("euler2d", "osher", 2),
    ("ns2d", "rusanov", 2), ("ns2d", "osher", 2), ("advdiff", "rusanov", 1),
    ("euler1d", "osher", 1), ("ncadvect", "rusanov", 2)])
def test_split_flux_equals_unsplit(system, flux, ndim):
    V = systems.SYSTEMS[system]["V"]
    if system in ("euler2d", "ns2d"):
        u0 = np.ascontiguousarray(systems.euler2d_modes(23, seed=3)[:17])
    elif system == "euler1d":
        u0 = systems.sod1d(45)
    else:
        n = (17, 23)[:ndim]
        u0 = 1.0 + 0.3 * np.sin(np.arange(np.prod(n) * V).reshape(n + (V,)))
    ref = _run(0, u0, [1.0] * ndim, system=systems.source(system), flux=flux)
    assert np.isfinite(ref).all()
    for variant in (1, 2):
        assert np.array_equal(_run(variant, u0, [1.0] * ndim, system=systems.source(system),
                                   flux=flux), ref), variant
