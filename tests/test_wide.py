"""Systems with more than eight variables (one wavefront per matrix and per
cell): the 17-variable GPR model against the oracle, bitwise."""
import numpy as np
import pytest

import cpu_checkers as cc
from pypde_amd import systems
from pypde_amd.solvers import Ensemble, Solver

# (ndim, order, stiff, b_quirk): both directions' B and F, time nodes staged
# together and one by one (order 6 in 2D), odd node counts for the half
# wavefronts, orders whose p(A) takes one and several products
CONFIGS = [(1, 1, True, 0), (1, 4, True, 0), (2, 2, True, 0), (2, 3, False, 1), (2, 6, False, 0)]


def _state(ndim):
    """A blast in a corner with sheared velocities: every variable varies."""
    n = (19,) if ndim == 1 else (7, 6)
    u = np.zeros(n + (17,))
    for i in np.ndindex(*n):
        r = 1.0 if sum(i) < sum(n) / 2 - 1 else 0.4
        u[i] = systems.gpr_state(r, r, (0.1 * r, -0.05 * sum(i) / 10, 0.02))
        u[i][5:14] += 0.01 * np.sin(np.arange(9) + sum(i))
        u[i][14:17] = 0.01 * np.cos(np.arange(3) + sum(i))
    return u


@pytest.mark.gpu
@pytest.mark.parametrize("ndim,order,stiff,quirk", CONFIGS)
def test_wide_systems_bitwise_equal_to_oracle(ndim, order, stiff, quirk):
    u0 = _state(ndim)
    steps = 2 if order == 6 else 6
    L = [1.0] * ndim
    uo, _, st, rc = cc.oracle_solve("gpr", u0, 1.0, L, 0, order, stiff=stiff, cfl=0.5,
                                    b_quirk=quirk, max_steps=steps)
    assert rc == 0 and np.isfinite(uo).all()
    sol = Solver(u0, L, systems.source("gpr"), order=order, stiff=stiff, cfl=0.5,
                 b_quirk=bool(quirk))
    sg = sol.run(1.0, max_steps=steps)
    ug = sol.state()
    sol.close()
    assert sg["steps"] == st.steps and sg["pred_iters"] == st.pred_iters
    assert np.array_equal(ug, uo)


@pytest.mark.gpu
def test_wide_ensemble_equals_single_runs():
    """Batched launches: each member bitwise equal to its own run."""
    src = systems.source("gpr")
    grids = [systems.gpr_riemann(n) for n in (9, 40, 23)]
    ens = Ensemble(grids, [[1.0]] * 3, src, order=2, stiff=True, cfl=0.6)
    ens.run(1.0, max_steps=5)
    for i, u in enumerate(grids):
        sol = Solver(u, [1.0], src, order=2, stiff=True, cfl=0.6)
        sol.run(1.0, max_steps=5)
        assert np.array_equal(ens.state(i), sol.state())
        sol.close()
    ens.close()
