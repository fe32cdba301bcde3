"""The step's last workgroup (which turns the wave-speed maximum into dt and
advances the clock) with one ticket and with two levels of tickets: grids of
128, 129, 193 and 256 workgroups, bit for bit against the oracle."""
import numpy as np
import pytest

import cpu_checkers as cc
from pypde_amd import systems
from pypde_amd.solvers import pde_solver


@pytest.mark.gpu
@pytest.mark.parametrize("n", [128 * 256 - 2, 128 * 256 - 1, 128 * 256, 128 * 256 + 1,
                               192 * 256 + 1, 256 * 256])
def test_steps_around_the_second_ticket_level(n):
    x = (np.arange(n) + 0.5) / n
    u = np.zeros((n, 3))
    rho = 1.0 + 0.3 * np.sin(2 * np.pi * 7 * x)
    vel = 0.4 + 0.2 * np.cos(2 * np.pi * 3 * x)
    p = 1.0 + 0.25 * np.sin(2 * np.pi * 5 * x + 0.3)
    u[:, 0], u[:, 1], u[:, 2] = rho, rho * vel, p / 0.4 + 0.5 * rho * vel ** 2
    tf = 3.2 * 0.9 / n / 8.0                      # a few steps
    want, _, st, rc = cc.oracle_solve("euler1d", u, tf, [1.0], 1, 2)
    assert rc == 0 and st.steps >= 2
    out = pde_solver(u, tf, [1.0], system=systems.source("euler1d"), boundaryTypes="periodic",
                     cfl=0.9, order=2, stiff=False, flux="rusanov", ndt=1)
    assert np.array_equal(np.asarray(out[-1]).reshape(want.shape), want)
