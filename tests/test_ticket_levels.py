"""The steps' tickets at the change from one level to two (128 workgroups): the
joint 1D kernel's (64 w-cells per workgroup) and, on the routes that keep the
separate kernels, the timestep's and the corrector's over several steps, each
of which finds the tickets as the one before left them.  Bit for bit against
the oracle."""
import numpy as np
import pytest

import cpu_checkers as cc
from pypde_amd import systems
from pypde_amd.solvers import Solver


def wave(n):
    x = (np.arange(n) + 0.5) / n
    rho = 1.0 + 0.3 * np.sin(2 * np.pi * 7 * x)
    vel = 0.4 + 0.2 * np.cos(2 * np.pi * 3 * x)
    p = 1.0 + 0.25 * np.sin(2 * np.pi * 5 * x + 0.3)
    return np.stack([rho, rho * vel, p / 0.4 + 0.5 * rho * vel ** 2], axis=1)


def check(u0, L, system, order, steps, **kw):
    want, _, st, rc = cc.oracle_solve(system, u0, 1e300, L, 1, order, max_steps=steps)
    assert rc == 0 and st.steps == steps
    sol = Solver(u0, L, systems.source(system), order=order, boundaryTypes="periodic", **kw)
    try:
        assert sol.run(1e300, max_steps=steps)["steps"] == steps
        assert np.array_equal(sol.state(), want)
    finally:
        sol.close()


@pytest.mark.gpu
@pytest.mark.parametrize("n", [64 * 128 - 2, 64 * 128 - 1, 64 * 193 - 2])
def test_joint_kernel(n):
    check(wave(n), [1.0], "euler1d", 2, 6)


@pytest.mark.gpu
@pytest.mark.parametrize("route", ["use_graph", "profile"])
@pytest.mark.parametrize("n", [256 * 128 - 2, 256 * 128 - 1, 256 * 128, 256 * 128 + 1])
def test_separate_kernels(n, route, monkeypatch):
    # one thread per cell: 256 w-cells (timestep) and cells (corrector) per workgroup
    monkeypatch.setenv("PYPDE_TUNE_FORCE", "0,0,0,0")
    check(wave(n), [1.0], "euler1d", 2, 6, **{route: True})


@pytest.mark.gpu
@pytest.mark.parametrize("ny", [64, 65])
@pytest.mark.parametrize("rows", [1, 2])
def test_corrector_rows(rows, ny, monkeypatch):
    # one variable and `rows` x-rows per thread: 4 * (128 rows / rows) * ny threads
    monkeypatch.setenv("PYPDE_TUNE_FORCE", f"0,0,{rows},0")
    nx = 128 * rows
    u0 = np.ascontiguousarray(np.tile(systems.euler2d_modes(64, seed=8), (4, 2, 1))[:nx, :ny])
    check(u0, [1.0, ny / nx], "euler2d", 2, 5)
