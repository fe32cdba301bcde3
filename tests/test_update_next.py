"""1D steps whose corrector also reconstructs and takes the next timestep:
grids around the workgroup's 64 w-cells, every boundary type, orders and
fluxes, odd and even step counts, runs continued after an odd one, and the
largest grid that takes this route -- bit for bit against the oracle."""
import numpy as np
import pytest

import cpu_checkers as cc
from pypde_amd import systems
from pypde_amd.solvers import Solver, pde_solver

REFL = [[1.0, -1.0, 1.0]]


def wave(n, V=3):
    x = (np.arange(n) + 0.5) / n
    rho = 1.0 + 0.3 * np.sin(2 * np.pi * x) + 0.1 * (x > 0.6)
    vel = 0.3 + 0.4 * np.cos(2 * np.pi * x)
    p = 1.0 + 0.25 * np.sin(4 * np.pi * x + 0.3)
    return np.stack([rho, rho * vel, p / 0.4 + 0.5 * rho * vel ** 2], axis=1)


@pytest.mark.gpu
@pytest.mark.parametrize("bc", ["transitive", "periodic", "reflective"])
@pytest.mark.parametrize("n,order,flux", [(8, 3, 0), (61, 3, 0), (62, 3, 1), (63, 2, 0), (64, 6, 0),
                                          (126, 3, 2), (127, 4, 0), (200, 3, 0), (1025, 3, 0)])
def test_steps_equal_the_oracle(n, order, flux, bc):
    u0, steps = wave(n), 7 + n % 2
    names = ["rusanov", "roe", "osher"]
    code = {"transitive": 0, "periodic": 1, "reflective": 2}[bc]
    want, wret, st, rc = cc.oracle_solve("euler1d", u0, 0.05 if n > 8 else 0.4, [1.0], code, order,
                                         ndt=3, max_steps=steps, flux=flux,
                                         reflect=REFL if code == 2 else None)
    assert rc == 0 and st.steps >= 2
    u, out = u0.copy(), {}
    ret = pde_solver(u, 0.05 if n > 8 else 0.4, [1.0], system=systems.source("euler1d"),
                     boundaryTypes=bc, order=order, ndt=3, stiff=False, flux=names[flux],
                     max_steps=steps, stats=out, reflect=REFL if code == 2 else None)
    assert out["steps"] == st.steps
    assert np.array_equal(np.asarray(ret[-1]), want)
    assert np.array_equal(np.asarray(ret)[:-1], wret[:-1])


@pytest.mark.gpu
def test_resident_steps_continue_after_odd_counts():
    n = 130
    sol = Solver(wave(n), [1.0], systems.source("euler1d"), order=3, stiff=False)
    try:
        done = 0
        for k in (1, 3, 2, 5, 1, 4):
            sol.step(k)
            done += k
            want, _, st, rc = cc.oracle_solve("euler1d", wave(n), 1e300, [1.0], 0, 3,
                                              max_steps=done)
            assert rc == 0 and st.steps == done
            assert np.array_equal(sol.state(), want)
    finally:
        sol.close()


@pytest.mark.gpu
@pytest.mark.parametrize("n", [2 ** 17 - 2, 2 ** 17 - 1])
def test_largest_grid_of_the_joint_kernel_and_the_next(n):
    u0 = wave(n)
    want, _, st, rc = cc.oracle_solve("euler1d", u0, 1e300, [1.0], 1, 2, max_steps=3)
    assert rc == 0 and st.steps == 3
    sol = Solver(u0, [1.0], systems.source("euler1d"), order=2, boundaryTypes="periodic",
                 stiff=False)
    try:
        sol.step(3)
        assert np.array_equal(sol.state(), want)
    finally:
        sol.close()


@pytest.mark.gpu
@pytest.mark.parametrize("name,order,stiff,bc", [("ncadvect", 3, False, 1), ("ncadvect", 2, True, 0),
                                                 ("reactive2d", 3, True, 0), ("advect", 4, False, 1)])
def test_source_and_nonconservative_terms(name, order, stiff, bc):
    n, V = 100, systems.SYSTEMS[name]["V"]
    if name == "reactive2d":
        u0 = np.ascontiguousarray(systems.reactive_channel(n, 8, seed=5)[:, 3])
        tf = 1e-2
    else:
        x = (np.arange(n) + 0.5) / n
        u0 = np.stack([1.0 + 0.3 * np.sin(2 * np.pi * (x + 0.2 * v)) for v in range(V)], axis=1)
        tf = 1.0
    want, _, st, rc = cc.oracle_solve(name, u0, tf, [1.0], bc, order, stiff=stiff, max_steps=9)
    assert rc == 0 and st.steps == 9 and np.isfinite(want).all()
    sol = Solver(u0, [1.0], systems.source(name), order=order, stiff=stiff,
                 boundaryTypes=["transitive", "periodic"][bc])
    try:
        got = sol.run(tf, max_steps=9)
        assert got["steps"] == 9
        assert np.array_equal(sol.state(), want)
    finally:
        sol.close()
