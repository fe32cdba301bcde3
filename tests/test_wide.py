"""Systems with more than eight variables (one wavefront per matrix and per
cell): the 17-variable GPR model against the oracle, bitwise."""
import os
import subprocess

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


CHAIN = """
#define PDE_HAS_F 1
PDE_FN void F(double *out, const double *Q, const double *dQ, int d) {
  for (int i = 0; i < NV; i++) {
    double l = i > 0 ? Q[i - 1] : 0.0, r = i < NV - 1 ? Q[i + 1] : 0.0;
    out[i] = (d == 0 ? 0.5 : -0.4) * (l + r) * (1.0 + 0.1 * Q[0]);
  }
}
"""
CHAIN_B = """
#define PDE_HAS_B 1
PDE_FN void B(double *out, const double *Q, int d) {
  for (int i = 0; i < NV * NV; i++) out[i] = 0.0;
  for (int i = 0; i < NV; i++) out[i * NV + i] = 0.2 + 0.1 * d;
  for (int i = 1; i < NV; i++) out[i * NV + i - 1] = out[(i - 1) * NV + i] = 0.05 * Q[0];
}
"""
CHAIN_S = """
#define PDE_HAS_S 1
PDE_FN void S(double *out, const double *Q) {
  for (int i = 0; i < NV; i++) out[i] = -(4.0 * i + 1.0) * Q[i] + 3.0 * Q[(i + 2) % NV] * Q[0];
}
"""
CHAIN_M = """
#define PDE_HAS_M 1
PDE_FN void M(double *out, const double *Q) {
  for (int i = 0; i < NV * NV; i++) out[i] = 0.0;
  for (int i = 0; i < NV; i++) {
    out[i * NV + i] = out[i * NV + i] - (4.0 * i + 1.0);
    out[i * NV + (i + 2) % NV] = out[i * NV + (i + 2) % NV] + 3.0 * Q[0];
    out[i * NV] = out[i * NV] + 3.0 * Q[(i + 2) % NV];
  }
}
"""


@pytest.mark.gpu
@pytest.mark.parametrize("V,parts,ndim,order,stiff", [
    (9, "FSM", 2, 2, True),     # the analytic source Jacobian, two directions
    (9, "BS", 1, 3, True),      # no F: the predictor's B term and the face path integral alone
    (12, "F", 2, 2, False),     # no source, no volume term
    (16, "FBS", 1, 2, False),   # an even matrix size
])
def test_wide_term_combinations_bitwise_equal_to_oracle(tmp_path, monkeypatch, V, parts, ndim,
                                                        order, stiff):
    """Every combination of terms the kernels are specialised for, on a made-up
    chain of V coupled variables; the oracle's callbacks are compiled here from
    the same text."""
    text = {"F": CHAIN, "B": CHAIN_B, "S": CHAIN_S, "M": CHAIN_M}
    src = f"#define NV {V}\n" + "".join(text[p] for p in parts)
    root, build = cc.ROOT, tmp_path / "oracle" / "_build"
    build.mkdir(parents=True)
    pde = tmp_path / "chain.pde"
    pde.write_text(src)
    name = f"chain{V}{parts}"
    subprocess.run(["gcc", "-O2", "-fPIC", "-ffp-contract=off", "-fno-fast-math", "-mfma",
                    "-std=c11", "-shared", "-I" + os.path.join(root, "pypde_amd", "systems"),
                    f'-DPDE_SYSTEM_FILE="{pde}"', "-o", str(build / f"sys_{name}.so"),
                    os.path.join(root, "oracle", "sys_wrap.c"), "-lm"], check=True)
    cc.oracle()   # loaded from the repository's own build
    monkeypatch.setattr(cc, "ROOT", str(tmp_path))
    n = (13,) if ndim == 1 else (6, 7)
    u0 = 1.0 + 0.3 * np.sin(np.arange(np.prod(n) * V).reshape(n + (V,)) ** 1.5)
    L = [1.0] * ndim
    uo, _, st, rc = cc.oracle_solve(name, u0, 1.0, L, 1, order, stiff=stiff, cfl=0.4, max_steps=4)
    assert rc == 0 and np.isfinite(uo).all()
    sol = Solver(u0, L, src, order=order, boundaryTypes="periodic", stiff=stiff, cfl=0.4)
    sg = sol.run(1.0, max_steps=4)
    ug = sol.state()
    sol.close()
    assert sg["steps"] == st.steps and sg["pred_iters"] == st.pred_iters
    assert np.array_equal(ug, uo)
