"""The stiff Newton with source terms that couple the variables both ways: the
correction is the exact solve of the linear system it says it is, so a linear
source takes few iterations at any strength, and the iterate is the fixed
point."""
import os
import subprocess

import numpy as np
import pytest

import cpu_checkers as cc
from pypde_amd.solvers import Solver

# a linear source whose matrix is full, not symmetric and stable
LINEAR = """
#define PDE_HAS_F 1
#define PDE_HAS_S 1
PDE_FN void F(double *out, const double *Q, const double *dQ, int d) {
  for (int i = 0; i < NV; i++) out[i] = (d == 0 ? 0.6 : -0.4) * Q[i];
}
PDE_FN void S(double *out, const double *Q) {
  for (int i = 0; i < NV; i++) {
    double a = 0.0;
    for (int j = 0; j < NV; j++) a += (j == i ? -1.0 - 0.3 * i : 0.4 / (1 + i + 2 * j)) * Q[j];
    out[i] = STRENGTH * a;
  }
}
"""


def text(V, strength):
    return f"#define NV {V}\n#define STRENGTH {strength}\n" + LINEAR


def build(name, source, tmp_path, monkeypatch):
    root, out = cc.ROOT, tmp_path / "oracle" / "_build"
    out.mkdir(parents=True, exist_ok=True)
    pde = tmp_path / f"{name}.pde"
    pde.write_text(source)
    subprocess.run(["gcc", "-O2", "-fPIC", "-ffp-contract=off", "-fno-fast-math", "-mfma",
                    "-std=c11", "-shared", "-I" + os.path.join(root, "pypde_amd", "systems"),
                    f'-DPDE_SYSTEM_FILE="{pde}"', "-o", str(out / f"sys_{name}.so"),
                    os.path.join(root, "oracle", "sys_wrap.c"), "-lm"], check=True)
    cc.oracle()   # loaded from the repository's own build
    monkeypatch.setattr(cc, "ROOT", str(tmp_path))


def field(shape, V):
    return 1.0 + 0.3 * np.sin(0.7 * np.arange(np.prod(shape) * V)).reshape(shape + (V,))


CASES = [(5, (24,), 3, 30.0), (5, (24,), 3, 1000.0), (2, (9, 8), 2, 200.0), (8, (7, 6), 3, 100.0),
         (4, (20,), 4, 300.0), (9, (20,), 2, 200.0), (12, (5, 6), 2, 1000.0), (17, (18,), 3, 30.0)]


@pytest.mark.parametrize("V,shape,order,strength", CASES)
def test_oracle_iterations_of_a_linear_source(V, shape, order, strength, tmp_path, monkeypatch):
    """The frozen Jacobian holds the source exactly and leaves out the flux
    alone, whose share falls with the strength: a few corrections suffice."""
    name = f"lin{V}_{int(strength)}"
    build(name, text(V, strength), tmp_path, monkeypatch)
    _, _, st, rc = cc.oracle_solve(name, field(shape, V), 1.0, [1.0] * len(shape), 1, order,
                                   stiff=True, cfl=0.5, max_steps=3)
    per_cell = st.pred_iters / st.pred_cells
    print(V, strength, "iterations per cell", per_cell, "most", st.pred_maxit)
    assert rc == 0 and st.pred_capped == 0
    # one correction per order in the flux, one that confirms, one for the
    # finite-difference Jacobian
    assert per_cell <= 2 * order + 2, per_cell


@pytest.mark.gpu
@pytest.mark.parametrize("V,shape,order,strength", CASES)
def test_gpu_equals_the_oracle(V, shape, order, strength, tmp_path, monkeypatch):
    name = f"lin{V}_{int(strength)}"
    build(name, text(V, strength), tmp_path, monkeypatch)
    u0, L = field(shape, V), [1.0] * len(shape)
    want, _, st, rc = cc.oracle_solve(name, u0, 1.0, L, 1, order, stiff=True, cfl=0.5, max_steps=3)
    assert rc == 0 and np.isfinite(want).all()
    print(V, shape, order, flush=True)
    sol = Solver(u0, L, text(V, strength), order=order, boundaryTypes="periodic", stiff=True,
                 cfl=0.5)
    got = sol.run(1.0, max_steps=3)
    u = sol.state()
    sol.close()
    assert got["steps"] == 3 and got["pred_iters"] == st.pred_iters
    assert got["pred_node_full"] > 0
    assert np.array_equal(u, want)
