"""Systems above eight variables have two forms of every kernel, one wavefront or
one lane per matrix and per cell; large grids take the second.  Both against the
oracle bit for bit, over every term, and the line between them."""
import os
import subprocess

import numpy as np
import pytest

import cpu_checkers as cc
from pypde_amd import systems
from pypde_amd.solvers import Ensemble, Solver
from test_wide import CHAIN, CHAIN_B, CHAIN_M, CHAIN_S

CSRC = os.path.join(cc.ROOT, "pypde_amd", "csrc")
TEXT = {"F": CHAIN, "B": CHAIN_B, "S": CHAIN_S, "M": CHAIN_M}


def source(V, parts):
    return f"#define NV {V}\n" + "".join(TEXT[p] for p in parts)


def build(name, text, tmp_path, monkeypatch):
    out = tmp_path / "oracle" / "_build"
    out.mkdir(parents=True, exist_ok=True)
    pde = tmp_path / f"{name}.pde"
    pde.write_text(text)
    subprocess.run(["gcc", "-O2", "-fPIC", "-ffp-contract=off", "-fno-fast-math", "-mfma",
                    "-std=c11", "-shared", "-I" + os.path.join(cc.ROOT, "pypde_amd", "systems"),
                    f'-DPDE_SYSTEM_FILE="{pde}"', "-o", str(out / f"sys_{name}.so"),
                    os.path.join(cc.ROOT, "oracle", "sys_wrap.c"), "-lm"], check=True)
    cc.oracle()   # loaded from the repository's own build
    monkeypatch.setattr(cc, "ROOT", str(tmp_path))


def test_line_between_the_forms(tmp_path):
    """More variables move it to larger grids, never back."""
    main = tmp_path / "line.cpp"
    main.write_text('#include <cstdio>\n#include "tune.h"\n'
                    "int main() { for (int v = 9; v <= 17; v++)"
                    ' printf("%ld\\n", pypde::wide_matrices(v)); }\n')
    exe = str(tmp_path / "line")
    subprocess.run(["g++", "-std=c++17", "-I", CSRC, "-o", exe, str(main)], check=True)
    out = subprocess.run([exe], check=True, capture_output=True, text=True).stdout
    line = [int(x) for x in out.split()]
    assert len(line) == 9 and line == sorted(line)
    # within the measured brackets of the face flux's crossing, in matrices
    assert line[0] < 80_000 and 8_000 <= line[3] < 80_000 and 80_000 <= line[8] < 400_000


@pytest.mark.gpu
@pytest.mark.parametrize("V,parts,ndim,order,stiff", [
    (9, "FSM", 2, 2, True), (9, "BS", 1, 3, True), (9, "FBS", 2, 1, False), (10, "F", 1, 4, False),
    (12, "F", 2, 2, False), (14, "FS", 1, 2, True)])
def test_lane_form_equals_the_oracle(V, parts, ndim, order, stiff, tmp_path, monkeypatch):
    text, name = source(V, parts), f"lane{V}{parts}"
    build(name, text, tmp_path, monkeypatch)
    n = (71,) if ndim == 1 else (9, 13)
    u0 = 1.0 + 0.3 * np.sin(np.arange(np.prod(n) * V).reshape(n + (V,)) ** 1.5)
    L = [1.0] * ndim
    want, _, st, rc = cc.oracle_solve(name, u0, 1.0, L, 1, order, stiff=stiff, cfl=0.4, max_steps=4)
    assert rc == 0 and np.isfinite(want).all()
    for form in ("0", "1"):
        print(V, parts, ndim, order, "form", form, flush=True)
        monkeypatch.setenv("PYPDE_WIDE", form)
        sol = Solver(u0, L, text, order=order, boundaryTypes="periodic", stiff=stiff, cfl=0.4)
        got = sol.run(1.0, max_steps=4)
        assert got["steps"] == st.steps and got["pred_iters"] == st.pred_iters
        assert np.array_equal(sol.state(), want), form
        sol.close()


@pytest.mark.gpu
def test_lane_form_of_the_17_variable_model(monkeypatch):
    u0 = systems.gpr_riemann(70)
    u0[:, 5:14] *= 1 + 0.02 * np.sin(0.3 * np.arange(70)[:, None] + np.arange(9))
    want, _, st, rc = cc.oracle_solve("gpr", u0, 1.0, [1.0], 0, 2, cfl=0.6, b_quirk=1, max_steps=6)
    assert rc == 0 and np.isfinite(want).all()
    monkeypatch.setenv("PYPDE_WIDE", "0")
    sol = Solver(u0, [1.0], systems.source("gpr"), order=2, cfl=0.6, b_quirk=True)
    got = sol.run(1.0, max_steps=6)
    assert got["steps"] == 6 and got["pred_iters"] == st.pred_iters
    assert np.array_equal(sol.state(), want)
    sol.close()


@pytest.mark.gpu
def test_members_of_an_ensemble_share_a_form(monkeypatch):
    """The members' matrices count together, so that small ones run the form of
    the launch they share; each equals its single run in either form."""
    text = source(9, "FS")
    sizes = (300, 40, 700, 15)
    grids = [1.0 + 0.3 * np.sin(0.01 * np.arange(n * 9).reshape(n, 9)) for n in sizes]
    ens = Ensemble(grids, [[1.0]] * 4, text, order=3, boundaryTypes="periodic", cfl=0.4)
    # 2 * 3 * (n + 1) matrices each; 6,354 together stay below the line, so force
    # the other form as well
    ens.run(1.0, max_steps=3)
    small = [ens.state(i) for i in range(4)]
    ens.close()
    monkeypatch.setenv("PYPDE_WIDE", "0")
    ens = Ensemble(grids, [[1.0]] * 4, text, order=3, boundaryTypes="periodic", cfl=0.4)
    ens.run(1.0, max_steps=3)
    for i, u in enumerate(grids):
        sol = Solver(u, [1.0], text, order=3, boundaryTypes="periodic", cfl=0.4)
        sol.run(1.0, max_steps=3)
        assert np.array_equal(ens.state(i), sol.state()) and np.array_equal(small[i], sol.state())
        sol.close()
    ens.close()


@pytest.mark.gpu
def test_a_large_grid_runs_at_the_lane_forms_rate():
    """Nine variables on 100,000 cells: the wavefront form takes some 10 ms a step,
    the lane form under one."""
    n = 100_000
    x = (np.arange(n) + 0.5) / n
    u0 = np.stack([1.0 + 0.3 * np.sin(2 * np.pi * (x + 0.1 * v)) for v in range(9)], axis=1)
    sol = Solver(u0, [1.0], source(9, "F"), order=2, boundaryTypes="periodic", cfl=0.5)
    sol.run(1e300, max_steps=4)
    sol.set_state(u0)
    ms = min(sol.run(1e300, max_steps=4)["ms_loop"] / 4 for _ in range(3))
    sol.close()
    print("ms a step", ms, flush=True)
    assert ms < 4.0
