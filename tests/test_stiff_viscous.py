"""The stiff predictor with a viscous F, whose face gradients every build of it
has to write: one kernel, and the split with either cold pass, on single grids
and in batched ensembles, bit for bit against the oracle.  The source acts in
part of the domain only, so both passes of the split take cells."""
import os
import re
import subprocess

import numpy as np
import pytest

import cpu_checkers as cc
from pypde_amd import _capi
from pypde_amd.solvers import Ensemble, Solver

SRC = """
#define PDE_HAS_F 1
#define PDE_HAS_S 1
#define PDE_SECOND_ORDER 1
PDE_FN void F(double *out, const double *Q, const double *dQ, int d) {
  const double a = d == 0 ? 0.8 : -0.5;
  out[0] = a * Q[0] - 0.01 * dQ[2 * d];
  out[1] = a * Q[1] + 0.1 * Q[0] - 0.02 * Q[0] * dQ[2 * d + 1];
}
PDE_FN void S(double *out, const double *Q) {
  const double k = Q[0] > 1.0 ? 60.0 * (Q[0] - 1.0) : 0.0;
  out[0] = -k * Q[1];
  out[1] = -2.0 * k * Q[0];
}
"""


def field(shape):
    i = np.arange(np.prod(shape) * 2).reshape(shape + (2,))
    return 1.0 + 0.3 * np.sin(0.37 * i)


@pytest.mark.parametrize("ndim", [1, 2])
def test_split_passes_take_the_gradient_buffer(ndim, tmp_path, monkeypatch):
    """Every predictor kernel of a viscous system has the same number of
    writable buffers and one more for the split's list of cells."""
    monkeypatch.setenv("PYPDE_HIP_CACHE", str(tmp_path))
    _capi.compile_only(SRC + f"/* {ndim} */", True, False, True, ndim, 2, 2, stiff=True, second=True)
    notes = ""
    for f in tmp_path.glob("*.hsaco"):
        notes += subprocess.run(["/opt/rocm/llvm/bin/llvm-readelf", "--notes", str(f)], check=True,
                                capture_output=True, text=True).stdout
    buffers = {}
    for block in notes.split("- .agpr_count")[1:]:
        name = re.search(r"\.name:\s+(k_\w+)", block).group(1)
        buffers.setdefault(name, block.count("global_buffer"))
    # wh, guess, tr, vol, qh, st, trd; the split has no guess and the list of cells
    assert buffers["k_predictor_static"] == 7
    for name in ("k_predictor_cold", "k_predictor_cold3", "k_predictor_hot"):
        assert buffers[name] == 7, name


def oracle_system(tmp_path, monkeypatch, name, text):
    root, build = cc.ROOT, tmp_path / "oracle" / "_build"
    build.mkdir(parents=True)
    pde = tmp_path / f"{name}.pde"
    pde.write_text(text)
    subprocess.run(["gcc", "-O2", "-fPIC", "-ffp-contract=off", "-fno-fast-math", "-mfma",
                    "-std=c11", "-shared", "-I" + os.path.join(root, "pypde_amd", "systems"),
                    f'-DPDE_SYSTEM_FILE="{pde}"', "-o", str(build / f"sys_{name}.so"),
                    os.path.join(root, "oracle", "sys_wrap.c"), "-lm"], check=True)
    cc.oracle()   # loaded from the repository's own build
    monkeypatch.setattr(cc, "ROOT", str(tmp_path))


@pytest.mark.gpu
@pytest.mark.parametrize("shape,order", [((37,), 3), ((13, 11), 2), ((9, 10), 3)])
def test_every_schedule_equals_the_oracle(shape, order, tmp_path, monkeypatch):
    name = "stiffvisc"
    oracle_system(tmp_path, monkeypatch, name, SRC)
    u0, L = field(shape), [1.0] * len(shape)
    want, _, st, rc = cc.oracle_solve(name, u0, 1.0, L, 1, order, stiff=True, cfl=0.4, max_steps=4,
                                      second=True)
    assert rc == 0 and np.isfinite(want).all()
    for schedule, label in ((0, "static"), (2, "split"), (3, "split3")):
        print(shape, order, label, flush=True)
        monkeypatch.setenv("PYPDE_TUNE_FORCE", f"0,0,1,{schedule}")
        sol = Solver(u0, L, SRC, order=order, boundaryTypes="periodic", stiff=True, cfl=0.4)
        got = sol.run(1.0, max_steps=4)
        u, used = sol.state(), sol.tuning()["predictor"]
        sol.close()
        assert used == label and got["steps"] == 4
        assert got["pred_iters"] == st.pred_iters
        assert got["pred_node_full"] > 0 and got["pred_node_short"] > 0
        assert np.array_equal(u, want), label


@pytest.mark.gpu
def test_batched_members_equal_single_runs(monkeypatch):
    grids = [field(s) for s in ((9, 10), (6, 14), (12, 5))]
    for schedule in (0, 2, 3):
        print("ensemble", schedule, flush=True)
        monkeypatch.setenv("PYPDE_TUNE_FORCE", f"0,0,1,{schedule}")
        ens = Ensemble(grids, [[1.0, 1.0]] * 3, SRC, order=3, boundaryTypes="periodic", stiff=True,
                       cfl=0.4)
        ens.run(1.0, max_steps=3)
        for i, u in enumerate(grids):
            sol = Solver(u, [1.0, 1.0], SRC, order=3, boundaryTypes="periodic", stiff=True, cfl=0.4)
            sol.run(1.0, max_steps=3)
            assert np.array_equal(ens.state(i), sol.state()), (schedule, i)
            sol.close()
        ens.close()
