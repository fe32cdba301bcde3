"""The stiff predictor's schedules (one kernel; the split with either cold
pass): the registers and LDS that decide how many of their wavefronts a
compute unit holds, and the same bits and counts from each, as the oracle's,
where F of all time nodes is staged at once and where one at a time."""
import re
import subprocess

import numpy as np
import pytest

import cpu_checkers as cc
from pypde_amd import _capi, systems
from pypde_amd.solvers import Solver


def kernels(tmp_path, monkeypatch, system, N, stiff=True):
    """{kernel: (registers, spilled, LDS bytes)} of the plain 2D predictor."""
    monkeypatch.setenv("PYPDE_HIP_CACHE", str(tmp_path))
    s = systems.SYSTEMS[system]
    _capi.compile_only(systems.source(system) + "/* footprint */", s["F"], s["B"], s["S"], 2, N,
                       s["V"], stiff=stiff, use_M=s["M"])
    out = {}
    for f in tmp_path.glob("*.hsaco"):
        notes = subprocess.run(["/opt/rocm/llvm/bin/llvm-readelf", "--notes", str(f)], check=True,
                               capture_output=True, text=True).stdout
        if "k_mlp_guess" in notes:
            continue
        for block in notes.split("- .agpr_count")[1:]:
            def num(key):
                return int(re.search(rf"\.{key}:\s+(\d+)", block).group(1))
            name = re.search(r"\.name:\s+(k_\w+)", block).group(1)
            out[name] = (num("vgpr_count"), num("vgpr_spill_count"),
                         num("group_segment_fixed_size"))
    return out


@pytest.mark.parametrize("order", [3, 4])
def test_footprint_of_the_reactive_predictor(order, tmp_path, monkeypatch):
    k = kernels(tmp_path, monkeypatch, "reactive2d", order)
    regs, spilled, lds = k["k_predictor_static"]
    # two wavefronts per SIMD of 512 registers; eight per compute unit of 160 KB
    assert regs <= 256 and spilled == 0 and lds * 8 <= 160 * 1024
    # twelve wavefronts of the cold pass per compute unit
    assert k["k_predictor_cold"][2] * 12 <= 160 * 1024


@pytest.mark.parametrize("system,order", [("euler2d", 5), ("reactive2d", 4)])
def test_footprint_of_the_picard_predictor(system, order, tmp_path, monkeypatch):
    regs, spilled, _ = kernels(tmp_path, monkeypatch, system, order, False)["k_predictor_static"]
    assert regs <= 256 and spilled <= 2   # two wavefronts per SIMD


def start(system, ndim):
    if system == "reactive2d":
        u = systems.reactive_channel(40, 12, seed=6)
        return u if ndim == 2 else np.ascontiguousarray(u[:, 3])
    return np.ascontiguousarray(systems.euler2d_modes(19, seed=2)[:, :14])


@pytest.mark.gpu
@pytest.mark.parametrize("system,ndim,order", [
    ("reactive2d", 2, 3),    # N V = 15: all time nodes at once
    ("euler2d", 2, 4),       # 16: all at once, no source
    ("reactive2d", 2, 4),    # 20: one at a time
    ("reactive2d", 1, 4),    # 20 in 1D: all at once
    ("reactive2d", 2, 6),    # 30: one at a time, one cell per wavefront
])
def test_schedules_equal_the_oracle(system, ndim, order, monkeypatch):
    u0 = start(system, ndim)
    L = [n / 1024 if system == "reactive2d" else 1.0 for n in u0.shape[:-1]]
    steps = 3 if order == 6 else 5
    want, _, st, rc = cc.oracle_solve(system, u0, 1.0, L, 1, order, stiff=True, max_steps=steps)
    assert rc == 0 and st.steps == steps and np.isfinite(want).all()
    runs = []
    for schedule, label in ((0, "static"), (2, "split"), (3, "split3")):
        print(system, ndim, order, label, flush=True)
        monkeypatch.setenv("PYPDE_TUNE_FORCE", f"0,0,1,{schedule}")
        sol = Solver(u0, L, systems.source(system), order=order, boundaryTypes="periodic",
                     stiff=True)
        got = sol.run(1.0, max_steps=steps)
        assert sol.tuning()["predictor"] == label
        assert np.array_equal(sol.state(), want), label
        sol.close()
        runs.append([got[k] for k in ("steps", "pred_iters", "pred_cells", "pred_maxit",
                                      "pred_capped", "pred_node_full", "pred_node_short")])
    assert runs[0] == runs[1] == runs[2]
    assert runs[0][:5] == [st.steps, st.pred_iters, st.pred_cells, st.pred_maxit, st.pred_capped]
