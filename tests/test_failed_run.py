"""A run that fails between two 1D steps: the state lies in the second buffer
every other step, and the calls that follow have to find it.  The failure
comes from the host, out of a stand-in for a HIP call that refuses one call
and otherwise passes it on."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SHIM = """
#define _GNU_SOURCE
#include <dlfcn.h>
static int launches = -1, copies = -1;
void refuse(int launch, int copy) { launches = launch; copies = copy; }
typedef int (*launch_t)(void *, unsigned, unsigned, unsigned, unsigned, unsigned, unsigned, unsigned,
                        void *, void **, void **);
typedef int (*copy_t)(void *, const void *, unsigned long, int, void *);
int hipModuleLaunchKernel(void *f, unsigned gx, unsigned gy, unsigned gz, unsigned bx, unsigned by,
                          unsigned bz, unsigned lds, void *s, void **a, void **e) {
  static launch_t real;
  if (!real) real = (launch_t)dlsym(RTLD_NEXT, "hipModuleLaunchKernel");
  if (launches >= 0 && launches-- == 0) return 1;
  return real(f, gx, gy, gz, bx, by, bz, lds, s, a, e);
}
int hipMemcpyAsync(void *d, const void *s, unsigned long n, int kind, void *stream) {
  static copy_t real;
  if (!real) real = (copy_t)dlsym(RTLD_NEXT, "hipMemcpyAsync");
  if (copies >= 0 && copies-- == 0) return 1;
  return real(d, s, n, kind, stream);
}
"""

CHILD = """
import ctypes, os, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
sys.path.insert(0, sys.argv[2])
os.environ["PYPDE_TUNE"] = "0"
import numpy as np
from pypde_amd import systems
from pypde_amd._capi import PypdeError
from pypde_amd.solvers import Solver

u0 = systems.sod1d(300)
u0[:, 1] += 0.1 * np.sin(np.arange(300))
make = lambda: Solver(u0, [1.0], systems.source("euler1d"), order=3)
ref, states = make(), [u0.copy()]
for _ in range(12):
    ref.step(1)
    states.append(ref.state())

def broken(launch, copy):
    sol = make()
    shim.refuse(launch, copy)
    try:
        sol.step(12)
    except PypdeError as e:
        print("refused", launch, copy, e, flush=True)
    else:
        raise SystemExit("the refused call went unnoticed")
    shim.refuse(-1, -1)
    return sol

# a step launches predictor, face flux and the joint corrector; the first one
# reconstruction and timestep before them.  Copies of step(): state down, state
# up, and one after each chunk of steps
for launch, copy in [(n, -1) for n in range(4, 13)] + [(-1, 2), (-1, 3)]:
    done = (launch - 2) // 3 if launch >= 0 else (4 if copy == 2 else 12)
    sol = broken(launch, copy)
    assert np.array_equal(sol.state(), states[done]), (launch, copy, "state")
    if done < 12:
        sol.step(12 - done)
        assert np.array_equal(sol.state(), states[12]), (launch, copy, "more steps")
    sol.close()
    sol = broken(launch, copy)
    sol.set_state(u0)
    sol.run(1e300, max_steps=5)
    assert np.array_equal(sol.state(), states[5]), (launch, copy, "another state")
    sol.close()
    sol = broken(launch, copy)
    sol.run(1e300, max_steps=1)
    one = make()
    one.set_state(states[done])
    one.run(1e300, max_steps=1)
    assert np.array_equal(sol.state(), one.state()), (launch, copy, "another run")
    sol.close()
    one.close()
print("all found", flush=True)
"""


@pytest.mark.gpu
def test_calls_after_a_failed_run_find_the_state(tmp_path):
    src, so = tmp_path / "shim.c", str(tmp_path / "libshim.so")
    src.write_text(SHIM)
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-o", so, str(src), "-Wl,--no-as-needed",
                    f"-L{rocm}/lib", f"-Wl,-rpath,{rocm}/lib", "-lamdhip64", "-ldl"], check=True)
    child = tmp_path / "child.py"
    child.write_text(CHILD)
    r = subprocess.run([sys.executable, "-u", str(child), so, ROOT], capture_output=True, text=True,
                       timeout=100)
    print(r.stdout[-3000:], r.stderr[-2000:], flush=True)
    assert r.returncode == 0 and "all found" in r.stdout
