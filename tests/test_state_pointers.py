"""set_state and get_state on memory that the runtime allocated: device, pinned
and ordinary host arrays give and take the same state."""
import ctypes as C

import numpy as np
import pytest

from pypde_amd import _capi, systems
from pypde_amd.learned import Dev
from pypde_amd.solvers import Solver


@pytest.mark.gpu
@pytest.mark.parametrize("n", [5, 100000])
def test_state_from_and_to_every_kind_of_memory(n):
    u = np.random.default_rng(n).standard_normal((n, 3))
    sol = Solver(np.zeros((n, 3)), [1.0], systems.source("euler1d"), order=2)
    lib = _capi.lib()

    def exchange(src, dst):
        sol.set_state(np.zeros((n, 3)))
        _capi.check(lib.pypde_set_state(sol.h, C.cast(C.c_void_p(src), _capi.PD)), "set_state")
        assert np.array_equal(sol.state(), u)
        _capi.check(lib.pypde_get_state(sol.h, C.cast(C.c_void_p(dst), _capi.PD)), "get_state")

    print("pageable", flush=True)
    back = np.zeros((n, 3))
    exchange(u.ctypes.data, back.ctypes.data)
    assert np.array_equal(back, u)

    print("device", flush=True)
    src = Dev.from_numpy(u.view(np.float32))
    dst = Dev.from_numpy(np.zeros_like(u).view(np.float32))
    exchange(src.ptr, dst.ptr)
    assert np.array_equal(dst.numpy().view(np.float64), u)

    print("pinned", flush=True)
    hip = C.CDLL("libamdhip64.so.7")     # the one that the library has loaded
    p = C.c_void_p()
    assert hip.hipHostMalloc(C.byref(p), C.c_size_t(2 * u.nbytes), 0) == 0
    pin = np.ctypeslib.as_array(C.cast(p, _capi.PD), (2, n, 3))
    pin[0], pin[1] = u, 0.0
    exchange(p.value, p.value + u.nbytes)
    assert np.array_equal(pin[1], u)
    del pin
    assert hip.hipHostFree(p) == 0
    sol.close()
