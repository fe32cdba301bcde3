"""weno_solver's rows formed in spans of the result (256 MB at a time): a result
of several spans equals those of its parts, and the device memory beside the
result's own stays a span."""
import ctypes as C
import threading

import numpy as np
import pytest

from pypde_amd import _capi, weno_solver


@pytest.mark.gpu
@pytest.mark.parametrize("shape,order", [((6_000_001, 3), 2), ((1203, 1801, 2), 3)])
def test_spans_of_the_result_join(shape, order):
    u = 1.0 + np.random.default_rng(3).random(shape)
    full = weno_solver(u, order)
    assert full.nbytes > 2 ** 28
    g = 2 * (order - 1)
    n = full.shape[0]
    cuts = [0, 1000, n // 2 - 37, n // 2 + 500, n - 700, n]
    for a, b in zip(cuts[:-1:2], cuts[1::2]):
        assert np.array_equal(weno_solver(np.ascontiguousarray(u[a:b + g]), order), full[a:b])
    # the rows on either side of where spans meet
    cells = int(np.prod(full.shape[:len(shape) - 1]))
    span = 2 ** 25 // (full.size // cells) // 64 * 64
    for c in range(span, cells, span):
        row = c // (full.shape[1] if len(shape) == 3 else 1)
        a, b = max(0, row - 200), min(n, row + 200)
        assert np.array_equal(weno_solver(np.ascontiguousarray(u[a:b + g]), order), full[a:b])


@pytest.mark.gpu
def test_device_memory_beside_the_result_is_one_span():
    """While a result of 1 GB is made, device memory holds it, the input as
    given and as planes, and one span of rows; not a second result."""
    _capi.lib()
    hip = C.CDLL("libamdhip64.so.7")     # the one that the library has loaded

    def free():
        f, t = C.c_size_t(), C.c_size_t()
        assert hip.hipMemGetInfo(C.byref(f), C.byref(t)) == 0
        return f.value

    n = 2 ** 30 // (6 * 8)
    u = np.ones((n, 1))
    weno_solver(u[:64], 6)               # its code object is loaded
    lowest, stop = [free()], threading.Event()
    before = lowest[0]

    def watch():
        while not stop.wait(0.002):
            lowest.append(free())

    t = threading.Thread(target=watch)
    t.start()
    try:
        out = weno_solver(u, 6)
    finally:
        stop.set()
        t.join()
    assert np.allclose(out, 1.0, rtol=0, atol=1e-12)
    held = before - min(lowest)
    print("held", held / 2 ** 20, "MB in", len(lowest), "samples", flush=True)
    assert out.nbytes + u.nbytes <= held <= out.nbytes + 2 * u.nbytes + 2 ** 28 + 2 ** 26
