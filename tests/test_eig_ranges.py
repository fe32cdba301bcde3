"""Wave-speed routines at the edges of their fast paths: the unscaled range of
the matrix, columns whose tail is just above or below "already reduced", and
reflectors with a dominant or vanishing head, bit for bit against the oracle."""
import numpy as np
import pytest

import cpu_checkers as cc
from pypde_amd import _capi, systems
from pypde_amd.solvers import Solver


def edge_matrices(V, seed, scales):
    rng = np.random.default_rng(seed)
    out = []
    for s in scales:                    # largest |entry| around 2^+-64 and far outside
        for _ in range(8):
            out.append(np.ldexp(rng.standard_normal((V, V)), s))
    # square norm of a column's tail around 2^-500 and 2^-900 (and nothing below)
    for e in (-240, -249, -250, -251, -300, -449, -450, -451, -480):
        for head in (1.0, -1.0, 0.0):
            A = rng.standard_normal((V, V))
            A[2:, 0] = np.ldexp(rng.standard_normal(V - 2), e)
            A[1, 0] *= head
            out.append(A)
            B = np.triu(rng.standard_normal((V, V)), -1)
            B[V - 1, V - 3] = np.ldexp(1.0, e)
            out.append(B)
    # one or two entries that dominate everything
    for s in (30, 60, 63):
        for _ in range(8):
            A = rng.standard_normal((V, V))
            A[rng.integers(V), rng.integers(V)] *= 2.0 ** s
            out.append(A)
    n = len(out) & ~1
    return np.ascontiguousarray(np.stack(out[:n]))


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["euler1d", "euler2d", "reactive2d"])
def test_wave_speed_at_the_edges_of_its_ranges(name):
    V = systems.SYSTEMS[name]["V"]
    ndim = 1 if name == "euler1d" else 2
    sol = Solver(np.ones((8,) * ndim + (V,)), [1.0] * ndim, systems.source(name), order=3,
                 stiff=name == "reactive2d")
    try:
        A = edge_matrices(V, 5 + V, (-900, -65, -64, -63, -10, 10, 63, 64, 65, 900))
        want = np.array([cc.oracle().oracle_max_abs_eig(cc.dp(a.copy()), V) for a in A])
        got = np.zeros(len(A))
        _capi.check(_capi.lib().pypde_eig_batch(sol.h, 0, _capi.dp(A), None, len(A),
                                                _capi.dp(got)), "eig_batch")
        assert np.array_equal(got, want)
    finally:
        sol.close()


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["euler1d", "euler2d"])
def test_abs_matrix_product_at_the_edges_of_its_ranges(name):
    V = systems.SYSTEMS[name]["V"]
    ndim = 1 if name == "euler1d" else 2
    sol = Solver(np.ones((8,) * ndim + (V,)), [1.0] * ndim, systems.source(name), order=3,
                 stiff=False, flux="roe")
    try:
        A = edge_matrices(V, 15 + V, (-200, -10, 10, 200))
        x = np.ascontiguousarray(np.random.default_rng(3).standard_normal((len(A), V)))
        want, got = np.zeros((len(A), V)), np.zeros((len(A), V))
        for i in range(len(A)):
            cc.oracle().oracle_abs_apply(cc.dp(A[i].copy()), cc.dp(x[i].copy()), V,
                                         cc.dp(want[i]))
        _capi.check(_capi.lib().pypde_eig_batch(sol.h, 2, _capi.dp(A), _capi.dp(x), len(A),
                                                _capi.dp(got)), "eig_batch")
        assert np.array_equal(got, want, equal_nan=True)
    finally:
        sol.close()
