"""Lowest eigenvalues of a tridiagonal (host, sixteen Sturm counts at a time) against
LAPACK: sizes and numbers of eigenvalues around the lane count, decoupled and
degenerate blocks.  Tolerance: 1e-13 of the spectrum's width, LAPACK's own error."""

import ctypes as C

import numpy as np
import pytest
import scipy.linalg as sl


def lowest(a, b, k):
    from hphi_amd import capi
    ev = np.zeros(max(k, 1))
    p = lambda v: np.ascontiguousarray(v).ctypes.data_as(C.POINTER(C.c_double))
    f = capi.lib().hphi_tridiag_lowest
    f.restype = C.c_int
    a, b = np.ascontiguousarray(a, float), np.ascontiguousarray(np.append(b, 0.0), float)
    n = f(p(a), p(b), len(a), k, p(ev))
    return ev[:n]


@pytest.mark.parametrize("kind", ["random", "decoupled", "equal", "zero"])
@pytest.mark.parametrize("n", [1, 2, 3, 16, 17, 40, 300])
def test_lowest_matches_lapack(n, kind):
    rng = np.random.default_rng(n)
    a, b = rng.standard_normal(n), 0.5 + rng.random(n - 1)
    if kind == "decoupled":
        b[::3] = 0.0
    if kind == "equal":
        a[:], b[:] = 2.0, 0.0
    if kind == "zero":
        a[:] = 0.0
    ref = sl.eigh_tridiagonal(a, b, eigvals_only=True) if n > 1 else a
    width = max(np.max(np.abs(ref)), 1.0)
    for k in (1, 2, 3, 5, 9, 15, 16, 17, 33):
        got = lowest(a, b, k)
        assert len(got) == min(k, n)
        assert np.all(np.diff(got) >= 0)
        assert np.max(np.abs(got - ref[: len(got)])) <= 1e-13 * width * max(n, 10) / 10, (kind, n, k)
