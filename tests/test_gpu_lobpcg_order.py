"""LOBPCG's H·v: equal bits with the class layout and without it (the phases of its
Ritz vectors follow rounding, so another order of summation would return others)."""

import numpy as np
import pytest

from hphi_amd import lattice as L
from tests.golden.cases import two_body_cases

pytestmark = pytest.mark.gpu


def hubbard(hop, interall):
    s = L.hubbard_chain(6)
    s.trans = [(i, a, j, b, hop.real, hop.imag if i < j else -hop.imag) for i, a, j, b, _, _ in s.trans] if hop else []
    s.interall = interall
    return s


def assisted(v):
    """n in the high half, hop in the low one"""
    return [(5, 0, 5, 0, 0, 0, 1, 0, v.real, v.imag), (1, 0, 0, 0, 5, 0, 5, 0, v.real, -v.imag),
            (4, 1, 4, 1, 1, 0, 2, 0, v.real, v.imag), (2, 0, 1, 0, 4, 1, 4, 1, v.real, -v.imag),
            (4, 0, 4, 0, 0, 0, 1, 0, 0.5 * v.real, 0.0), (1, 0, 0, 0, 4, 0, 4, 0, 0.5 * v.real, 0.0),
            (0, 1, 1, 1, 4, 0, 5, 0, 0.3, 0.0), (5, 0, 4, 0, 1, 1, 0, 1, 0.3, 0.0)]


CASES = [("chain12", L.heisenberg_chain(12)), ("hub6", L.hubbard_chain(6)), ("hub6_complex", hubbard(1 + 0.3j, [])),
         ("assisted", hubbard(0.0, assisted(0.2 + 0j))), ("hops_assisted", hubbard(1.0 + 0j, assisted(0.2 + 0j))),
         ("hops_assisted_complex", hubbard(1 + 0.3j, assisted(0.2 + 0.1j)))]
CASES += [(n, s) for n, s in two_body_cases().items() if s.model in (L.SPIN, L.HUBBARD)]


@pytest.mark.parametrize("k", [1, 2, 8])
@pytest.mark.parametrize("name,spec", CASES, ids=[c[0] for c in CASES])
def test_lobpcg_hv_has_the_gather_kernels_bits(name, spec, k):
    from hphi_amd import capi as A
    import ctypes as C
    lib = A.lib()
    lib.hphi_lb_hv.argtypes = [C.c_void_p, C.c_int, C.c_void_p, C.c_void_p]
    out = []
    for cls in (0, -1):
        e = A.Engine.from_spec(spec)
        e.tune(cls=cls)
        e.diagonalcalc(copy=False)
        x, y = A.DeviceArray(e.dim * k), A.DeviceArray(e.dim * k)
        e.fill_random(x, k, 9)
        A.check(lib.hphi_lb_hv(e.h, k, y.ptr, x.ptr))
        A.check(lib.hphi_synchronize())
        out.append(y.download())
        e.close()
    assert np.max(np.abs(out[0] - out[1])) == 0.0
