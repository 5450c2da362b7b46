"""Terms without a flip among the off-diagonal ones (a density product handed
over as InterAll entry instead of a diagonal one) on the two-pass H·v: whichever
half their mask lies in, every kernel applies them.  Reference: the same product
as a diagonal entry, in one pass.  Tolerance: the suite's H·v bar, 1e-12."""

import numpy as np
import pytest

from hphi_amd import lattice as L

pytestmark = pytest.mark.gpu
TOL = 1e-12


# both bits in the low half, one in each, both in the high half
@pytest.mark.parametrize("pair", [(0, 0, 1, 1), (1, 0, 5, 1), (4, 0, 5, 1)], ids=["low", "mixed", "high"])
@pytest.mark.parametrize("tune", [dict(cls=0, hi_split=0), dict(cls=0, hi_split=1), dict(cls=1, hi_split=0),
                                  dict(cls=1, hi_split=1), dict(cls=1, hi_split=1, hi_fuse_copy=0),
                                  dict(cls=1, cls_order=1, hi_split=1)], ids=str)
def test_density_products_among_the_off_diagonal_terms(pair, tune):
    from hphi_amd import capi as A
    a, s, b, u = pair
    spec = L.hubbard_chain(6)
    t = L.processed_terms(spec)
    diag, off = dict(t), dict(t)
    diag["interall_diag_idx"] = np.array([[a, s, b, u]], np.int32)
    diag["interall_diag_V"] = np.array([0.7])
    off["interall_idx"] = np.array([[a, s, a, s, b, u, b, u]], np.int32)
    off["interall_V"] = np.array([[0.7, 0.0]])
    out = []
    for terms, knobs in ((diag, dict(cls=0, hi_split=0)), (off, tune)):
        e = A.Engine.from_terms(spec.model, spec.nsite, spec.nup, spec.ndown, terms)
        e.tune(**knobs)
        e.sz(copy=False)
        assert e.get_tune("hi_split") == knobs["hi_split"] and e.get_tune("cls") == knobs["cls"]
        v = np.random.default_rng(12).standard_normal(2 * e.dim).view(np.complex128)
        out.append(e.hv(v))
        e.close()
    (x, p), (y, q) = out
    assert np.max(np.abs(x - y)) <= TOL * np.max(np.abs(x))
    assert abs(p - q) <= TOL * np.linalg.norm(v) * np.linalg.norm(x)
