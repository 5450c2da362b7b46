"""Canonical H·v by classes (hv_class.hip) against the oracle, for 1, 2 and 4
blocks per wave, at the edges of its tiles of 64 ranks and of its block groups,
and against k_hv_canon for terms the oracle does not cover.  Tolerance: the
suite's H·v bar, 1e-12 of the largest entry."""

import numpy as np
import pytest

from hphi_amd import lattice as L
from tests.golden.cases import two_body_cases

pytestmark = pytest.mark.gpu
TOL = 1e-12


@pytest.fixture(scope="module")
def A():
    from hphi_amd import capi
    capi.lib()
    return capi


def ring(n, nup):
    """J1-J2 ring with a far bond, so that every group has terms."""
    s = L.spin_model(f"ring{n}_{nup}", n, [(i, (i + d) % n, 1.0 / d) for d in (1, 2) for i in range(n)]
                     + [(0, n // 2, 0.3)], two_sz=2 * nup - n)
    return s


# sizes: two sites; classes of 1..3 states; 70-, 126- and 924-state classes (below, just past and
# many tiles of 64); odd site numbers (an uneven split); nearly empty and nearly full sectors
CASES = [("s2", ring(4, 2)), ("s7", ring(7, 3)), ("s15", ring(15, 7)), ("s18", ring(18, 9)), ("s23_4", ring(23, 4)),
         ("s20_18", ring(20, 18)), ("s12_1", ring(12, 1)), ("j1j2_5x4", L.j1j2_square(5, 4)),
         ("hub4", L.hubbard_chain(4)), ("hub7", L.hubbard_chain(7, ncond=5)), ("hub9", L.hubbard_chain(9)),
         ("hub_3x3", L.hubbard_square(3, 3, ncond=8)), ("hub6_1", L.hubbard_chain(6, ncond=1))]


@pytest.mark.parametrize("name,spec", CASES, ids=[c[0] for c in CASES])
def test_class_kernel_matches_oracle(A, oracle_lib, name, spec):
    orc = oracle_lib.Oracle(spec, L.processed_terms(spec)).prepare()
    v = oracle_lib.fill_vector(3, spec.dim)
    hv, p = orc.hv(v)
    scale = max(np.max(np.abs(hv)), 1e-300)
    for cb in (1, 2, 4):
        print(f"[gpu] class kernel {name} blocks {cb}", flush=True)
        e = A.Engine.from_spec(spec)
        e.tune(cls=1, cls_blocks=cb, cls_wgs_per_cu=1 if cb == 2 else 256)
        e.sz(copy=False)
        assert e.get_tune("cls") == 1
        got, pr = e.hv(v)
        assert np.max(np.abs(got - hv)) <= TOL * scale
        assert abs(pr - p) <= TOL * np.linalg.norm(v) * max(np.linalg.norm(hv), 1e-300)
        v1, v0 = A.DeviceArray(e.dim).upload(v), A.DeviceArray(e.dim).upload(np.full(e.dim, np.nan + 0j))
        e.mltply_dev_scaled(v0, v1, 3.0, -0.5, overwrite=True)  # v0 is not read
        assert np.max(np.abs(v0.download() + 0.5 * hv)) <= TOL * scale
        e.mltply_dev_scaled(v0, v1, -2.0, 0.25)
        assert np.max(np.abs(v0.download() - 1.25 * hv)) <= 2 * TOL * scale
        e.close()


@pytest.mark.parametrize("cb", [1, 2, 4])
@pytest.mark.parametrize("name", [n for n, s in two_body_cases().items() if s.model in (L.SPIN, L.HUBBARD)])
def test_class_kernel_two_body_terms(A, name, cb):
    """Complex value-predicate terms, pair hops, four-orbital flips: equal to k_hv_canon."""
    spec = two_body_cases()[name]
    out = []
    for cls in (0, 1):
        e = A.Engine.from_spec(spec)
        e.tune(cls=cls, cls_blocks=cb)
        e.sz(copy=False)
        assert e.get_tune("cls") == cls
        v = np.random.default_rng(5).standard_normal(2 * e.dim).view(np.complex128)
        out.append(e.hv(v))
        e.close()
    assert np.max(np.abs(out[0][0] - out[1][0])) <= TOL * np.max(np.abs(out[0][0]))
    assert abs(out[0][1] - out[1][1]) <= TOL * np.linalg.norm(v) * np.linalg.norm(out[0][0])


@pytest.mark.parametrize("cb", [1, 4])
@pytest.mark.parametrize("spec", [L.j1j2_square(5, 4), L.hubbard_chain(9)], ids=["spin", "hubbard"])
def test_class_kernel_before_the_high_half_pass(A, spec, cb):
    """As the first pass of the two-pass H·v, with and without the fused copy."""
    res = []
    for tune in (dict(cls=0, hi_split=0), dict(cls=1, hi_split=1), dict(cls=1, hi_split=1, hi_fuse_copy=0)):
        e = A.Engine.from_spec(spec)
        e.tune(cls_blocks=cb, **tune)
        e.sz(copy=False)
        v = np.random.default_rng(6).standard_normal(2 * e.dim).view(np.complex128)
        res.append(e.hv(v)[0])
        e.close()
    for r in res[1:]:
        assert np.max(np.abs(r - res[0])) <= TOL * np.max(np.abs(res[0]))


TWO_BODY = [(n, s) for n, s in two_body_cases().items() if s.model in (L.SPIN, L.HUBBARD)]


@pytest.mark.parametrize("k", [2, 4, 8, 16])
@pytest.mark.parametrize("name,spec", CASES + TWO_BODY, ids=[c[0] for c in CASES + TWO_BODY])
def test_class_kernel_block(A, name, spec, k):
    """Blocks of k columns equal k_hv_blk's, with and without allocations."""
    out = []
    for tune in (dict(cls=0), dict(cls=1), dict(cls=1, cls_blocks=4, cls_wgs_per_cu=1)):
        print(f"[gpu] class kernel {name} k {k} {tune}", flush=True)
        e = A.Engine.from_spec(spec)
        e.tune(**tune)
        e.sz(copy=False)
        e.diagonalcalc(copy=False)
        assert e.get_tune("cls") == tune["cls"]
        rng = np.random.default_rng(7)
        v = rng.standard_normal(2 * e.dim * k).view(np.complex128)
        w = rng.standard_normal(2 * e.dim * k).view(np.complex128)
        v1, v0 = A.DeviceArray(e.dim * k).upload(v), A.DeviceArray(e.dim * k).upload(w)
        p = e.mltply_block_dev(k, v0, v1)
        a = v0.download()
        v0.upload(w)
        q = e.mltply_block_dev_noalloc(k, v0, v1)
        assert np.array_equal(v0.download(), a) and np.array_equal(p, q)
        out.append((a, p, np.linalg.norm(v) * np.linalg.norm(a)))
        e.close()
    a, p, s = out[0]
    for b, q, _ in out[1:]:
        assert np.max(np.abs(b - a)) <= TOL * np.max(np.abs(a))
        assert np.max(np.abs(q - p)) <= TOL * s


@pytest.mark.parametrize("k", [1, 2, 16])
@pytest.mark.parametrize("name,spec", CASES, ids=[c[0] for c in CASES])
def test_units_by_index_equal_units_by_class(A, name, spec, k):
    """The order for vectors beyond the caches, for 1, 2 and 4 blocks per wave."""
    out = []
    for tune in [dict(cls_order=0)] + [dict(cls_order=1, cls_blocks=cb, cls_wgs_per_cu=w) for cb, w in ((1, 256), (2, 1), (4, 256))]:
        print(f"[gpu] class order {name} k {k} {tune}", flush=True)
        e = A.Engine.from_spec(spec)
        e.tune(cls=1, **tune)
        e.sz(copy=False)
        e.diagonalcalc(copy=False)
        assert e.get_tune("cls_order") == tune["cls_order"]
        v = np.random.default_rng(8).standard_normal(2 * e.dim * k).view(np.complex128)
        v1, v0 = A.DeviceArray(e.dim * k).upload(v), A.DeviceArray(e.dim * k).upload(2 * v)
        p = e.mltply_block_dev(k, v0, v1)
        out.append((v0.download(), p))
        e.close()
    a, p = out[0]
    for b, q in out[1:]:
        assert np.max(np.abs(b - a)) <= TOL * np.max(np.abs(a))
        assert np.max(np.abs(q - p)) <= TOL * np.linalg.norm(v) * np.linalg.norm(a)
