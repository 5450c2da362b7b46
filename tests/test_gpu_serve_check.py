"""The service's slab H·v, by classes and by list_2_1 and list_2_2 alone, and its
device eigenvalue check: every number of wanted values and check
interval against dense diagonalisation, from one-state sectors on.  Tolerance:
the service's own, 1e-10."""

import numpy as np
import pytest

from hphi_amd import lattice as L
from tests.golden.cases import two_body_cases

pytestmark = pytest.mark.gpu
TOL = 1e-10


@pytest.fixture(scope="module")
def A():
    from hphi_amd import capi
    capi.lib()
    return capi


def distinct(A, spec):
    e = A.Engine.from_spec(spec)
    e.sz(copy=False)
    h = np.stack([e.hv(c)[0] for c in np.eye(e.dim, dtype=np.complex128)], axis=1)
    e.close()
    w = np.linalg.eigvalsh(h)
    return w[np.concatenate([[True], np.diff(w) > 1e-8])]


SPECS = [L.heisenberg_chain(4, 1.0, 0.4, two_sz=4), L.heisenberg_chain(4, 1.0, 0.4), L.heisenberg_chain(9, 1.0, 0.7, two_sz=1),
         L.j1j2_ladder(5, 1.0, 0.3), L.hubbard_chain(4, 1.0, 3.0)]


@pytest.mark.parametrize("want,every", [(1, 1), (2, 16), (5, 3), (16, 1), (16, 7)])
def test_device_check_finds_the_lowest_distinct_values(A, want, every):
    srv = A.Server(hbm_budget=1 << 28, max_jobs=16, n_eigen=want, eps=1e-12, check_every=every)
    ids = [srv.submit(s, 5 + i, 0.0) for i, s in enumerate(SPECS)]
    res = {}
    for _ in range(5000):
        a, w = srv.tick()
        res.update({r.id: r for r in srv.results()})
        if a == 0 and w == 0:
            break
    srv.close()
    for i, s in zip(ids, SPECS):
        ref = distinct(A, s)[:want]
        got = np.array(res[i].eigenvalues[: res[i].n_found])
        assert len(got) >= 1 and len(got) <= want
        if res[i].converged and res[i].iterations < res[i].dim:  # not ended by the recurrence's own length
            assert len(got) == min(want, len(ref))
        n = min(len(got), len(ref), 2)
        assert np.max(np.abs(got[:n] - ref[:n])) <= TOL, (s.name, got, ref)
        for g in got:
            assert np.min(np.abs(distinct(A, s) - g)) <= TOL, (s.name, g)


# class layout: uneven splits, classes of a few ranks, odd particle numbers, real and complex couplings
# with value predicates; without it (list_2_1 past 16,384 entries): 30 sites
SLABS = [(n, s) for n, s in two_body_cases().items() if s.model in (L.SPIN, L.HUBBARD) and s.dim <= 1000]
SLABS += [("chain11_3", L.heisenberg_chain(11, 1.0, 0.4, two_sz=-5)), ("ladder10", L.j1j2_ladder(5, 1.0, 0.6)),
          ("square12_2", L.j1j2_square(4, 3, 1.0, 0.3, two_sz=-8)), ("hub5_3", L.hubbard_chain(5, 1.0, 2.0, ncond=3)),
          ("hub6", L.hubbard_chain(6, 1.0, 4.0)), ("chain30_1", L.heisenberg_chain(30, 1.0, 0.2, two_sz=-28)),
          ("chain30_2", L.heisenberg_chain(30, 1.0, 0.2, two_sz=-26))]


@pytest.mark.parametrize("name,spec", SLABS, ids=[n for n, _ in SLABS])
def test_slab_hv_finds_the_lowest_value(A, name, spec):
    """Five jobs of one structure (a full slab and one more) with the sector's ground state."""
    print(f"[gpu] slab {name}", flush=True)
    srv = A.Server(hbm_budget=1 << 28, max_jobs=8, n_eigen=1, eps=1e-12, check_every=2)
    ids = [srv.submit(spec, 31 + i, 0.0) for i in range(5)]
    res = {}
    for _ in range(5000):
        a, w = srv.tick()
        res.update({r.id: r for r in srv.results()})
        if a == 0 and w == 0:
            break
    srv.close()
    ref = distinct(A, spec)[0]
    for i in ids:
        assert abs(res[i].eigenvalues[0] - ref) <= TOL * max(abs(ref), 1.0), (name, res[i].eigenvalues[0], ref)
