"""The service's slabs by classes, which only large sectors take by themselves: every
slab the layout fits, alone and in one tick with slabs it does not fit, and the
eigenvalue check on histories longer than its LDS.  Tolerance: the service's own, 1e-10."""

import numpy as np
import pytest

from hphi_amd import lattice as L
from tests.test_gpu_serve_check import SLABS, distinct

pytestmark = pytest.mark.gpu
TOL = 1e-10


@pytest.fixture(scope="module")
def A():
    from hphi_amd import capi
    capi.lib()
    return capi


def serve(A, specs, cls, **kw):
    args = dict(hbm_budget=1 << 29, max_jobs=32, n_eigen=1, eps=1e-12, check_every=2)
    args.update(kw)
    srv = A.Server(**args)
    srv.tune(cls=cls)
    ids = [srv.submit(s, 31 + i, 0.0) for i, s in enumerate(specs)]
    res = {}
    for _ in range(5000):
        a, w = srv.tick()
        res.update({r.id: r for r in srv.results()})
        if a == 0 and w == 0:
            break
    srv.close()
    return [res[i] for i in ids]


@pytest.mark.parametrize("cls", [0, 1])
@pytest.mark.parametrize("name,spec", SLABS, ids=[n for n, _ in SLABS])
def test_slab_by_classes_finds_the_lowest_value(A, name, spec, cls):
    print(f"[gpu] slab {name} cls {cls}", flush=True)
    ref = distinct(A, spec)[0]
    for r in serve(A, [spec] * 5, cls):
        assert abs(r.eigenvalues[0] - ref) <= TOL * max(abs(ref), 1.0), (name, r.eigenvalues[0], ref)


def test_slabs_of_both_kinds_in_one_tick(A):
    """30 sites have no class layout; the others run by classes beside them, in both arrival orders."""
    specs = [dict(SLABS)[n] for n in ("chain30_2", "hub6", "ladder10", "chain30_1", "chain11_3")]
    jobs = [(s, distinct(A, s)[0]) for s in specs]
    for order in (jobs * 3, jobs[::-1] * 3):
        for (s, ref), r in zip(order, serve(A, [s for s, _ in order], 1)):
            assert abs(r.eigenvalues[0] - ref) <= TOL * max(abs(ref), 1.0), s.name


@pytest.mark.parametrize("want", [2, 5, 16])
def test_converged_jobs_return_the_lowest_values_in_order(A, want):
    """Every returned value is the next distinct level, not just one of the spectrum."""
    specs = [L.heisenberg_chain(9, 1.0, 0.7, two_sz=1), L.j1j2_ladder(5, 1.0, 0.3), L.hubbard_chain(4, 1.0, 3.0)]
    ended = 0
    for s, r in zip(specs, serve(A, specs, -1, n_eigen=want, check_every=3)):
        got, ref = np.array(r.eigenvalues[: r.n_found]), distinct(A, s)[:want]
        if r.converged and r.iterations < r.dim:
            ended += 1
            assert len(got) == len(ref) and np.max(np.abs(got - ref)) <= TOL, (s.name, got, ref)
    assert ended


def test_check_of_a_history_longer_than_its_lds(A):
    """2,100 steps that no eps ends: alpha and beta come from memory instead of LDS."""
    spec = L.j1j2_square(4, 4, 1.0, 0.4)
    e = A.Engine.from_spec(spec)
    ref = e.lanczos(n_eigen=2, max_iter=600, eps=1e-12, mode=1, seed=3)
    e.close()
    assert ref.converged
    for r in serve(A, [spec] * 2, -1, n_eigen=2, eps=1e-290, check_every=16, max_iter=2100):
        assert r.n_found == 2 and r.iterations == 2100
        assert np.max(np.abs(np.array(r.eigenvalues[:2]) - np.array(ref.eigenvalues[:2]))) <= TOL


def test_results_by_classes_do_not_depend_on_the_mix(A):
    """Bit for bit the same alone and beside others, as without the class layout."""
    spec = L.hubbard_chain(6, 1.0, 4.0)
    alone = serve(A, [spec], 1, n_eigen=3)[0]
    mixed = serve(A, [spec, L.j1j2_ladder(5, 1.0, 0.6), spec, L.heisenberg_chain(30, 1.0, 0.2, two_sz=-26), spec], 1, n_eigen=3)[0]
    assert alone.iterations == mixed.iterations
    assert list(alone.eigenvalues) == list(mixed.eigenvalues)
