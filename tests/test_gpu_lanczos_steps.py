"""Lanczos steps queued in batches (and a batch ahead) against the same run one step
at a time, as a run that writes its restart files takes them: the same operations
in the same order, so equal bits.  Check intervals below, at and past the batch
length, step limits inside a batch, sectors that end the recurrence early."""

import numpy as np
import pytest

from hphi_amd import lattice as L

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def A():
    from hphi_amd import capi
    capi.lib()
    return capi


SPECS = [L.heisenberg_chain(4, 1.0, 0.3), L.heisenberg_chain(6, 1.0, 0.3), L.heisenberg_chain(12, 1.0, 0.4),
         L.hubbard_chain(6, 1.0, 4.0), L.hubbard_chain_gc(4, 1.0, 4.0, mu=0.3)]


@pytest.mark.parametrize("every,max_iter", [(1, 2000), (5, 2000), (16, 37), (17, 60), (40, 2000)])
@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("spec", SPECS, ids=[f"{s.name}_{s.dim}" for s in SPECS])
def test_batched_steps_equal_single_steps(A, tmp_path, spec, mode, every, max_iter):
    kw = dict(n_eigen=2 if mode else 1, max_iter=max_iter, eps=1e-12, seed=9, check_every=every, mode=mode)
    e = A.Engine.from_spec(spec)
    a = e.lanczos(**kw)
    e.close()
    e = A.Engine.from_spec(spec)
    b = e.lanczos_restart(restart_out=(str(tmp_path / "tm.dat"), str(tmp_path / "vec.dat")), **kw)
    e.close()
    assert (a.iterations, a.converged, a.n_found) == (b.iterations, b.converged, b.n_found)
    assert np.array_equal(np.array(a.eigenvalues), np.array(b.eigenvalues))


def test_restart_continues_after_batches(A, tmp_path):
    """Ten steps, written, then continued: the values of the uninterrupted run."""
    spec = L.heisenberg_chain(12, 1.0, 0.4)
    f = (str(tmp_path / "tm.dat"), str(tmp_path / "vec.dat"))
    e = A.Engine.from_spec(spec)
    e.lanczos_restart(restart_out=f, max_iter=10, eps=1e-13, seed=4)
    e.close()
    e = A.Engine.from_spec(spec)
    r = e.lanczos_restart(restart_in=f, max_iter=500, eps=1e-13, seed=4)
    e.close()
    e = A.Engine.from_spec(spec)
    ref = e.lanczos(max_iter=500, eps=1e-13, seed=4)
    e.close()
    assert abs(r.eigenvalues[0] - ref.eigenvalues[0]) <= 1e-10 * abs(ref.eigenvalues[0])
