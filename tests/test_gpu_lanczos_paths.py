"""Lanczos steps queued with their scale factors on the device, on each H·v that takes
them from there: the grand-canonical tiles, and the two-pass H·v behind the class
kernel in either order of its units and behind the gather kernel.  Against the same
run one step at a time (equal bits) and against another H·v (1e-10)."""

import numpy as np
import pytest

from hphi_amd import lattice as L

pytestmark = pytest.mark.gpu

TRI = L.triangular_xxz_gc(10, 2, 1.0, 0.8, 0.1)
RUNS = [("tiles", TRI, dict(gc_tile=1), dict(gc_tile=0), "gc_tile"),
        ("split_class", L.j1j2_square(5, 4), dict(cls=1, cls_order=0, hi_split=1), dict(cls=0, hi_split=0), "hi_split"),
        ("split_index", L.j1j2_square(5, 4), dict(cls=1, cls_order=1, hi_split=1), dict(cls=0, hi_split=0), "hi_split"),
        ("split_index_hubbard", L.hubbard_chain(8), dict(cls=1, cls_order=1, hi_split=1), dict(cls=0, hi_split=0), "hi_split"),
        ("split_gather", L.j1j2_square(5, 4), dict(cls=0, hi_split=1), dict(cls=0, hi_split=0), "hi_split"),
        ("index", L.hubbard_chain(8), dict(cls=1, cls_order=1), dict(cls=0), "cls")]


@pytest.mark.parametrize("every,max_iter", [(5, 300), (16, 37)])
@pytest.mark.parametrize("name,spec,on,off,knob", RUNS, ids=[r[0] for r in RUNS])
def test_batched_steps_on_every_hv(tmp_path, name, spec, on, off, knob, every, max_iter):
    from hphi_amd import capi as A
    print(f"[gpu] lanczos {name} every {every}", flush=True)
    kw = dict(n_eigen=2, max_iter=max_iter, eps=1e-12, seed=9, check_every=every, mode=1)
    res = []
    for knobs, single in ((on, False), (on, True), (off, False)):
        e = A.Engine.from_spec(spec)
        e.tune(**knobs)
        e.diagonalcalc(copy=False)
        assert e.get_tune(knob) == knobs[knob]
        if single:
            res.append(e.lanczos_restart(restart_out=(str(tmp_path / "tm.dat"), str(tmp_path / "vec.dat")), **kw))
        else:
            res.append(e.lanczos(**kw))
        e.close()
    a, b, c = res
    assert (a.iterations, a.converged, a.n_found) == (b.iterations, b.converged, b.n_found)
    assert np.array_equal(np.array(a.eigenvalues), np.array(b.eigenvalues))
    n = min(a.n_found, c.n_found)
    assert n >= 1
    if a.converged and c.converged:
        assert np.max(np.abs(np.array(a.eigenvalues[:n]) - np.array(c.eigenvalues[:n]))) <= 1e-10 * abs(c.eigenvalues[0])
