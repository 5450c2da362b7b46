"""Column kernels of the block drivers at the edges of their tiles: norms and
dots of k columns against numpy, and the layout change between the callers'
vectors and the state-major block through the runs that use it.

Sums of n products: relative error at most n eps of the sum of magnitudes
(1e-12 for the sizes here).  Layouts are copies: bit for bit."""

import ctypes as C

import numpy as np
import pytest

from hphi_amd import lattice as L

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def A():
    from hphi_amd import capi
    capi.lib()
    return capi


# dims 2, 6, 252, 924, 12870 and 184756: below a wave, below a tile, ragged, many workgroups
@pytest.mark.parametrize("k", [1, 2, 3, 4, 7, 8, 16])
@pytest.mark.parametrize("n", [2, 4, 10, 12, 16, 20])
def test_column_sums(A, n, k):
    print(f"[gpu] column sums n={n} k={k}", flush=True)
    e = A.Engine.from_spec(L.spin_model("ring", n, [(i, (i + 1) % n, 1.0) for i in range(n)], two_sz=0))
    e.sz(copy=False)
    rng = np.random.default_rng(100 * n + k)
    x, y = (rng.standard_normal((e.dim, k)) + 1j * rng.standard_normal((e.dim, k)) for _ in range(2))
    dx, dy = (A.DeviceArray(e.dim * k).upload(v) for v in (x, y))
    out, dot = (C.c_double * k)(), (C.c_double * (2 * k))()
    A.check(A.lib().hphi_vec_norm2(e.h, dx.ptr, k, out))
    A.check(A.lib().hphi_vec_dot(e.h, dx.ptr, dy.ptr, k, dot))
    assert np.allclose(np.array(out), np.sum(np.abs(x) ** 2, 0), rtol=1e-12, atol=0)
    z = np.array(dot)[0::2] + 1j * np.array(dot)[1::2]
    assert np.all(np.abs(z - np.sum(x.conj() * y, 0)) <= 1e-12 * np.sum(np.abs(x * y), 0))
    e.close()


@pytest.mark.parametrize("k", [1, 2, 4, 8, 16])
@pytest.mark.parametrize("n", [6, 11, 13])
def test_block_layout_round_trip(A, n, k):
    """One TPQ step from given vectors: the last step's vectors are the start
    vectors over their norm, in the callers' order, in both layouts."""
    print(f"[gpu] layout n={n} k={k}", flush=True)
    e = A.Engine.from_spec(L.spin_model("ring", n, [(i, (i + 1) % n, 1.0) for i in range(n)], two_sz=None))
    rng = np.random.default_rng(n + k)
    w = rng.standard_normal((k, e.dim)) + 1j * rng.standard_normal((k, e.dim))
    for layout in (1, 0):
        start, end = A.DeviceArray(e.dim * k).upload(w), A.DeviceArray(e.dim * k)
        rows, _ = e.tpq_from(start, k, 1, W_end=end, layout=layout, large_value=4.0)
        got, nrm = end.download().reshape(k, e.dim), np.linalg.norm(w, axis=1)
        assert np.allclose(rows[0, :, 3], nrm, rtol=1e-13)
        assert np.allclose(got, w / nrm[:, None], rtol=1e-13, atol=0)
        rows, _ = e.ctpq_from(start, k, 1, W_end=end, large_value=4.0)
        assert np.allclose(end.download().reshape(k, e.dim), w / nrm[:, None], rtol=1e-13, atol=0)
    e.close()
