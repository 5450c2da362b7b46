"""A block size without a kernel is an error at every entry that takes one,
before any grid is computed from it (k = 65 once divided by zero)."""

import numpy as np
import pytest

from hphi_amd import lattice as L

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("spec", [L.heisenberg_chain(8), L.hubbard_chain(4), L.triangular_xxz_gc(3, 2, 1.0, 0.8, 0.1)],
                         ids=["spin", "hubbard", "spingc"])
def test_block_sizes_without_a_kernel_are_errors(spec):
    from hphi_amd import capi as A
    e = A.Engine.from_spec(spec)
    v0, v1 = A.DeviceArray(e.dim * 2).zero(), A.DeviceArray(e.dim * 2)
    e.fill_random(v1, 2, 3)
    e.sz(copy=False)
    e.diagonalcalc(copy=False)
    for k in (-1, 0, 3, 5, 17, 32, 64, 65, 128, 1024, 1028):
        print(f"[gpu] {spec.name} k={k}", flush=True)
        for call in (lambda: A.check(A.lib().hphi_mltply_block_dev(e.h, k, v0.ptr, v1.ptr, None)),
                     lambda: A.check(A.lib().hphi_mltply_block_dev_noalloc(e.h, k, v0.ptr, v1.ptr, None)),
                     lambda: e.time_mltply(k, v0, v1, 1, 1), lambda: e.autotune(k, v0, v1, 1)):
            with pytest.raises(A.HphiError, match=f"k={k} not in"):
                call()
    assert np.all(v0.download() == 0)
    e.mltply_block_dev(2, v0, v1)
    assert np.any(v0.download() != 0)
    e.close()
