"""The allocation-free H·v with the two-pass H·v asked for after the tables were
built: it builds none of that pass's tables and gives the single pass's bits."""

import numpy as np
import pytest

from hphi_amd import lattice as L

pytestmark = pytest.mark.gpu


# few workgroups (partial sums in pinned memory) and more than 256 of them
@pytest.mark.parametrize("spec", [L.heisenberg_chain(12), L.j1j2_square(5, 4), L.hubbard_chain(6)],
                         ids=["s12", "s20", "hub6"])
def test_noalloc_builds_no_tables_of_the_two_pass_hv(spec):
    from hphi_amd import capi as A
    e = A.Engine.from_spec(spec)
    e.tune(hi_split=0)
    e.sz(copy=False)
    e.diagonalcalc(copy=False)
    v1, v0 = A.DeviceArray(e.dim), A.DeviceArray(e.dim).zero()
    e.fill_random(v1, 1, 4)
    p0 = e.mltply_block_dev(1, v0, v1)
    one = v0.download()
    before = e.device_bytes
    e.tune(hi_split=1)
    assert e.get_tune("hi_split") == 1
    p = e.mltply_block_dev_noalloc(1, v0.zero(), v1)
    assert e.device_bytes == before
    assert np.array_equal(v0.download(), one) and np.array_equal(p, p0)
    e.mltply_block_dev(1, v0.zero(), v1)  # this entry may allocate: the pass's tables
    assert e.device_bytes > before
    assert np.max(np.abs(v0.download() - one)) <= 1e-12 * np.max(np.abs(one))
    e.close()
