"""The autotuner as the first call on an engine: it builds what the class and tile
kernels need, offers them, and leaves a right H·v."""

import re

import numpy as np
import pytest

from hphi_amd import lattice as L

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("spec,k,knob", [(L.j1j2_square(5, 4), 1, "cls"), (L.j1j2_square(5, 4), 4, "cls"),
                                         (L.hubbard_chain(8), 2, "cls"),
                                         (L.triangular_xxz_gc(10, 2, 1.0, 0.8, 0.1), 1, "gc_tile"),
                                         (L.triangular_xxz_gc(10, 2, 1.0, 0.8, 0.1), 8, "gc_tile")],
                         ids=["spin_1", "spin_4", "hubbard_2", "spingc_1", "spingc_8"])
def test_autotune_on_a_fresh_engine(spec, k, knob):
    from hphi_amd import capi as A
    print(f"[gpu] autotune fresh {spec.name} k={k}", flush=True)
    ref = A.Engine.from_spec(spec)
    V1, V0 = A.DeviceArray(ref.dim * k), A.DeviceArray(ref.dim * k).zero()
    ref.fill_random(V1, k, 8)
    ref.mltply_block_dev(k, V0, V1)
    want = V0.download()
    ref.close()
    e = A.Engine.from_spec(spec)
    report = e.autotune(k, V0, V1, reps=1)
    lines = report.strip().split("\n")
    for v in (1, 0):
        assert any(re.search(rf"\b{knob}(_k\d+)?={v} ", ln) for ln in lines), report
    e.mltply_block_dev(k, V0.zero(), V1)
    assert np.max(np.abs(V0.download() - want)) <= 1e-12 * np.max(np.abs(want))
    e.close()
