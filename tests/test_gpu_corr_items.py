"""Green's function items: numbers of entries around the eight of a workgroup, of
both kinds, repeated entries, and states of more than 32 bits, against sums over
the basis.  Tolerance: 1e-13 for a normalised vector, a few hundred roundings."""

import numpy as np
import pytest

from hphi_amd import lattice as L

pytestmark = pytest.mark.gpu
TOL = 1e-13


@pytest.fixture(scope="module")
def A():
    from hphi_amd import capi
    capi.lib()
    return capi


def expected(basis, v, entry):
    i, s, _, s2, k, t, _, t2 = (int(q) for q in entry)
    at = {int(x): j for j, x in enumerate(basis)}
    total = 0.0 + 0.0j
    for j, x in enumerate(basis):  # |i:s><i:s2| |k:t><k:t2| between x and its source y
        x = int(x)
        bi, bk = (x >> i) & 1, (x >> k) & 1
        if s == s2 and t == t2:
            if i == k and s != t:
                continue
            if bi == s and bk == t:
                total += abs(v[j]) ** 2
        elif bi == s and bk == t:
            total += np.conj(v[j]) * v[at[x ^ (1 << i) ^ (1 << k)]]
    return total


@pytest.mark.parametrize("n", [1, 7, 8, 9, 16, 40])
@pytest.mark.parametrize("spec", [L.heisenberg_chain(9, 1.0, 0.3, two_sz=1), L.heisenberg_chain(34, 1.0, 0.3, two_sz=-30)],
                         ids=["9_sites", "34_sites"])
def test_entries_against_basis_sums(A, spec, n):
    rng = np.random.default_rng(n)
    e = A.Engine.from_spec(spec)
    basis = np.asarray(e.sz()[0])[1:].astype(np.uint64)
    v = rng.standard_normal(2 * e.dim).view(np.complex128)
    v /= np.linalg.norm(v)
    entries = []
    while len(entries) < n:
        i, k = (int(q) for q in rng.choice(spec.nsite, 2, replace=False))
        s, t = (int(q) for q in rng.integers(0, 2, 2))
        entries.append((i, s, i, s, k, t, k, t) if rng.random() < 0.5 else (i, s, i, 1 - s, k, 1 - s, k, s))
        if rng.random() < 0.3:
            entries.append(entries[-1])
            entries.append(entries[-1][4:] + entries[-1][:4])
    entries = entries[:n]
    got = e.cisajscktalt(A.DeviceArray(e.dim).upload(v), np.array(entries, np.int32))
    e.close()
    for g, q in zip(np.asarray(got).ravel(), entries):
        assert abs(g - expected(basis, v, q)) <= TOL, (q, g, expected(basis, v, q))
