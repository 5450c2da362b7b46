"""Grand-canonical H·v in LDS tiles (hv_gc.hip) against the oracle and, for the
terms the oracle does not cover, against the gather kernels.

The tile of k columns holds 4096 amplitudes: 12, 11 and 10 state bits for
k = 1, 2 and k >= 4.  Sizes: the smallest sector the path takes (three bits
outside the tile), ones between, several column groups, one and several
passes, terms left to the gather loop.  Tolerance: the suite's H·v bar, 1e-12
of the largest entry (the sums run in another order)."""

import numpy as np
import pytest

from hphi_amd import lattice as L

pytestmark = pytest.mark.gpu
TOL = 1e-12


@pytest.fixture(scope="module")
def A():
    from hphi_amd import capi
    capi.lib()
    return capi


def spin_mixed(n):
    """SpinGC ring: exchange, far bonds, pair lift, a field of two strengths and two-site flips of every form."""
    s = L.spin_model(f"mixed{n}", n, [(i, (i + d) % n, 1.0 / d) for d in (1, 3, n // 2) for i in range(n)], two_sz=None)
    s.pairlift = [(0, 1, 0.3), (n - 1, 2, -0.2)]
    for i in range(n):
        s.trans += [(i, 0, i, 1, 0.2 + 0.01 * i, 0.1), (i, 1, i, 0, 0.2 + 0.01 * i, -0.1)]
    s.interall = [(0, 1, 0, 1, 3, 1, 3, 0, 0.2, 0.1), (3, 0, 3, 1, 0, 1, 0, 1, 0.2, -0.1),
                  (n - 1, 1, n - 1, 0, 4, 1, 4, 0, 0.15, 0.05), (4, 0, 4, 1, n - 1, 0, n - 1, 1, 0.15, -0.05)]
    return s


def hubbard_mixed(n):
    """HubbardGC ring: hops, complex spin flips, a four-orbital flip, a density-assisted hop, pair hopping, exchange."""
    h = L.hubbard_chain_gc(n, 1.0, 3.0, mu=0.4, flip=complex(0.2, 0.1))
    h.interall = [(0, 0, 1, 1, 2, 0, 3, 0, 0.15, -0.05), (3, 0, 2, 0, 1, 1, 0, 0, 0.15, 0.05),
                  (n - 1, 1, n - 1, 1, 0, 0, 1, 0, 0.2, 0.0), (1, 0, 0, 0, n - 1, 1, n - 1, 1, 0.2, 0.0)]
    h.pairhop = [(1, 3, 0.25)]
    h.exchange = [(0, n - 1, -0.3)]
    return h


ORACLE = [("tri_5x3", L.triangular_xxz_gc(5, 3, 1.0, 0.8, 0.1), (1, 2, 4, 8, 16)),
          ("tri_8x2", L.triangular_xxz_gc(8, 2, 1.0, 0.8, 0.1), (1, 2, 4, 8, 16)),
          ("ring_13", L.spin_model("ring", 13, [(i, (i + d) % 13, 1.0 / d) for d in (1, 2) for i in range(13)],
                                   two_sz=None), (4, 8)),
          ("no_diagonal", L.spin_model("xy", 15, [(i, (i + 1) % 15, 1.0) for i in range(15)], two_sz=None,
                                       jz_scale=0.0), (1, 16))]


@pytest.mark.parametrize("name,spec,ks", ORACLE, ids=[c[0] for c in ORACLE])
def test_gc_tiles_match_oracle(A, oracle_lib, name, spec, ks):
    orc = oracle_lib.Oracle(spec, L.processed_terms(spec)).prepare()
    for k in ks:
        print(f"[gpu] gc tiles {name} k={k}", flush=True)
        e = A.Engine.from_spec(spec)
        e.tune(gc_tile=1)
        e.diagonalcalc(copy=False)
        assert e.get_tune("gc_tile") == 1
        V1, V0 = A.DeviceArray(e.dim * k), A.DeviceArray(e.dim * k)
        e.fill_random(V1, k, 70)
        e.fill_random(V0, k, 30)
        before = V0.download().reshape(e.dim, k)
        pr = e.mltply_block_dev(k, V0, V1)
        got = V0.download().reshape(e.dim, k) - before
        for c in range(k):
            v = oracle_lib.fill_vector(70 + c, e.dim)
            hv, p = orc.hv(v)
            assert np.max(np.abs(got[:, c] - hv)) <= TOL * np.max(np.abs(hv)), (k, c)
            assert abs(pr[c] - p) <= TOL * np.linalg.norm(v) * np.linalg.norm(hv), (k, c)
        e.close()


MIXED = [("spin_15", spin_mixed(15), (1, 2, 8)), ("spin_17", spin_mixed(17), (1, 4, 16)),
         ("hubbard_8", hubbard_mixed(8), (1, 2, 4, 16))]


@pytest.mark.parametrize("name,spec,ks", MIXED, ids=[c[0] for c in MIXED])
def test_gc_tiles_match_gather_kernels(A, name, spec, ks):
    """Every term form, accumulating, overwriting (v0 not read) and scaled."""
    for k in ks:
        print(f"[gpu] gc tiles {name} k={k}", flush=True)
        out = []
        for tile in (0, 1):
            e = A.Engine.from_spec(spec)
            e.tune(gc_tile=tile)
            e.diagonalcalc(copy=False)
            assert e.get_tune("gc_tile") == tile
            V1, V0 = A.DeviceArray(e.dim * k), A.DeviceArray(e.dim * k)
            e.fill_random(V1, k, 5)
            e.fill_random(V0, k, 50)
            pr = list(e.mltply_block_dev(k, V0, V1))
            res = [V0.download()]
            if k == 1:
                pr.append(e.mltply_dev_scaled(V0, V1, -0.3, 0.7))
                res.append(V0.download())
                V0.upload(np.full(e.dim, np.nan + 0j))
                pr.append(e.mltply_dev_scaled(V0, V1, 5.0, -1.5, overwrite=True))
                res.append(V0.download())
            out.append((np.concatenate(res), np.array(pr), np.linalg.norm(V1.download())))
            e.close()
        (a, pa, n), (b, pb, _) = out
        assert np.max(np.abs(a - b)) <= TOL * np.max(np.abs(a)), k
        assert np.max(np.abs(pa - pb)) <= TOL * n * np.linalg.norm(a), k


def test_gc_tile_rule(A):
    """By default the tiles serve sectors with at least 256 of them; a block
    shape set by hand keeps the gather kernel."""
    small, large = (A.Engine.from_spec(L.triangular_xxz_gc(n, 2)) for n in (7, 10))
    for e in (small, large):
        e.diagonalcalc(copy=False)
    assert small.get_tune("gc_tile") == 0 and large.get_tune("gc_tile") == 1
    large.tune(gc_tile=0)
    assert large.get_tune("gc_tile") == 0
    small.close()
    large.close()
