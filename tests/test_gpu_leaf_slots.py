"""P2M and L2P on the matrix cores with slots as columns, at the sizes where
their tiles can go wrong: leaves beyond 64 points (several passes), a few to
hundreds of slots a leaf, points and slots off a multiple of 16, grids of L^3
off a multiple of 16 and of 4, orders of either tile size, distinct targets.
Far-field evaluations are compared with the oracle's far field and repeated."""
import sys

import numpy as np
import pytest

import oracle_api as oa

pytestmark = pytest.mark.gpu


def _say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


@pytest.mark.parametrize("geo,n,m,nl,L,ncrit", [
    ("sphere", 3000, 0, 6, 4, 33),
    ("cube_edges", 12000, 4000, 6, 6, 150),
    ("cube_edges", 1500, 0, 10, 2, 20),
    ("ellipsoid", 1500, 0, 10, 9, 65),
    ("sphere", 1500, 0, 2, 10, 130),
    ("clusters", 8000, 3000, 6, 3, 100),
    ("cube_edges", 2000, 0, 9, 8, 40),
    ("sphere", 1500, 0, 5, 7, 18),
])
def test_far_field_matches_oracle(geo, n, m, nl, L, ncrit):
    import defmm_amd as dm
    from defmm_amd import workloads as wl
    src = wl.GEOMETRIES[geo](n, seed=31)
    trg = wl.GEOMETRIES[geo](m, seed=77) if m else src
    kappa = wl.kappa_for(nl, src, trg)
    q = wl.charges(n, seed=13)
    _say(f"case: {geo} N={n} targets {len(trg)} {nl} wavelengths L={L} Ncrit={ncrit}, far only")
    po, _, _, _ = oa.fmm(src, trg, q, L, ncrit, kappa, mode=2)
    for prec, l2max, mxmax in ((dm.FP64, 1e-12, 1e-10), (dm.MIXED, 3e-6, 3e-5)):
        A = dm.IBFMM_Mat(precision=prec)
        A.setSourceParticles(src)
        A.setTargetParticles(trg)
        A.prcmpt(L, ncrit, kappa)
        p = A.apply(q, parts=2)
        again = A.apply(q, parts=2)
        A.destroy()
        d = np.abs(p - po)
        l2 = np.sqrt((d ** 2).sum() / (np.abs(po) ** 2).sum())
        mx = d.max() / np.abs(po).max()
        _say(f"  precision {prec}: rel L2 {l2:.3e} max {mx:.3e}")
        assert l2 <= l2max and mx <= mxmax
        assert np.array_equal(p, again)
