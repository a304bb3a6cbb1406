"""P2M and L2P of plans with enough slots for the matrix cores at every order
(and of some that stay on the vector kernels: kappa = 0, order 3), with points
and slots off a multiple of 16, leaves beyond 64 points, distinct targets and
more than 2,048 leaves.  Far-field evaluations are compared with the oracle's
far field, at the bounds of the other comparisons, and repeated."""
import sys

import numpy as np
import pytest

import oracle_api as oa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("geo,n,m,nl,L,ncrit", [
    ("clusters", 9000, 0, 12, 2, 33),
    ("sphere", 40000, 0, 8, 3, 9),
    ("cube_edges", 6000, 0, 6, 4, 150),
    ("sphere", 9000, 0, 10, 5, 33),
    ("cube_edges", 20000, 0, 20, 5, 90),
    ("sphere", 12000, 4000, 12, 6, 20),
    ("clusters", 9000, 0, 0, 6, 33),
    ("sphere", 8000, 0, 9, 7, 33),
    ("cube_edges", 8000, 0, 10, 8, 33),
    ("ellipsoid", 7000, 0, 24, 9, 33),
    ("sphere", 4000, 0, 8, 10, 18),
])
def test_far_field_matches_oracle(geo, n, m, nl, L, ncrit):
    import defmm_amd as dm
    from defmm_amd import workloads as wl
    src = wl.GEOMETRIES[geo](n, seed=31)
    trg = wl.GEOMETRIES[geo](m, seed=77) if m else src
    kappa = wl.kappa_for(nl, src, trg) if nl else 0.0
    q = wl.charges(n, seed=13)
    print(f"case: {geo} N={n} targets {len(trg)} {nl} wavelengths L={L} Ncrit={ncrit}, far only",
          flush=True)
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
        print(f"  precision {prec}: rel L2 {l2:.3e} max {mx:.3e}", flush=True)
        assert l2 <= l2max and mx <= mxmax
        assert np.array_equal(p, again)
    sys.stdout.flush()
