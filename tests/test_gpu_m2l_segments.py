"""M2L launches of several segments (3, 4 and 8: from 16,384 groups on, at least
8,192 a segment) and several chunks of right-hand sides, against single
evaluations, at the bounds of the other comparisons of that kind (M2L's sums
are the same at every width)."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("geo,L,n,ncrit,nl,segments", [
    ("sphere", 7, 9000, 33, 14, 3), ("cube_edges", 8, 12000, 40, 14, 4),
    ("sphere", 8, 20000, 65, 16, 8)])
def test_batches_match_single(geo, L, n, ncrit, nl, segments):
    import defmm_amd as dm
    from defmm_amd import workloads as wl
    pts = wl.GEOMETRIES[geo](n, seed=3)
    kappa = wl.kappa_for(nl, pts)
    for prec, tol, nr in ((dm.FP64, 1e-13, 3), (dm.MIXED, 1e-6, 7)):
        Q = np.stack([wl.charges(n, seed=70 + r) for r in range(nr)])
        A = dm.IBFMM_Mat(precision=prec)
        A.setSourceParticles(pts)
        A.setTargetParticles(pts)
        A.prcmpt(L, ncrit, kappa)
        groups = A.stats()["m2l_groups"]
        assert max(1, min(8, groups // 8192)) == segments, groups
        single = np.stack([A.apply(Q[r]) for r in range(nr)])
        A.set_rhs(nr)
        assert A.m2l_mode() == dm.M2L_STORED  # (batches would have fewer groups)
        P = A.apply_batch(Q)
        A.destroy()
        d = np.abs(P - single)
        l2 = np.sqrt((d ** 2).sum() / (np.abs(single) ** 2).sum())
        mx = d.max() / np.abs(single).max()
        print(f"case: {geo} L={L} N={n} {nr} right-hand sides precision {prec}: {groups} groups, "
              f"rel L2 {l2:.3e} max {mx:.3e}", flush=True)
        sys.stdout.flush()
        assert l2 <= tol and mx <= 10 * tol
