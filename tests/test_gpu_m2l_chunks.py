"""M2L launches of several chunks of right-hand sides, in segments: numbers of
right-hand sides around the chunk widths and beyond one launch's chunks, on
plans of a few groups (one segment) and of many (several), against single
evaluations.  FP64 and mixed sums of a target take the same terms in the same
order at every width, so M2L differs by nothing but the near field's and the
matrix cores' order of summation: the bounds are those of a few roundings of
the sums (double 1e-13, float 1e-6, the largest entry 10 times that)."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def _diff(a, b):
    d = np.abs(a - b)
    return np.sqrt((d ** 2).sum() / (np.abs(b) ** 2).sum()), d.max() / np.abs(b).max()


@pytest.mark.parametrize("L,n,ncrit,nl", [(4, 900, 12, 2), (4, 20000, 33, 16), (5, 9000, 40, 12),
                                          (7, 5000, 20, 6), (8, 6000, 40, 10)])
@pytest.mark.parametrize("nr", [5, 19])
def test_batches_match_single(L, n, ncrit, nl, nr):
    import defmm_amd as dm
    from defmm_amd import workloads as wl
    pts = wl.cube_edges(n, seed=3)
    kappa = wl.kappa_for(nl, pts)
    Q = np.stack([wl.charges(n, seed=70 + r) for r in range(nr)])
    for prec, tol in ((dm.FP64, 1e-13), (dm.MIXED, 1e-6)):
        A = dm.IBFMM_Mat(precision=prec)
        A.setSourceParticles(pts)
        A.setTargetParticles(pts)
        A.prcmpt(L, ncrit, kappa)
        groups = A.stats()["m2l_groups"]
        assert groups > 0
        single = np.stack([A.apply(Q[r]) for r in range(nr)])
        A.set_rhs(nr)
        P = A.apply_batch(Q)
        again = A.apply_batch(Q)
        A.destroy()
        l2, mx = _diff(P, single)
        _say(f"case: L={L} N={n} {nr} right-hand sides precision {prec}: {groups} groups, "
             f"rel L2 {l2:.3e} max {mx:.3e}")
        assert l2 <= tol and mx <= 10 * tol
        assert np.array_equal(P, again)
