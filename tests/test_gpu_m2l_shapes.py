"""M2L block shapes that depend on the order and on the groups' length: order 2
(one value a lane, up to 8 right-hand sides a launch) and long groups at orders
9 and 10 (one block a CU for one right-hand side in float).  Far fields are
compared with the oracle's, batches with single evaluations, at the bounds of
the other comparisons of that kind."""
import sys

import numpy as np
import pytest

import oracle_api as oa

pytestmark = pytest.mark.gpu


def _plan(dm, pts, L, ncrit, kappa, prec):
    A = dm.IBFMM_Mat(precision=prec)
    A.setSourceParticles(pts)
    A.setTargetParticles(pts)
    A.prcmpt(L, ncrit, kappa)
    return A


def _diff(a, b):
    d = np.abs(a - b)
    return np.sqrt((d ** 2).sum() / (np.abs(b) ** 2).sum()), d.max() / np.abs(b).max()


@pytest.mark.parametrize("geo,n,ncrit,nl", [("sphere", 6000, 20, 8), ("clusters", 9000, 40, 0)])
def test_order_2_far_field_matches_oracle(geo, n, ncrit, nl):
    import defmm_amd as dm
    from defmm_amd import workloads as wl
    pts = wl.GEOMETRIES[geo](n, seed=3)
    kappa = wl.kappa_for(nl, pts) if nl else 0.0
    q = wl.charges(n, seed=13)
    print(f"case: {geo} N={n} {nl} wavelengths L=2 Ncrit={ncrit}, far only", flush=True)
    po, _, _, _ = oa.fmm(pts, pts, q, 2, ncrit, kappa, mode=2)
    for prec, l2max, mxmax in ((dm.FP64, 1e-12, 1e-10), (dm.MIXED, 3e-6, 3e-5)):
        A = _plan(dm, pts, 2, ncrit, kappa, prec)
        p = A.apply(q, parts=2)
        again = A.apply(q, parts=2)
        A.destroy()
        l2, mx = _diff(p, po)
        print(f"  precision {prec}: rel L2 {l2:.3e} max {mx:.3e}", flush=True)
        assert l2 <= l2max and mx <= mxmax
        assert np.array_equal(p, again)
    sys.stdout.flush()


@pytest.mark.parametrize("nr", [2, 7, 8, 19])
def test_order_2_batches_match_single(nr):
    import defmm_amd as dm
    from defmm_amd import workloads as wl
    n = 5000
    pts = wl.sphere(n, seed=3)
    kappa = wl.kappa_for(7, pts)
    Q = np.stack([wl.charges(n, seed=70 + r) for r in range(nr)])
    print(f"case: sphere N={n} 7 wavelengths L=2, {nr} right-hand sides", flush=True)
    for prec, tol in ((dm.FP64, 1e-13), (dm.MIXED, 1e-6)):
        A = _plan(dm, pts, 2, 33, kappa, prec)
        single = np.stack([A.apply(Q[r]) for r in range(nr)])
        A.set_rhs(nr)
        P = A.apply_batch(Q)
        A.set_m2l(dm.M2L_BATCHED)
        B = A.apply_batch(Q)
        A.destroy()
        for x in (P, B):
            l2, mx = _diff(x, single)
            print(f"  precision {prec}: rel L2 {l2:.3e} max {mx:.3e}", flush=True)
            assert l2 <= tol and mx <= 10 * tol
    sys.stdout.flush()


@pytest.mark.parametrize("L", [9, 10])
@pytest.mark.parametrize("n,ncrit,nl,long", [(15000, 65, 0, True), (4000, 40, 5, False)])
def test_long_groups_match_pairs(L, n, ncrit, nl, long):
    """A pair takes another shape than its members, with the same sums."""
    import defmm_amd as dm
    from defmm_amd import workloads as wl
    pts = wl.GEOMETRIES["clusters"](n, seed=3)
    kappa = wl.kappa_for(nl, pts) if nl else 0.0
    Q = np.stack([wl.charges(n, seed=70 + r) for r in range(2)])
    print(f"case: clusters N={n} {nl} wavelengths L={L}, one right-hand side and two", flush=True)
    A = _plan(dm, pts, L, ncrit, kappa, dm.MIXED)
    s = A.stats()
    assert (s["m2l_group_entries"] >= 32 * s["m2l_groups"]) == long
    single = np.stack([A.apply(q) for q in Q])
    A.set_rhs(2)
    P = A.apply_batch(Q)
    A.destroy()
    l2, mx = _diff(P, single)
    print(f"  rel L2 {l2:.3e} max {mx:.3e}", flush=True)
    sys.stdout.flush()
    assert l2 <= 1e-6 and mx <= 1e-5
