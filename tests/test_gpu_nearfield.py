"""Near field at the sizes where its work items can go wrong: leaves of one
point up to several chunks of 8 targets, source runs around a multiple of 64
lanes, every phase evaluation (Laplace, table, kappa * r formed first) and
every number of right-hand sides a launch takes.  Near-only evaluations are
compared with the oracle's near field, batches with single evaluations."""
import sys

import numpy as np
import pytest

import oracle_api as oa

pytestmark = pytest.mark.gpu


def _say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def _diff(a, b):
    d = np.abs(a - b)
    return np.sqrt((d ** 2).sum() / (np.abs(b) ** 2).sum()), d.max() / np.abs(b).max()


def _plan(dm, src, trg, L, ncrit, kappa, prec):
    A = dm.IBFMM_Mat(precision=prec)
    A.setSourceParticles(src)
    A.setTargetParticles(trg)
    A.prcmpt(L, ncrit, kappa)
    return A


@pytest.mark.parametrize("kappa", [0.0, 6.0, 1e-31])
@pytest.mark.parametrize("n,ncrit", [(700, 8), (1500, 18), (3000, 130)])
def test_near_only_matches_oracle(n, ncrit, kappa):
    import defmm_amd as dm
    from defmm_amd import workloads as wl
    src = wl.sphere(n, seed=21)
    trg = np.concatenate([wl.sphere(n // 2 + 3, seed=5), src[:40]])  # some targets are sources
    q = wl.charges(n, seed=9)
    _say(f"case: sphere N={n} Ncrit={ncrit} kappa={kappa}, near only")
    po, _, _, _ = oa.fmm(src, trg, q, 3, ncrit, kappa, mode=1)
    for prec, l2max, mxmax in ((dm.FP64, 1e-12, 1e-10), (dm.MIXED, 3e-6, 3e-5)):
        A = _plan(dm, src, trg, 3, ncrit, kappa, prec)
        p = A.apply(q, parts=1)
        again = A.apply(q, parts=1)
        A.destroy()
        l2, mx = _diff(p, po)
        _say(f"  precision {prec}: rel L2 {l2:.3e} max {mx:.3e}")
        assert l2 <= l2max and mx <= mxmax
        assert np.array_equal(p, again)


@pytest.mark.parametrize("nr", [2, 3, 4, 7, 8, 9])
def test_right_hand_side_counts_match_single(nr):
    import defmm_amd as dm
    from defmm_amd import workloads as wl
    n = 2500
    pts = wl.cube_edges(n, seed=8)
    kappa = wl.kappa_for(3, pts)
    Q = np.stack([wl.charges(n, seed=40 + r) for r in range(nr)])
    _say(f"case: edge-refined cube N={n} L=3 Ncrit=21, {nr} right-hand sides")
    for prec, tol in ((dm.FP64, 1e-13), (dm.MIXED, 1e-6)):
        A = _plan(dm, pts, pts, 3, 21, kappa, prec)
        single = np.stack([A.apply(Q[r]) for r in range(nr)])
        A.set_rhs(nr)
        P = A.apply_batch(Q)
        A.destroy()
        l2, mx = _diff(P, single)
        _say(f"  precision {prec}: batch vs single rel L2 {l2:.3e} max {mx:.3e}")
        assert l2 <= tol and mx <= 10 * tol


# 16 right-hand sides take the matrix cores (float): row blocks of 16 targets,
# two per item, stages of 16 sources, sums to double every 64.  Single
# evaluations (compared with the oracle above) round the same float values in
# another order: the bounds of the test above.
@pytest.mark.parametrize("kappa", [0.0, 6.0, 1e-31])
@pytest.mark.parametrize("n,ncrit", [(900, 4), (1500, 18), (2500, 34), (3000, 130)])
def test_sixteen_right_hand_sides(n, ncrit, kappa):
    import defmm_amd as dm
    from defmm_amd import workloads as wl
    src = wl.sphere(n, seed=23)
    trg = np.concatenate([wl.sphere(n // 2 + 3, seed=6), src[:40]])  # some targets are sources
    nr = 17
    Q = np.stack([wl.charges(n, seed=60 + r) for r in range(nr)])
    _say(f"case: sphere N={n} Ncrit={ncrit} kappa={kappa}, {nr} right-hand sides")
    A = _plan(dm, src, trg, 3, ncrit, kappa, dm.MIXED)
    single = np.stack([A.apply(Q[r]) for r in range(nr)])
    A.set_rhs(nr)
    P = A.apply_batch(Q)
    again = A.apply_batch(Q)
    A.destroy()
    l2, mx = _diff(P, single)
    _say(f"  batch vs single rel L2 {l2:.3e} max {mx:.3e}")
    assert l2 <= 1e-6 and mx <= 1e-5
    assert np.array_equal(P, again)
