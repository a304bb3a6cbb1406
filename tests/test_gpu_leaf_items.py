"""Plans whose source leaves have no direction slots (their cells take part in
no M2L): all of them, some of them, and sources far from a small patch of
targets.  Whole evaluations of 1 and of 17 right-hand sides (matrix cores and
one more) are compared with the oracle, at the bounds of the other
comparisons with it."""
import sys

import numpy as np
import pytest

import oracle_api as oa

pytestmark = pytest.mark.gpu


def _say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


@pytest.mark.parametrize("n,m,ncrit,nl", [(200, 0, 5, 10), (300, 0, 5, 10), (4000, 200, 33, 8)])
def test_leaves_without_slots(n, m, ncrit, nl):
    import defmm_amd as dm
    from defmm_amd import workloads as wl
    src = trg = wl.sphere(n, seed=31)
    if m:  # a cap around a pole
        t = wl.sphere(40 * m, seed=5)
        trg = np.ascontiguousarray(t[np.argsort(-t[:, 2])[:m]])
    kappa = wl.kappa_for(nl, src, trg)
    q = wl.charges(n, seed=13)
    st = dm.build_plan_stats(src, trg, 4, ncrit, kappa)
    _say(f"case: sphere N={n} targets {len(trg)} {nl} wavelengths L=4 Ncrit={ncrit}: "
         f"{st['hf_leaves']} leaves, {st['src_slots']} source slots")
    po, _, _, _ = oa.fmm(src, trg, q, 4, ncrit, kappa)
    for prec, l2max, mxmax in ((dm.FP64, 1e-12, 1e-10), (dm.MIXED, 3e-6, 3e-5)):
        A = dm.IBFMM_Mat(precision=prec)
        A.setSourceParticles(src)
        A.setTargetParticles(trg)
        A.prcmpt(4, ncrit, kappa)
        p = A.apply(q)
        A.set_rhs(17)
        P = A.apply_batch(np.stack([q * (1 + r) for r in range(17)]))
        A.destroy()
        for r, x in [(0, p)] + [(r, P[r]) for r in range(17)]:
            d = np.abs(x - po * (1 + r))
            l2 = np.sqrt((d ** 2).sum() / (np.abs(po * (1 + r)) ** 2).sum())
            mx = d.max() / np.abs(po * (1 + r)).max()
            if r in (0, 16):
                _say(f"  precision {prec} right-hand side {r}: rel L2 {l2:.3e} max {mx:.3e}")
            assert l2 <= l2max and mx <= mxmax
