"""Near field of 8 right-hand sides on the matrix cores (float): row blocks of
16 targets, two per item, stages of 16 sources, sums to double every 64, real
and imaginary parts in the two halves of one result; 8 alone, with the vector
kernels for the rest (15) and after 16 (24).  Single evaluations (compared with
the oracle elsewhere) round the same float values in another order: the bounds
are those of a few roundings of the sums, as for 16 right-hand sides."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nr", [8, 15, 24])
@pytest.mark.parametrize("n,ncrit,kappa", [(900, 4, 6.0), (1500, 18, 0.0), (2500, 34, 6.0),
                                           (3000, 130, 1e-31), (3000, 130, 6.0)])
def test_eight_right_hand_sides(n, ncrit, kappa, nr):
    import defmm_amd as dm
    from defmm_amd import workloads as wl
    src = wl.sphere(n, seed=23)
    trg = np.concatenate([wl.sphere(n // 2 + 3, seed=6), src[:40]])  # some targets are sources
    Q = np.stack([wl.charges(n, seed=60 + r) for r in range(nr)])
    print(f"case: sphere N={n} Ncrit={ncrit} kappa={kappa}, {nr} right-hand sides", flush=True)
    A = dm.IBFMM_Mat(precision=dm.MIXED)
    A.setSourceParticles(src)
    A.setTargetParticles(trg)
    A.prcmpt(3, ncrit, kappa)
    single = np.stack([A.apply(Q[r]) for r in range(nr)])
    A.set_rhs(nr)
    P = A.apply_batch(Q)
    again = A.apply_batch(Q)
    A.set_option(dm.OPT_P2P_MFMA, 0)
    V = A.apply_batch(Q)
    A.destroy()
    for x in (P, V):
        d = np.abs(x - single)
        l2 = np.sqrt((d ** 2).sum() / (np.abs(single) ** 2).sum())
        mx = d.max() / np.abs(single).max()
        print(f"  batch vs single rel L2 {l2:.3e} max {mx:.3e}", flush=True)
        assert l2 <= 1e-6 and mx <= 1e-5
    assert np.array_equal(P, again)
    sys.stdout.flush()
