"""Rounding errors of the mixed path with 8 right-hand sides (against FP64
single evaluations of the same points): the near field on the matrix cores is
no less exact than with a lane per source."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("geo,n,waves,L,ncrit", [("cube_edges", 20000, 32, 8, 257),
                                                 ("cube_edges", 20000, 16, 5, 65),
                                                 ("ellipsoid", 20000, 16, 6, 97)])
def test_eight_right_hand_sides_round_as_single_ones(geo, n, waves, L, ncrit):
    import defmm_amd as dm
    from defmm_amd import workloads as wl
    print(f"case: {geo} N={n} {waves} wavelengths L={L} Ncrit={ncrit}, 8 right-hand sides",
          flush=True)
    pts = wl.GEOMETRIES[geo](n, seed=3)
    kappa = wl.kappa_for(waves, pts)
    Q = np.stack([wl.charges(n, seed=9 + r).astype(np.complex64).astype(np.complex128)
                  for r in range(8)])
    A = dm.IBFMM_Mat(precision=dm.FP64)
    A.setSourceParticles(pts)
    A.setTargetParticles(pts)
    A.prcmpt(L, ncrit, kappa)
    exact = np.stack([A.apply(q) for q in Q])
    A.set_precision(dm.MIXED)
    A.set_rhs(8)

    def err(mfma):
        A.set_option(dm.OPT_P2P_MFMA, mfma)
        d = A.apply_batch(Q) - exact
        return np.sqrt((np.abs(d) ** 2).sum() / (np.abs(exact) ** 2).sum())

    lanes, cores = err(0), err(1)
    A.destroy()
    print(f"  rel L2: a lane per source {lanes:.4e}, matrix cores {cores:.4e}", flush=True)
    # 8 x 20,000 errors: the two means of squares scatter by well below 2%
    assert cores <= 1.02 * lanes
