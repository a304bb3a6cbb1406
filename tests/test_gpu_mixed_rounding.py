"""Rounding errors of the mixed path's far field (against FP64 of the same
plan, which differs by nothing but rounding) for single right-hand sides,
whose L2P of leaves with 24 slots and more runs on the matrix cores: no larger
than with the vector kernel for every leaf, which was measured on the same
points and charges (40,000 points on a sphere, 24 wavelengths, Ncrit 65, mean
over three right-hand sides)."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,vector", [(5, 3.6487e-7), (6, 4.7713e-7), (7, 6.4473e-7),
                                      (8, 8.4806e-7)])
def test_far_field_rounds_no_worse_than_the_vector_kernel(L, vector):
    import defmm_amd as dm
    from defmm_amd import workloads as wl
    n = 40000
    pts = wl.sphere(n, seed=3)
    kappa = wl.kappa_for(24, pts)
    Q = [wl.charges(n, seed=9 + r).astype(np.complex64).astype(np.complex128) for r in range(3)]
    print(f"case: sphere N={n} 24 wavelengths L={L}, far only", flush=True)
    p = {}
    for prec in (dm.FP64, dm.MIXED):
        A = dm.IBFMM_Mat(precision=prec)
        A.setSourceParticles(pts)
        A.setTargetParticles(pts)
        A.prcmpt(L, 65, kappa)
        p[prec] = [A.apply(q, parts=2) for q in Q]
        A.destroy()
    err = np.mean([np.sqrt((np.abs(a - b) ** 2).sum() / (np.abs(b) ** 2).sum())
                   for a, b in zip(p[dm.MIXED], p[dm.FP64])])
    print(f"  rel L2 {err:.4e}, vector kernel {vector:.4e}", flush=True)
    sys.stdout.flush()
    assert err <= vector
