"""Near-field work items in the plan's statistics: those of the kernel that the
plan's precision and width take (targets in chunks of 8 with a lane per source,
of 32 on the matrix cores: mixed precision, 8 right-hand sides and more)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_p2p_items_follow_precision_and_width():
    import defmm_amd as dm
    from defmm_amd import workloads as wl
    pts = wl.sphere(3000, seed=3)
    print("case: sphere N=3000 Ncrit=40, items of the near field", flush=True)
    A = dm.IBFMM_Mat(precision=dm.FP64)
    A.setSourceParticles(pts)
    A.setTargetParticles(pts)
    A.prcmpt(3, 40, wl.kappa_for(3, pts))
    lane = A.stats()["p2p_items"]
    A.set_rhs(16)
    assert A.stats()["p2p_items"] == lane
    A.set_precision(dm.MIXED)
    wide = A.stats()["p2p_items"]
    A.set_option(dm.OPT_P2P_MFMA, 0)
    assert A.stats()["p2p_items"] == lane
    A.set_option(dm.OPT_P2P_MFMA, 1)
    A.set_rhs(8)
    assert A.stats()["p2p_items"] == wide
    A.set_rhs(7)
    assert A.stats()["p2p_items"] == lane
    A.destroy()
    assert 0 < wide < lane
