"""Aspheres of no, odd and even numbers of terms, alone and as the first child
of a Sum, whose two Newton iterations both test for terms: the plan kernels of
analytic surfaces and of perturbed mirrors and the per-surface kernels against
the oracle, bit for bit."""
import numpy as np
import pytest

import batoid_amd as bt
from oracle.host import HostRays, HostPlan
from batoid_amd.plan import PlanSpec, collect_steps
from helpers import random_rays, assert_cols_identical, bicubic_surface, zernike_surface, FCOLS, BCOLS

pytestmark = pytest.mark.gpu

TERMS = [1e-3, -2e-4, 3e-5, -4e-6, 5e-7, -6e-8, 7e-9]


@pytest.mark.parametrize("n", range(8))
@pytest.mark.parametrize("layout", ["alone", "sum"])
@pytest.mark.parametrize("fused", [True, False])
def test_terms(n, layout, fused):
    surf = bt.Asphere(9.0, -0.9, TERMS[:n], imin=1)
    if layout == "sum":
        surf = bt.Sum(surf, zernike_surface(seed=71, jmax=28), bicubic_surface(seed=9))
    optic = bt.CompoundOptic([
        bt.Mirror(surf, name="M"),
        bt.Detector(bt.Plane(), name="D", coordSys=bt.CoordSys(origin=[0, 0, 2.5]))],
        name="o", inMedium=bt.ConstMedium(1.0))
    base = HostRays(**random_rays(1000, seed=6, z0=2.0, spread=0.05, radius=1.1))
    ref = HostPlan(PlanSpec(collect_steps(optic), bt.CoordSys())).trace(base.copy(), niter=5)
    rv = bt.RayVector(**{k: base[k] for k in FCOLS}, vignetted=base["vignetted"].astype(bool),
                      failed=base["failed"].astype(bool))
    if fused:
        optic.trace(rv)
    else:
        for item in optic.items:
            item.interact(rv)
    assert_cols_identical({k: getattr(rv, k) for k in FCOLS + BCOLS}, ref.cols, what=f"{n} {layout}")
