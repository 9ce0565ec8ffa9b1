"""Frame changes by the unit matrix, which the kernels of analytic surfaces
compute with FMAs: bit for bit (signs of zeros too) the oracle's products and
sums, on rays with zeros of either sign, infinities, NaNs and denormals, for
unit matrices with zeros of either sign and for one an ulp beside it."""
import numpy as np
import pytest

import batoid_amd as bt
from oracle.host import HostRays, HostPlan
from batoid_amd import _device, _lib
from batoid_amd.plan import DevicePlan, PlanSpec, collect_steps
from helpers import random_rays, FCOLS, BCOLS

pytestmark = pytest.mark.gpu


def _rot(kind):
    m = np.eye(3)
    if kind == "ulp":
        m[1, 1] = np.nextafter(1.0, 2.0)
    elif kind == "rotated":
        m = bt.RotX(1e-3) @ bt.RotY(2e-3)
    return m


@pytest.mark.parametrize("kind", ["unit", "signed", "ulp", "rotated"])
@pytest.mark.parametrize("n", [1, 63, 65, 1000])
def test_unrotated_frames(kind, n):
    cs = [bt.CoordSys(origin=[0, 0, z], rot=_rot(kind)) for z in (0.0, 2.5, 5.0)]
    optic = bt.CompoundOptic([
        bt.Mirror(bt.Paraboloid(10.0), name="M", coordSys=cs[0]),
        bt.RefractiveInterface(bt.Sphere(-30.0), name="L", coordSys=cs[1],
                               inMedium=bt.ConstMedium(1.0), outMedium=bt.ConstMedium(1.4)),
        bt.Detector(bt.Plane(), name="D", coordSys=cs[2])], name="o", inMedium=bt.ConstMedium(1.0))
    base = HostRays(**random_rays(n, seed=5, z0=2.0, spread=0.05, radius=1.1))
    special = [0.0, -0.0, np.nan, np.inf, -np.inf, 5e-324, -5e-324]
    for j, c in enumerate(("x", "y", "vx", "vy", "z", "vz")):
        for k, v in enumerate(special[:2] if c in ("z", "vz") else special):
            if 7 * j + k + 1 < n // 2:
                base[c][7 * j + k + 1] = v
    base["x"][-1:] = -0.0
    base["vx"][-1:] = -0.0
    spec = PlanSpec(collect_steps(optic), bt.CoordSys())
    assert spec.flags & _lib.PLAN_ANALYTIC
    if kind == "signed":
        for j, step in enumerate(spec.steps):
            for e in ((1, 5, 6, 7), (2, 3, 5), (1, 2, 3, 5, 6, 7))[j]:
                step.drot[e] = -0.0
    with np.errstate(all="ignore"):
        ref = HostPlan(spec).trace(base.copy(), niter=5)
    rv = bt.RayVector(**{k: base[k] for k in FCOLS}, vignetted=base["vignetted"].astype(bool),
                      failed=base["failed"].astype(bool))
    plan = DevicePlan(spec)
    _lib.call("bt_trace_plan", plan.struct, rv._rays, rv._rays, 5, _device.stream())
    for k in FCOLS:
        got, want = getattr(rv, k), ref.cols[k]
        same = (got.view(np.uint64) == want.view(np.uint64)) | (np.isnan(got) & np.isnan(want))
        assert same.all(), k
    for k in BCOLS:
        np.testing.assert_array_equal(getattr(rv, k), np.asarray(ref.cols[k], dtype=bool))
