"""A beam wider than the pupil, part of which leaves the lenses' aspheres: the
oracle's bits, and no second pass over what its waves had already traced."""
import os

import numpy as np
import pytest
import torch

import batoid_amd as bt
from batoid_amd import _device, _lib
from batoid_amd.plan import PlanSpec, collect_steps

from helpers import FCOLS, BCOLS, assert_cols_identical
from oracle.host import HostRays, HostPlan

pytestmark = pytest.mark.gpu

GOLD = os.path.join(os.path.dirname(__file__), "golden", "optics")


def beam(optic, nx, width, theta):
    return bt.RayVector.asGrid(optic=optic, wavelength=620e-9, nx=nx, theta_x=theta,
                               theta_y=0.3 * theta, lx=optic.pupilSize * width)


@pytest.mark.parametrize("name", ["HSC.yaml", "DECam.yaml", "LSST_r.yaml"])
@pytest.mark.parametrize("width", [1.0, 1.6, 3.0])
def test_overfilled_bit_exact(name, width):
    optic = bt.Optic.fromYaml(os.path.join(GOLD, name))
    rv = beam(optic, 48, width, 0.004)
    ref = HostRays.from_rv(rv)
    HostPlan(PlanSpec(collect_steps(optic), rv.coordSys)).trace(ref)
    optic.trace(rv)
    assert_cols_identical({k: getattr(rv, k) for k in FCOLS + BCOLS}, ref.cols, what=name)


def test_overfilled_waves_stop_where_they_leave():
    """208 us with the plan run to its end in the plain and then in the full
    form, against 126 for the beam as wide as the pupil; 152 and 128 now."""
    optic = bt.Optic.fromYaml(os.path.join(GOLD, "HSC.yaml"))

    def kernel_time(width):
        rv = beam(optic, 512, width, 0.0)
        plan, out = optic._plan(rv.coordSys, False, None), rv.copy()
        best = np.inf
        for _ in range(8):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            for _ in range(20):
                _lib.call("bt_trace_plan", plan.struct, rv._rays, out._rays, 5, _device.stream())
            b.record()
            b.synchronize()
            best = min(best, a.elapsed_time(b) / 20)
        return best, out

    kernel_time(1.0)
    (filled, _), (over, out) = kernel_time(1.0), kernel_time(1.6)
    assert out.failed.mean() > 0.2
    assert over < 1.45 * filled, f"{over * 1e3} us, {filled * 1e3} for the filled pupil"
