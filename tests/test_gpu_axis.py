"""Rays that meet surfaces at their vertices (the chief ray of a centred field):
the oracle's bits, zeros' signs included, and one pass of the kernel."""
import numpy as np
import pytest
import torch

import batoid_amd as bt
from batoid_amd import _device, _lib, workloads
from batoid_amd.plan import PlanSpec, collect_steps

from helpers import (FCOLS, BCOLS, assert_cols_identical, bicubic_surface, random_rays,
                     zernike_surface)
from oracle.host import HostRays, HostPlan

pytestmark = pytest.mark.gpu

SURFACES = dict(
    sphere=bt.Sphere(2.3), sphere_back=bt.Sphere(-3.1), quadric=bt.Quadric(6.1, -0.7),
    quadric_back=bt.Quadric(-8.0, 0.4), paraboloid=bt.Paraboloid(-4.5), plane=bt.Plane(),
    tilted=bt.Tilted(0.0, -0.0), asphere=bt.Asphere(5.0, 0.2, [1e-3, -2e-4, 3e-6], imin=1),
    asphere_back=bt.Asphere(-5.0, -1.0, []), polynomial=zernike_surface(),
    apb=bt.Sum(bt.Asphere(9.0, -0.9, [1e-4]), zernike_surface(seed=58), bicubic_surface(seed=6)),
    flat=bt.Sum(bt.Quadric(-7.0, -0.4), bt.Sphere(40.0)),
    nested=bt.Sum(bt.Sum(bt.Sphere(9.0), bt.Plane()), bt.Quadric(30.0, 1.0)))


def axis_rays(every):
    """Rays at and to the vertex with zeros of either sign among others; some
    come to it from the side, some at right angles to the axis."""
    c = random_rays(1000, seed=6, z0=2.0, spread=0.05, radius=0.5, prefail=0, previg=0)
    zeros = [0.0, -0.0]
    for k, i in enumerate(range(0, 1000, every)):
        for j, name in enumerate(("x", "y", "vx", "vy")):
            c[name][i] = zeros[k >> j & 1]
        c["vz"][i] = [-1.0, 1.0, -0.5, -1.0][k // 16 % 4]
        c["z"][i] = [2.0, 0.0, 1.0, -0.0][k // 64 % 4]
        if k % 5 == 3:                               # x + vx dt = 0 at z = 0
            c["x"][i], c["vx"][i], c["z"][i], c["vz"][i] = -0.25, 0.125, 2.0, -1.0
        if k % 50 == 7:
            c["x"][i], c["z"][i], c["vx"][i], c["vz"][i] = 0.0, 0.0, 1.0, 0.0
    return c


@pytest.mark.parametrize("name", list(SURFACES))
@pytest.mark.parametrize("every", [1, 3, 70])
@pytest.mark.parametrize("refract", [False, True])
def test_vertex_bit_exact(name, every, refract):
    glass, air = bt.ConstMedium(1.5), bt.ConstMedium(1.0)
    if refract:
        first = bt.RefractiveInterface(SURFACES[name], name="S", inMedium=air, outMedium=glass)
    else:
        first = bt.Mirror(SURFACES[name], name="S", inMedium=air, outMedium=air)
    last = bt.Mirror(bt.Sphere(50.0), name="T", coordSys=bt.CoordSys(origin=[0, 0, 4.0]),
                     inMedium=first.outMedium, outMedium=first.outMedium)
    optic = bt.CompoundOptic([first, last], name="o", inMedium=air)
    base = HostRays(**axis_rays(every))
    ref = HostPlan(PlanSpec(collect_steps(optic), bt.CoordSys())).trace(base.copy(), niter=5)
    for fused in (True, False):
        rv = bt.RayVector(**{k: base[k] for k in FCOLS})
        if fused:
            optic.trace(rv)
        else:
            for item in optic.items:
                item.interact(rv)
        assert_cols_identical({k: getattr(rv, k) for k in FCOLS + BCOLS}, ref.cols,
                              what=f"{name} {every} {refract} {fused}")


@pytest.mark.parametrize("name", ["tma", "perturbed"])
def test_centred_field_takes_one_pass(name):
    """A wave with the chief ray of a centred field ran in the plain and then in
    the full form: 2.0 and 1.9 times the time of the same rays off the axis."""
    optic = dict(tma=workloads.tma, perturbed=workloads.perturbed_tma)[name]()

    def kernel_time(theta):
        rv = bt.RayVector.asGrid(optic=optic, wavelength=620e-9, nx=7, theta_x=theta, theta_y=0.0)
        assert (theta == 0) == bool(((rv.x == 0) & (rv.y == 0)).any())
        plan, out = optic._plan(rv.coordSys, False, None), rv.copy()
        best = np.inf
        for _ in range(8):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            for _ in range(40):
                _lib.call("bt_trace_plan", plan.struct, rv._rays, out._rays, 5, _device.stream())
            b.record()
            b.synchronize()
            best = min(best, a.elapsed_time(b) / 40)
        return best

    kernel_time(0.0)
    on, off = kernel_time(0.0), kernel_time(0.01)
    assert on < 1.4 * off, f"{on * 1e3} us on the axis, {off * 1e3} off"
