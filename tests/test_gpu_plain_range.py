"""Rays where x*x + y*y, a discriminant or the square of a velocity is below
2^-767, the least argument of the plain form's roots (some subnormal): the
oracle's bits, alone in a wave and among ordinary rays."""
import numpy as np
import pytest

import batoid_amd as bt
from batoid_amd import workloads
from batoid_amd.plan import PlanSpec, collect_steps

from helpers import assert_cols_identical, random_rays
from oracle.host import HostRays, HostPlan

pytestmark = pytest.mark.gpu

# one size for each wave of 64: a square that is 0 sends its wave to the full form
TINY = 10.0 ** -np.arange(110.0, 164.0, 2.0)


def scales(rng, i):
    """Sizes for rays ``i``, TINY[k mod len] for wave k."""
    return TINY[(i // 64) % len(TINY)] * rng.uniform(1, 10, len(i))


def check(optic, rv, what):
    ref = HostRays.from_rv(rv)
    HostPlan(PlanSpec(collect_steps(optic), rv.coordSys)).trace(ref)
    optic.trace(rv)
    assert_cols_identical({k: getattr(rv, k) for k in ref.cols}, ref, what=what)


@pytest.mark.parametrize("name", ["tma", "perturbed", "freeform"])
@pytest.mark.parametrize("every", [1, 3])
def test_both_coordinates_tiny(name, every):
    optic = dict(tma=workloads.tma, perturbed=workloads.perturbed_tma,
                 freeform=workloads.freeform_tma)[name]()
    thx, thy = workloads.tma_fields()
    rv = workloads.tma_rays(optic, thx[5], thy[5], 620e-9, nrad=14, naz=130)
    cols = {k: getattr(rv, k).copy() for k in ("x", "y", "z", "vx", "vy", "vz", "t")}
    rng = np.random.default_rng(12)
    i = np.arange(0, len(rv), every)
    th = rng.uniform(0, 2 * np.pi, len(i))
    cols["x"][i], cols["y"][i] = scales(rng, i) * np.array([np.cos(th), np.sin(th)])
    cols["z"][i] = 14.0
    cols["vx"][i], cols["vy"][i], cols["vz"][i] = 0.0, -0.0, -1.0
    check(optic, bt.RayVector(**cols, wavelength=620e-9, coordSys=rv.coordSys), f"{name} {every}")


MIRRORS = [bt.Sphere(2.3), bt.Sphere(-3.1), bt.Paraboloid(4.5), bt.Quadric(6.1, -0.7),
           bt.Asphere(9.0, -0.9, [1e-3, -2e-4], imin=1)]


@pytest.mark.parametrize("surface", MIRRORS, ids=lambda s: type(s).__name__ + str(s.R))
@pytest.mark.parametrize("every", [1, 3])
@pytest.mark.parametrize("lens", [False, True])
def test_tiny_velocities(surface, every, lens):
    """Discriminants and 1/|v| of velocities whose squares are tiny; into the
    lens along the axis, where they refract."""
    glass, air = bt.ConstMedium(1.1), bt.ConstMedium(1.0)
    items = [bt.RefractiveInterface(bt.Plane(), name="L", inMedium=air, outMedium=glass)] if lens \
        else [bt.Mirror(surface, name="M", inMedium=air, outMedium=air)]
    optic = bt.CompoundOptic(items + [
        bt.Detector(bt.Plane(), name="D", coordSys=bt.CoordSys(origin=[0, 0, -3.0 if lens else 3.0]))],
        name="o", inMedium=air)
    n = 64 * len(TINY)
    c = random_rays(n, seed=6, z0=2.0, spread=0.05, radius=1.1, prefail=0, previg=0)
    rng = np.random.default_rng(4)
    i = np.arange(0, n, every)
    scale = scales(rng, i)
    if lens:
        c["vx"][i], c["vy"][i], c["vz"][i] = 0.0, 0.0, -1.0
    for k in ("vx", "vy", "vz"):
        c[k][i] *= scale
    check(optic, bt.RayVector(**c), f"{surface!r} {every}")
