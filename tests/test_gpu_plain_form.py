"""The plain form of the trace kernels (roots, reciprocals and quotients
without range handling) and the vote that sends a wave to the full form:
rays at the edges of the plain range, alone and among ordinary ones, give the
oracle's bits, whatever shares their wave."""
import numpy as np
import pytest

import batoid_amd as bt
from batoid_amd import workloads
from batoid_amd.plan import PlanSpec, collect_steps

from helpers import assert_cols_identical
from oracle.host import HostRays, HostPlan

pytestmark = pytest.mark.gpu

# positions and direction slopes at and beyond the plain range
EDGES = [0.0, -0.0, 1e-17, 1e-115, 1e-120, 1e-180, 1e-182, 1e-300, 5e-324, 2.5, 4.0, 1e60, 1e155,
         1e200, np.inf, np.nan]


def edge_rays(optic, every, nrad=14, naz=130):
    """Ordinary pupil rays with an edge ray at each ``every``-th place."""
    thx, thy = workloads.tma_fields()
    rv = workloads.tma_rays(optic, thx[5], thy[5], 620e-9, nrad=nrad, naz=naz)
    cols = {k: getattr(rv, k).copy() for k in ("x", "y", "z", "vx", "vy", "vz", "t")}
    n = len(rv)
    pairs = [(a, b) for a in EDGES for b in EDGES]
    for k, i in enumerate(range(0, n, every)):
        a, b = pairs[(7 * k) % len(pairs)]
        cols["x"][i], cols["y"][i], cols["z"][i] = a, b, 14.0
        if k % 3 == 0:                               # along the axis
            cols["vx"][i], cols["vy"][i], cols["vz"][i] = 0.0, -0.0, -1.0
        elif k % 3 == 1:
            cols["vx"][i], cols["vy"][i], cols["vz"][i] = 1e-300, 0.0, -1.0
    return bt.RayVector(**cols, wavelength=620e-9, coordSys=rv.coordSys)


def optic_of(name):
    return dict(tma=workloads.tma, perturbed=workloads.perturbed_tma,
                freeform=workloads.freeform_tma)[name]()


@pytest.mark.parametrize("name", ["tma", "perturbed", "freeform"])
@pytest.mark.parametrize("every", [1, 3, 64, 191])
def test_edge_rays_bit_exact(name, every):
    optic = optic_of(name)
    rv = edge_rays(optic, every)
    ref = HostRays.from_rv(rv)
    HostPlan(PlanSpec(collect_steps(optic), rv.coordSys)).trace(ref)
    step = rv.copy()
    optic.trace(rv)
    assert_cols_identical({k: getattr(rv, k) for k in ref.cols}, ref, what=f"{name} {every}")
    for iface, _, _ in collect_steps(optic):         # the per-surface kernels
        iface.trace(step)
    assert_cols_identical({k: getattr(step, k) for k in ref.cols}, ref,
                          what=f"{name} {every} by surface")


@pytest.mark.parametrize("name", ["tma", "perturbed", "freeform"])
def test_conic_start_is_independent_of_the_wave(name):
    optic = optic_of(name)
    rv = edge_rays(optic, 3)
    mixed = optic.trace(rv.copy(), start="conic")
    edge = np.arange(len(rv)) % 3 == 0
    for part in (edge, ~edge):
        alone = optic.trace(rv[part], start="conic")
        cols = ("x", "y", "z", "vx", "vy", "vz", "t", "vignetted", "failed")
        assert_cols_identical({k: getattr(alone, k) for k in cols},
                              {k: getattr(mixed, k)[part] for k in cols}, cols=cols, what=name)


@pytest.mark.parametrize("policy", ["nan", "zero"])
@pytest.mark.parametrize("table", ["wavy", "flat", "descending", "two"])
@pytest.mark.parametrize("reciprocals", [True, False])
def test_bicubic_cells_bit_exact(policy, table, reciprocals):
    """Rays on grid lines and nodes, on and past the edges, through a Bicubic
    with and without its record's optional reciprocals of the steps."""
    nx, ny = (2, 2) if table == "two" else (9, 7)
    xs, ys = np.linspace(-0.8, 0.8, nx), np.linspace(-0.6, 0.6, ny)
    if table == "descending":
        xs = xs[::-1]
    zs = 0.0 * np.add.outer(ys, xs) if table == "flat" else \
        1e-3 * np.add.outer(np.sin(5 * ys), np.cos(4 * xs))
    surf = bt.Bicubic(xs, ys, zs, nanpolicy=policy)
    if not reciprocals:
        recs = surf._leaf_record

        def without():
            rec, arrs = recs()
            rec.p[4] = rec.p[5] = 0.0
            return rec, arrs
        surf._leaf_record = without
    optic = bt.CompoundOptic([bt.Mirror(surf, name="M"),
                              bt.Detector(bt.Plane(), name="D",
                                          coordSys=bt.CoordSys().shiftGlobal([0, 0, 1]))])
    rng = np.random.default_rng(3)
    n = 6 * 64 + 5
    x, y = rng.uniform(-0.9, 0.9, n), rng.uniform(-0.7, 0.7, n)
    x[::3], y[1::3] = rng.choice(xs, len(x[::3])), rng.choice(ys, len(y[1::3]))
    x[5::50], y[5::50] = 0.0, -0.0
    x[7::50] = np.nextafter(0.8, 1)
    vx = np.where(np.arange(n) % 2, 0.0, rng.normal(0, 1e-2, n))
    rv = bt.RayVector(x, y, 1.0, vx, 0.0, -1.0, wavelength=500e-9)
    ref = HostRays.from_rv(rv)
    HostPlan(PlanSpec(collect_steps(optic), rv.coordSys)).trace(ref)
    optic.trace(rv)
    assert_cols_identical({k: getattr(rv, k) for k in ref.cols}, ref, what=f"{table} {policy}")
