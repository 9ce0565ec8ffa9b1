"""Sums whose first child runs a Newton iteration of its own and whose records
hold optional tables: polynomials without a trim table, without streams, with
streams, first or later, in every kernel for Sums, against the oracle, bit for
bit; some of the rays miss or do not converge."""
import numpy as np
import pytest

import batoid_amd as bt
from batoid_amd import _lib
from batoid_amd.plan import PlanSpec, collect_steps

from helpers import (FCOLS, BCOLS, assert_cols_identical, bicubic_surface, random_rays,
                     zernike_surface)
from oracle.host import HostRays, HostPlan

pytestmark = pytest.mark.gpu


def polynomial(tables, seed):
    z = zernike_surface(seed=seed, jmax=28)
    rec, arrs = z._leaf_record()
    assert rec.flags == _lib.POLY_STREAMS
    if tables != "streams":
        rec.flags = 0
        kept = arrs[3][:1 + 3 * rec.n2].copy() if tables == "trim" else None
        z._leaf_record = lambda: (rec, arrs[:3] + (kept,))
    return z


def layouts(tables):
    asph = bt.Asphere(9.0, -0.9, [1e-3, -2e-4], imin=1)
    poly, grid = polynomial(tables, 71), bicubic_surface(seed=9)
    return dict(
        alone=poly,
        polynomial_first=bt.Sum(poly, asph, grid),
        polynomial_between=bt.Sum(asph, poly, grid),
        two_polynomials=bt.Sum(polynomial("streams", 72), poly),
        grid_first=bt.Sum(grid, poly),
        nested=bt.Sum(bt.Sum(poly, bt.Tilted(0.001, 0.0005)), asph))


@pytest.mark.parametrize("tables", ["none", "trim", "streams"])
@pytest.mark.parametrize("layout", list(layouts("none")))
@pytest.mark.parametrize("niter", [0, 1, 5])
def test_optional_tables(tables, layout, niter, monkeypatch):
    from batoid_amd import global_vars
    monkeypatch.setattr(global_vars, "_batoid_niter", niter)
    optic = bt.CompoundOptic([
        bt.Mirror(layouts(tables)[layout], name="M"),
        bt.Detector(bt.Plane(), name="D", coordSys=bt.CoordSys(origin=[0, 0, 2.5]))],
        name="o", inMedium=bt.ConstMedium(1.0))
    base = HostRays(**random_rays(1000, seed=6, z0=2.0, spread=0.4, radius=1.3))
    ref = HostPlan(PlanSpec(collect_steps(optic), bt.CoordSys())).trace(base.copy(), niter=niter)
    for fused in (True, False):
        rv = bt.RayVector(**{k: base[k] for k in FCOLS}, vignetted=base["vignetted"].astype(bool),
                          failed=base["failed"].astype(bool))
        if fused:
            optic.trace(rv)
        else:
            for item in optic.items:
                item.interact(rv)
        assert_cols_identical({k: getattr(rv, k) for k in FCOLS + BCOLS}, ref.cols,
                              what=f"{tables} {layout} {fused}")
        assert rv.failed.any() and (niter < 5 or not rv.failed.all())
