"""Host side of a polynomial's record: its trim tables and streams take no longer
to make than the trim tables alone did with a numpy call per row, since a new
optic makes them before its first trace."""
import time

import numpy as np
import pytest

import batoid_amd as bt


def _trim_by_rows(tables):
    out = []
    for flat, nx, ny in tables:
        flat = np.ascontiguousarray(flat, dtype=np.float64).ravel()
        if ny > 0 and nx > 0:
            rows = flat[:nx * ny].reshape(ny, nx).view(np.uint64) != 0
            lens = [int(np.flatnonzero(row)[-1]) + 1 if row.any() else 0 for row in rows]
        else:
            lens = [0] * max(ny, 0)
        out += [max([i for i, n in enumerate(lens) if n > 0], default=-1)] + lens
    return np.array(out, dtype=np.int32)


def _tables(jmax):
    z = bt.Zernike(np.random.default_rng(jmax).normal(0, 5e-8, jmax + 1), R_outer=4.0)
    n = len(z._xycoef)
    return z, [(z._xycoef, n, n), (z._xycoef_gradx, n - 1, n - 1), (z._xycoef_grady, n - 1, n - 1)]


def _best(f):
    best = np.inf
    for _ in range(40):
        t = time.perf_counter()
        for _ in range(20):
            f()
        best = min(best, time.perf_counter() - t)
    return best / 20


@pytest.mark.parametrize("jmax", [1, 4, 28, 66])
def test_trim_by_rows(jmax):
    from batoid_amd.surface import _horner_trim
    _, tables = _tables(jmax)
    np.testing.assert_array_equal(_horner_trim(tables), _trim_by_rows(tables))


@pytest.mark.parametrize("jmax", [28, 66])
def test_record_takes_no_longer_than_its_trim_did(jmax):
    from batoid_amd.surface import _horner_trim, _horner_streams
    _, tables = _tables(jmax)
    _horner_streams(tables, _horner_trim(tables))
    for _ in range(3):                               # a busy machine: try again
        now = _best(lambda: _horner_streams(tables, _horner_trim(tables)))
        before = _best(lambda: _trim_by_rows(tables))
        if now < before:
            return
    assert now < before, f"{now * 1e6:.0f} us, {before * 1e6:.0f} us before"
