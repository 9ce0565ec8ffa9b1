"""Polynomial tables as streams of quads: the layout against the full 2-D
Horner loops in numpy on the CPU, and the GPU's sags and normals against the
oracle.  Sizes straddle what a stream holds: one coefficient, rows at and
beside multiples of four, 64 quads, and one row more (no stream).  Bar: the
full loops' bits (the steps added are +0.0 * y + 0.0)."""
import numpy as np
import pytest

import batoid_amd as bt
import oracle
from oracle.host import host_records, nthreads
from batoid_amd import _lib
from batoid_amd.surface import _horner_streams, _horner_trim


def _table(n, seed, holes):
    t = np.random.default_rng(seed).normal(size=(n, n)) * 0.3
    if holes and n > 2:
        t[n // 2] = 0.0                      # a row of +0.0
        t[0, 1:] = 0.0                       # a row of one coefficient
        t[-1, n // 3] = -0.0
        t[:, -1] = 0.0                       # no row runs to its end
    return t


def _full(x, y, t):
    r = np.float64(0.0)
    for row in t[::-1]:
        h = np.float64(0.0)
        for c in row[::-1]:
            h = h * y
            h = h + c
        r = r * x
        r = r + h
    return r


def _streamed(x, y, a3, n2, which):
    """The table as the device walks it; None without a stream."""
    start = -(-(1 + 3 * n2) // 16) * 16
    nquad, first = a3[start + 4 * which:start + 4 * which + 2]
    ends = int(a3[start + 4 * which + 2:start + 4 * which + 4].view(np.uint64)[0])
    data = a3[start + 16:].view(np.float64)
    assert first + 4 * nquad + 4 <= len(data)        # the quad read ahead
    if nquad == 0:
        return None
    r, h = np.float64(0.0), np.float64(0.0)
    for k in range(nquad):
        for c in data[first + 4 * k:first + 4 * k + 4]:
            h = h * y
            h = h + c
        if ends >> k & 1:
            r = r * x
            r = r + h
            h = np.float64(0.0)
    return r


@pytest.mark.parametrize("n", [1, 2, 4, 5, 8, 9, 16, 17])
@pytest.mark.parametrize("holes", [False, True])
def test_streams_give_the_full_loops_bits(n, holes):
    tables = [(_table(n, 3, holes), n, n)] + [
        (_table(n - 1, 4 + k, holes), n - 1, n - 1) for k in (0, 1)]
    a3 = _horner_streams(tables, _horner_trim(tables))
    assert a3.dtype == np.int32
    np.testing.assert_array_equal(a3[:1 + 3 * n], _horner_trim(tables))
    for x, y in [(0.3, -0.7), (-1.4, 1.1), (0.0, -0.0), (-0.0, 0.6), (1.2, 0.0), (1e-300, -1e300)]:
        x, y = np.float64(x), np.float64(y)
        for which, (t, nx, ny) in enumerate(tables):
            with np.errstate(all="ignore"):
                got, want = _streamed(x, y, a3, n, which), _full(x, y, t)
            if got is None:
                assert nx == 0 or nx == 17
                continue
            assert np.float64(got).tobytes() == np.float64(want).tobytes() or \
                (np.isnan(got) and np.isnan(want))


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 2, 4, 5, 8, 9, 16, 17])
@pytest.mark.parametrize("flagged", [True, False])
def test_polynomials_against_the_oracle(n, flagged):
    """Records with streams, and as they were without (trim table alone)."""
    z = bt.Zernike(np.zeros(4))
    z._xycoef = _table(n, 3, n % 2 == 0)
    z._xycoef_gradx = _table(n - 1, 4, n % 2 == 0)
    z._xycoef_grady = _table(n - 1, 5, False)
    if not flagged:
        rec, arrs = z._leaf_record()
        assert rec.flags == _lib.POLY_STREAMS
        rec.flags = 0
        z._leaf_record = lambda: (rec, arrs[:3] + (arrs[3][:1 + 3 * n].copy(),))
    N = 1000
    rng = np.random.default_rng(8)
    x, y = rng.uniform(-1.2, 1.2, N), rng.uniform(-1.2, 1.2, N)
    x[:3], y[1:4] = [0.0, -0.0, 0.0], [0.0, -0.0, 0.0]
    x[700], y[900] = np.nan, np.inf               # two waves of the full loops
    sag, nrm = np.empty(N), np.empty(3 * N)
    tab = host_records(z)
    O = oracle.load()
    with np.errstate(all="ignore"):
        O.or_sag_n(tab.ptr(), x.ctypes.data, y.ctypes.data, sag.ctypes.data, N, nthreads())
        O.or_normal_n(tab.ptr(), x.ctypes.data, y.ctypes.data, nrm.ctypes.data, N, nthreads())
    np.testing.assert_array_equal(z.sag(x, y), sag)
    np.testing.assert_array_equal(z.normal(x, y).T.ravel(), nrm)
