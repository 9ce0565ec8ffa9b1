"""The batched PSF's units (64 x 128 halves of a tile, or 64 x 64 quarters
where halves would leave the chip idle) and its two reductions: a segment's
image does not depend on the batch it is in."""
import numpy as np
import pytest

from batoid_amd import workloads
from batoid_amd.batch import PSFBatch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp32", "bf16x3"])
@pytest.mark.parametrize("out,chunk", [(1, 8), (33, 8), (64, 64), (75, 8), (128, 8), (130, 16),
                                       (257, 8)])
def test_image_is_independent_of_the_batch(out, chunk, precision):
    """Six segments (1,300 items of 8 rays and fewer: halves, and for the
    larger images one lane per pixel) against each alone (quarters).  The
    FP32 sums are the same operations; the items' FP64 sum may be in another
    order: at most K terms of at most max|part| each, K 2^-53 relative."""
    optic = workloads.tma()
    thx, thy = workloads.tma_fields()
    nx = np.array([61, 58, 17, 60, 2, 59])
    args = dict(nxOut=out, dx=0.5e-6, precision=precision, chunk=chunk)
    many = PSFBatch(optic, thx[:6], thy[:6], 620e-9, nx, **args).run().amplitudes()
    for s in range(6):
        one = PSFBatch(optic, thx[s:s + 1], thy[s:s + 1], 620e-9, nx[s:s + 1],
                       **args).run().amplitudes()[0]
        terms = nx[s] ** 2 / chunk + 1
        tol = terms ** 2 * 2.0 ** -53 * chunk        # K terms of up to `chunk` unit amplitudes
        assert np.abs(many[s] - one).max() <= tol
