"""A segment's image is the same bits whatever else is in the batch: units of
halves or quarters, one or eight lanes per pixel in the reduction (2^18 pixels
and more, or fewer).  Fluxes over twelve decades: FP64 sums of like FP32
numbers are exact and would hide their order."""
import numpy as np
import pytest
import torch

from batoid_amd import workloads
from batoid_amd.batch import PSFBatch

pytestmark = pytest.mark.gpu


def amplitudes(optic, thx, thy, nx, first, **args):
    """Of segments ``first`` on; segment s has the fluxes of seed s."""
    batch = PSFBatch(optic, thx, thy, 620e-9, nx, **args)
    flux = np.concatenate([10.0 ** np.random.default_rng(first + s).uniform(-12, 0, n * n)
                           for s, n in enumerate(nx)])
    batch.rays_in.torch("flux").copy_(torch.from_numpy(flux))
    return batch.run().amplitudes()


@pytest.mark.parametrize("precision", ["fp32", "bf16x3"])
@pytest.mark.parametrize("out,segments", [(1, 6), (75, 6), (75, 47), (130, 6), (257, 6)])
def test_same_bits_in_any_batch(out, segments, precision):
    optic = workloads.tma()
    thx, thy = workloads.tma_fields()
    thx, thy = np.resize(thx, segments), np.resize(thy, segments)
    nx = np.resize([61, 58, 17, 60, 2, 59], segments)
    args = dict(nxOut=out, dx=0.5e-6, precision=precision, chunk=8)
    many = amplitudes(optic, thx, thy, nx, 0, **args)
    for s in (0, 1, 2, 4, segments - 1):
        one = amplitudes(optic, thx[s:s + 1], thy[s:s + 1], nx[s:s + 1], s, **args)[0]
        np.testing.assert_array_equal(many[s].view(np.uint64), one.view(np.uint64))
