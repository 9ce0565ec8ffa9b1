"""PSFBatch.autotune's choice from measured times: the shortest run, but no
longer FP32 sums (larger chunks) than a real difference pays for."""
import pytest

from batoid_amd.batch import PSFBatch


@pytest.mark.parametrize("times,chosen", [
    ({(1024, 512): 25.17, (1024, 1024): 25.14, (2048, 512): 24.98, (2048, 1024): 24.94,
      (4096, 512): 25.9, (4096, 1024): 25.92}, (1024, 1024)),
    ({(1024, 512): 31.0, (1024, 1024): 31.1, (2048, 512): 25.0, (2048, 1024): 24.9,
      (4096, 512): 24.8, (4096, 1024): 26.0}, (2048, 1024)),
    ({(1024, 512): 9.0, (1024, 1024): 9.0, (2048, 512): 8.0, (2048, 1024): 8.5,
      (4096, 512): 4.0, (4096, 1024): 4.01}, (4096, 512)),
])
def test_choice(times, chosen):
    batch = PSFBatch.__new__(PSFBatch)
    batch.graph = None

    def configure(chunk, nwg):
        batch.chunk, batch.nwg = chunk, nwg
    batch._configure = configure
    batch.time = lambda reps: times[batch.chunk, batch.nwg]
    assert batch.autotune(chunks=(1024, 2048, 4096), nwgs=(512, 1024)) == times
    assert (batch.chunk, batch.nwg) == chosen
