"""Runs cut into batches on both sides of every size at which the passes change
their kernel or layout: a probe's bits do not depend on the batch."""
import numpy as np
import pytest

from cudamultislice_amd import MultisliceSimulation
from cudamultislice_amd import structures as S

pytestmark = pytest.mark.gpu


# rows: the loop over waves begins at 16 waves of 512 and 17 of 1024, and at
# 2048 takes over from the plain kernel at 4; columns: half-width tiles up to
# 64 waves of 64, 32 of 256 and 1 of 1024, the small layout up to 4 of 512,
# the loop over waves at 2048 (which forms its propagator factors once for all
# waves: a launch of one wave there takes the plain kernel and rounds otherwise)
@pytest.mark.parametrize("n,batches", [(64, (130, 65, 64, 63, 1)), (128, (40, 17, 16, 1)), (256, (66, 33, 32, 31, 1)),
                                       (512, (40, 17, 16, 15, 8, 5, 4, 1)), (1024, (20, 17, 16, 15, 8, 2, 1)),
                                       (2048, (6, 4, 3, 2))])
def test_a_probe_has_the_same_bits_on_both_sides(n, batches):
    probes = batches[0]
    rng = np.random.default_rng(n)
    px, py = (rng.integers(0, n, probes).astype(np.int32) for _ in range(2))
    with MultisliceSimulation() as g:
        g.set_atoms(*S.srtio3(2, 2, 2))
        g.GetParameterisation()
        g.UploadBinnedAtoms()
        g.ApplyMicroscopeParameters(200.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 15.0)
        g.STEMSetCalculationVariables(12.0 / n, 0.0, n, n, 1, 1, 1)
        g.PreCalculateFrequencies()
        want = g.stem_batched(px, py, dz=1.0, nslices=3, adf=(5.0, 40.0), batch=probes, exit_waves=True)
        for b in batches[1:]:
            got = g.stem_batched(px, py, dz=1.0, nslices=3, adf=(5.0, 40.0), batch=b, exit_waves=True)
            assert np.array_equal(got["exit"], want["exit"]), b
            assert np.array_equal(got["adf"], want["adf"]), b
