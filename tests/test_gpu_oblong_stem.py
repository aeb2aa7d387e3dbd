"""Batched STEM on oblong grids, whose column tiles differ from those of a
column as long as the rows."""
import numpy as np
import pytest

from cudamultislice_amd import MultisliceSimulation
from cudamultislice_amd import structures as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [(1024, 512), (1024, 64), (512, 1024), (64, 2048), (1024, 2048), (2048, 1024),
                                   (512, 256)])
def test_the_fused_detector_sums_the_exit_waves_annulus(nx, ny):
    """4 + 2 waves of the same run: the detector's sums against those of its
    exit waves in 64 bits (FP32 transforms and sums: 1e-5)."""
    ps = 0.06
    with MultisliceSimulation() as g:
        g.set_atoms(*S.srtio3(2, 2, 2))
        g.GetParameterisation()
        g.UploadBinnedAtoms()
        g.ApplyMicroscopeParameters(300.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 15.0)
        g.STEMSetCalculationVariables(ps, 0.0, nx, ny, 1, 1, 10.0)
        g.PreCalculateFrequencies()
        k = np.hypot(np.fft.fftfreq(nx, ps)[None, :], np.fft.fftfreq(ny, ps)[:, None]) * g.info()["wavelength"] * 1e3
        at = (k >= 3.0) & (k < 14.0)
        px, py = (np.array([0, n // 2, n - 1, 5, 3, 7], np.int32) for n in (nx, ny))
        run = dict(dz=2.0, nslices=2, adf=(3.0, 14.0))
        waves = g.stem_batched(px, py, exit_waves=True, **run)["exit"][0]
        want = np.array([(np.abs(np.fft.fft2(w.astype(np.complex128))) ** 2 * at).sum() / (nx * ny) for w in waves])
        for more in (dict(), dict(batch=4), dict(batch=4, use_graph=True), dict(pacbed=True)):
            got = g.stem_batched(px, py, **run, **more)["adf"]
            assert np.max(np.abs(got - want) / want) < 1e-5, more
