"""The chirp transforms run in 64 bits: their results carry the rounding of the
FP32 stores alone."""
import numpy as np
import pytest

from cudamultislice_amd import MultisliceSimulation
from cudamultislice_amd import structures as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [(33, 32), (61, 257), (513, 1024), (1002, 668), (5, 2049), (4100, 6), (2004, 1336),
                                   (3, 8190)])
def test_only_the_stores_round(nx, ny):
    """Rows, then columns, store FP32 values: at most 2^-24 each, 2^-24 sqrt(2)
    = 8.4e-8 (transforms in FP32 are off by 1.5e-7 and more).  An image has
    two more and the CTF's product between, twice that in its square, and the
    square's own: 2 * 2^-24 sqrt(5) + 2^-23 = 3.9e-7."""
    with MultisliceSimulation() as g:
        g.set_atoms(*S.silicon(1, 1, 1))
        g.GetParameterisation()
        g.UploadBinnedAtoms()
        g.ApplyMicroscopeParameters(200.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 1.0e6)
        g.SetCalculationVariables(0.05, 0.0, nx, ny, 1, 1, 9.0, 2.0, 2.0)
        g.PreCalculateFrequencies()
        g.InitialiseWavefunctions(1.0)
        rng = np.random.default_rng(nx * 10007 + ny)
        w = (rng.standard_normal((ny, nx)) + 1j * rng.standard_normal((ny, nx))).astype(np.complex64)
        g.set_wave(w, 0)
        got = g.GetSTEMExitWave()
        img = g.ctf_sweep([0.0, 0.0])
    want = np.fft.fft2(w.astype(np.complex128))
    at = [np.where(np.arange(n) >= n // 2, np.arange(n) - n // 2, np.arange(n) + n // 2) for n in (ny, nx)]
    want = want[at[0]][:, at[1]]
    assert np.linalg.norm(got - want) < 2.0 ** -24 * np.sqrt(2.0) * np.linalg.norm(want)
    ref = np.abs(w.astype(np.complex128)) ** 2
    for k in range(2):
        assert np.linalg.norm(img[k] - ref) < (2 * 2.0 ** -24 * np.sqrt(5.0) + 2.0 ** -23) * np.linalg.norm(ref)
