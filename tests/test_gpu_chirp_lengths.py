"""Grid sides that are not powers of two (chirp transforms, k_generic.hip):
lengths at the edges of the transform sizes, primes, a power of two beside
another length, sides past 2048, and batches of images."""
import numpy as np
import pytest

from cudamultislice_amd import structures as S

pytestmark = pytest.mark.gpu


def _handle(nx, ny):
    from cudamultislice_amd import MultisliceSimulation
    g = MultisliceSimulation()
    g.set_atoms(*S.silicon(1, 1, 1))
    g.GetParameterisation()
    g.UploadBinnedAtoms()
    g.ApplyMicroscopeParameters(200.0, -300.0, 0.0, 0.0, 1.2e7, 0.0, 0.0, 1000.0)
    g.SetCalculationVariables(0.05, -300.0, nx, ny, 1, 1, 9.0, 2.0, 2.0)
    g.PreCalculateFrequencies()
    g.InitialiseWavefunctions(1.0)
    return g


# 2 n - 1 just below and above a power of two (33: 65 > 64), primes, powers
# of two beside other lengths, lengths of one workgroup per line
SIDES = [(33, 32), (65, 64), (128, 100), (61, 257), (513, 1024), (2, 30), (1025, 3), (3, 1027), (2050, 4), (5, 2049),
         (4100, 6), (6, 4099), (8191, 2), (3, 8190)]


@pytest.mark.parametrize("nx,ny", SIDES)
def test_transforms_of_any_length_match_numpy(nx, ny):
    """The centred spectrum of a random wave against numpy's 64-bit FFT.
    Tolerance: a transform of length M in FP32 is off by about
    eps sqrt(log2 M) (6e-8 x 3.8 at 16384); a chirp transform does two, on two
    axes, with three products each: 4 x 2.3e-7 + 6 x 6e-8 < 1.3e-6."""
    g = _handle(nx, ny)
    rng = np.random.default_rng(nx * 10007 + ny)
    w = (rng.standard_normal((ny, nx)) + 1j * rng.standard_normal((ny, nx))).astype(np.complex64)
    g.set_wave(w, 0)
    got = g.GetSTEMExitWave()
    want = np.fft.fft2(w.astype(np.complex128))
    at = [np.where(np.arange(n) >= n // 2, np.arange(n) - n // 2, np.arange(n) + n // 2) for n in (ny, nx)]
    want = want[at[0]][:, at[1]]
    assert np.linalg.norm(got - want) / np.linalg.norm(want) < 1.3e-6
    # and back: the image of an open aperture at zero defocus and Cs is |w|^2
    g.ApplyMicroscopeParameters(200.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 1.0e6)
    img = g.ctf_sweep([0.0, 0.0, 0.0])
    ref = np.abs(w.astype(np.complex128)) ** 2
    for k in range(3):  # twice the transforms, squared
        assert np.linalg.norm(img[k] - ref) / np.linalg.norm(ref) < 4 * 1.3e-6
    g.close()
