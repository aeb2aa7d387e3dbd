"""maxposEW / minposEW (U.cu:2261-2262) and maxposIm / minposIm /
imagecontrast (U.cu:2430-2491) as the device finds them, against numpy on the
arrays that the same calls return: one block, an odd count past one block,
more elements than one pass of all blocks, and values that are no number."""
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
    g.ApplyMicroscopeParameters(200.0, -300.0, 0.0, 0.0, 1.2e7, 0.0, 0.0, 20.0)
    g.SetCalculationVariables(0.05, -300.0, nx, ny, 1, 1, 9.0, 2.0, 2.0)
    g.PreCalculateFrequencies()
    g.InitialiseWavefunctions(1.0)
    return g


def _modulus(w):
    w = np.asarray(w, np.complex64)
    return np.sqrt(w.real * w.real + w.imag * w.imag)


@pytest.mark.parametrize("nx,ny", [(16, 16), (37, 29), (600, 530), (1024, 2048)])
def test_exit_wave_and_image_statistics(nx, ny):
    g = _handle(nx, ny)
    rng = np.random.default_rng(nx + ny)
    w = (rng.standard_normal((ny, nx)) + 1j * rng.standard_normal((ny, nx))).astype(np.complex64)
    g.set_wave(w, 0)
    a = _modulus(g.GetExitWave())
    i = g.info()
    assert i["maxposEW"] == a.max() and i["minposEW"] == a.min()  # the same FP32 values
    a = _modulus(g.GetSTEMExitWave())
    i = g.info()
    assert i["maxposEW"] == a.max() and i["minposEW"] == a.min()
    im = g.SimulateImage(1.0)
    i = g.info()
    assert i["maxposIm"] == np.abs(im).max() and i["minposIm"] == np.abs(im).min()
    corner = np.abs(im[:min(512, ny), :min(512, nx)]).astype(np.float64)
    # 64-bit sums rounded to FP32
    assert i["imagecontrast"] == pytest.approx(float(corner.std()), rel=1e-6)
    g.close()


def test_extrema_pass_over_values_that_are_no_number():
    g = _handle(64, 32)
    w = np.full((32, 64), 0.5 + 0j, np.complex64)
    w[0, 0] = np.nan
    w[3, 5] = 2.0
    w[7, 9] = 0.25
    g.set_wave(w, 0)
    g.GetExitWave()
    i = g.info()
    assert i["maxposEW"] == 2.0 and i["minposEW"] == 0.25
    g.set_wave(np.full((32, 64), np.nan, np.complex64), 0)
    g.GetExitWave()
    i = g.info()
    assert np.isnan(i["maxposEW"]) and np.isnan(i["minposEW"])
    g.close()
