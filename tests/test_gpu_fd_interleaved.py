"""Finite-difference steps with other calls between them: the Laplacian that a
step leaves for the next must be that of the wave."""
import numpy as np
import pytest

from cudamultislice_amd import MultisliceSimulation
from cudamultislice_amd import structures as S

pytestmark = pytest.mark.gpu

N = 128


def _handle():
    g = MultisliceSimulation()
    g.set_atoms(*S.silicon(2, 2, 3))
    g.GetParameterisation()
    g.UploadBinnedAtoms()
    g.ApplyMicroscopeParameters(200.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 20.0)
    g.SetCalculationVariables(0.12, 0.0, N, N, 1, 1, 18.0)
    g.PreCalculateFrequencies()
    g.InitialiseWavefunctions()
    return g


def _stem(g):
    p = np.arange(5, dtype=np.int32) * 9
    g.stem_batched(p, p, 2.0, nslices=3, adf=(5.0, 40.0), pacbed=True)


def _rebin(g):
    d = np.zeros(S.silicon(2, 2, 3)[0].size, np.float32)
    g.upload_binned_atoms_displaced(d, d, d)


CALLS = {
    "batched STEM": _stem,
    "exit wave": lambda g: g.GetExitWave(),
    "spectrum": lambda g: g.GetSTEMExitWave(),
    "image": lambda g: g.SimulateImage(1.0),
    "sweep": lambda g: g.ctf_sweep([0.0, 100.0]),
    "detector": lambda g: g.adf(5.0, 40.0),
    "binning": _rebin,
    "tables": lambda g: g.PreCalculateFrequencies(),
    "potential": lambda g: g.potential_slice(3, 1.0),
}


@pytest.mark.parametrize("call", CALLS)
def test_reads_between_steps_change_nothing(call):
    """The Laplacian made again, from the wave, or carried over: the same steps
    within rounding (twenty steps of FP32: 1e-5, the bound of these steps
    against the oracle)."""
    waves = []
    for between in (False, True):
        with _handle() as g:
            i = g.info()
            first = int(0.4 * (i["MaximumZ"] - i["MinimumZ"]) / i["dzFD"])
            for it in range(first, first + 20):
                g.MultisliceStep(it)
                if between and it % 3 == 0:
                    CALLS[call](g)
            waves.append(g.get_wave())
    assert np.max(np.abs(waves[0] - 1.0)) > 1e-3
    assert np.linalg.norm(waves[1] - waves[0]) < 1e-5 * np.linalg.norm(waves[0])


def test_a_wave_set_between_steps_is_the_one_that_goes_on():
    rng = np.random.default_rng(4)
    w, m = ((1.0 + 0.05 * (rng.standard_normal((N, N)) + 1j * rng.standard_normal((N, N)))).astype(np.complex64)
            for _ in range(2))
    waves = []
    for before in (0, 4):
        with _handle() as g:
            i = g.info()
            first = int(0.4 * (i["MaximumZ"] - i["MinimumZ"]) / i["dzFD"])
            for it in range(first - before, first):
                g.MultisliceStep(it)
            g.set_wave(w, 0)
            g.set_wave(m, 1)
            for it in range(first, first + 5):
                g.MultisliceStep(it)
            waves.append(g.get_wave())
    assert np.array_equal(waves[0], waves[1])
