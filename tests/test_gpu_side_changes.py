"""One handle taken from sides to sides, each with tables of its own."""
import numpy as np
import pytest

from cudamultislice_amd import MultisliceSimulation
from cudamultislice_amd import structures as S

pytestmark = pytest.mark.gpu

SIDES = [(100, 90), (64, 64), (100, 90), (334, 167), (501, 128), (100, 90), (90, 100), (256, 32), (90, 100)]


def _run(g, nx, ny):
    g.ApplyMicroscopeParameters(200.0)
    g.SetCalculationVariables(15.0 / max(nx, ny), 0.0, nx, ny, 1, 1, 15.0, 2.0, 2.0)
    g.PreCalculateFrequencies()
    g.InitialiseWavefunctions(1.0)
    for it in range(1, 5):
        g.MultisliceStepConv(it)
    return g.GetExitWave()


def test_a_handle_gives_the_bits_of_a_fresh_one():
    def handle():
        g = MultisliceSimulation()
        g.set_atoms(*S.silicon(2, 2, 2))
        g.GetParameterisation()
        g.UploadBinnedAtoms()
        return g
    fresh = {}
    for s in set(SIDES):
        with handle() as g:
            fresh[s] = _run(g, *s)
    with handle() as g:
        for s in SIDES:
            assert np.array_equal(_run(g, *s), fresh[s]), s
