"""Finite-difference steps on grids much wider than high, and of a power of two
beside another side."""
import numpy as np
import pytest

from cudamultislice_amd import MultisliceSimulation
from cudamultislice_amd import structures as S
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [(2048, 16), (2048, 512), (2048, 1024), (1024, 16), (16, 1024),
                                   (256, 60), (60, 256)])
def test_steps_match_the_oracle(fp, nx, ny):
    Z, x, y, z = S.silicon(2, 2, 2)
    with MultisliceSimulation() as g:
        g.set_atoms(Z, x, y, z)
        g.GetParameterisation()
        g.UploadBinnedAtoms()
        o = O.OracleSim()
        o.set_atoms(Z, x, y, z)
        o.set_fparams(fp)
        o.bin()
        ps = 0.1
        g.ApplyMicroscopeParameters(200.0)
        g.SetCalculationVariables(ps, 0.0, nx, ny, 1, 1, 15.0)
        g.PreCalculateFrequencies()
        o.apply_microscope(200.0)
        o.set_calc(ps, 0.0, nx, ny, 1, 1, 15.0)
        g.InitialiseWavefunctions()
        o.init_plane_fd()
        e = o.extents()
        first = int(0.5 * (e[4] - e[5]) / o.scalars()["dzFD"])
        for it in range(first, first + 3):
            g.MultisliceStep(it)
            o.step_fd(it)
        w, want = g.get_wave(), o.wave()
    assert np.max(np.abs(want - 1.0)) > 1e-5
    # three steps of FP32 transforms: 1e-5, as the other steps against the oracle
    assert np.linalg.norm(w - want) < 1e-5 * np.linalg.norm(want)
