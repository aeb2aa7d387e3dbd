"""The passes of a few waves at the lengths that take the small layouts (rows
of 64 to 256, columns of 64 to 512) and at their edges: square grids, and
oblong ones that mix them with the other layouts, against the oracle."""
import numpy as np
import pytest

from cudamultislice_amd import MultisliceSimulation
from cudamultislice_amd import structures as S
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [(64, 64), (16, 512), (512, 16), (128, 256), (256, 128), (64, 1024), (32, 64),
                                   (1024, 512), (256, 2048)])
def test_steps_of_one_wave_match_the_oracle(fp, nx, ny):
    """Four conventional steps of a noisy wave: 16 transforms of at most
    2^20 points in FP32 (2^-24 sqrt(20) each, random signs: 1.1e-6 in all)
    and potentials right to some 1e-6: within 2e-5."""
    Z, x, y, z = S.silicon(2, 2, 2)
    g = MultisliceSimulation()
    g.set_atoms(Z, x, y, z)
    g.GetParameterisation()
    g.UploadBinnedAtoms()
    o = O.OracleSim()
    o.set_atoms(Z, x, y, z)
    o.set_fparams(fp)
    o.bin()
    ps = 15.0 / nx
    g.ApplyMicroscopeParameters(200.0)
    g.SetCalculationVariables(ps, 0.0, nx, ny, 1, 1, 15.0)
    g.PreCalculateFrequencies()
    g.InitialiseWavefunctions(1.0)
    o.apply_microscope(200.0)
    o.set_calc(ps, 0.0, nx, ny, 1, 1, 15.0)
    o.init_plane(1.0)
    rng = np.random.default_rng(nx + ny)
    w = (1.0 + 0.1 * (rng.standard_normal((ny, nx)) + 1j * rng.standard_normal((ny, nx)))).astype(np.complex64)
    g.set_wave(w)
    o.set_wave(w)
    for it in range(1, 5):
        g.MultisliceStepConv(it)
        o.step_conv(it)
    got, want = g.get_wave(), o.wave()
    assert np.linalg.norm(got - want) < 2e-5 * np.linalg.norm(want)
    g.close()


@pytest.mark.parametrize("n", [64, 256, 512, 1024])
def test_a_probe_has_the_same_bits_in_every_batch(n):
    """Launches of one to nine waves of a batched run cross the rules' sizes;
    layouts they may choose among share a plan: the same bits."""
    Z, x, y, z = S.srtio3(2, 2, 2)
    g = MultisliceSimulation()
    g.set_atoms(Z, x, y, z)
    g.GetParameterisation()
    g.UploadBinnedAtoms()
    g.ApplyMicroscopeParameters(200.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 15.0)
    g.STEMSetCalculationVariables(12.0 / n, 0.0, n, n, 1, 1, 1)
    g.PreCalculateFrequencies()
    g.STEMInitialiseWavefunctions(n // 2, n // 2)
    px = np.arange(9, dtype=np.int32) * (n // 16) + 3
    runs = [g.stem_batched(px, px[::-1].copy(), dz=1.0, nslices=4, adf=(5.0, 40.0), batch=b, exit_waves=True)
            for b in (9, 1, 2, 5)]
    for r in runs[1:]:
        assert np.array_equal(r["exit"], runs[0]["exit"]) and np.array_equal(r["adf"], runs[0]["adf"])
    g.close()
