"""The fused finite-difference step (U.cu:2040-2083) on grids of powers of
two: its Laplacian is left by one step for the next, so a step after anything
else that writes the wave has to make its own; with and without a band that
lets it skip columns, on square and oblong grids, against the oracle."""
import numpy as np
import pytest

from cudamultislice_amd import structures as S
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _pair(fp, nx, ny, physical=False):
    from cudamultislice_amd import MultisliceSimulation
    Z, x, y, z = S.silicon(2, 2, 2)
    g = MultisliceSimulation(physical=physical)
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
    o.apply_microscope(200.0)
    o.set_calc(ps, 0.0, nx, ny, 1, 1, 15.0)
    g.InitialiseWavefunctions()
    o.init_plane_fd()
    e = o.extents()
    return g, o, int(0.5 * (e[4] - e[5]) / o.scalars()["dzFD"])


def _rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("nx,ny", [(16, 16), (32, 64), (128, 128), (256, 64), (512, 128), (64, 1024)])
def test_consecutive_steps_match_the_oracle(fp, nx, ny):
    """Psi, PsiMinus after ten steps within the 1e-4 that the engine's
    finite-difference tests use."""
    g, o, first = _pair(fp, nx, ny)
    for it in range(first, first + 10):
        g.MultisliceStep(it)
        o.step_fd(it)
    for which in (0, 1):
        assert _rel(g.get_wave(which), o.wave(which)) < 1e-4
    g.close()


def test_a_wave_written_between_steps_gets_its_own_laplacian(fp):
    """After set_wave the step is the one a handle takes that never stepped
    before: the same bits, for a wave with frequencies past the band."""
    g, _, first = _pair(fp, 128, 128)
    h, _, _ = _pair(fp, 128, 128)
    rng = np.random.default_rng(2)
    w = [(1.0 + 0.1 * (rng.standard_normal((128, 128)) + 1j * rng.standard_normal((128, 128)))).astype(np.complex64)
         for _ in range(2)]
    for it in range(first, first + 3):
        g.MultisliceStep(it)
    for s in (g, h):
        s.set_wave(w[0], 0)
        s.set_wave(w[1], 1)
        s.MultisliceStep(first + 3)
    assert np.array_equal(g.get_wave(0), h.get_wave(0)) and np.array_equal(g.get_wave(1), h.get_wave(1))
    # reading results between steps changes nothing
    for s in (g, h):
        s.MultisliceStep(first + 4)
        if s is g:
            s.GetExitWave()
            s.GetSTEMExitWave()
            s.AllocTDS()
            s.AddTDSWaves()
            s.adf(1.0, 50.0)
            s.ctf_sweep([10.0])
        s.MultisliceStep(first + 5)
    assert np.array_equal(g.get_wave(0), h.get_wave(0))
    # nor does a conventional step leave a stale one behind
    for s in (g, h):
        s.set_wave(w[0], 0)
    h.set_wave(w[1], 1)
    g.set_wave(w[1], 1)
    g.MultisliceStepConv(2)
    h.MultisliceStepConv(2)
    g.MultisliceStep(first)
    h.MultisliceStep(first)
    assert np.array_equal(g.get_wave(0), h.get_wave(0))
    g.close()
    h.close()


def test_steps_under_the_wider_physical_band(fp):
    """compat=physical keeps |k| <= 2/3 of the Nyquist frequency: no columns
    are skipped; three steps agree with the 64-bit filters of numpy on the
    oracle's potential within 1e-5."""
    g, o, first = _pair(fp, 64, 64, physical=True)
    i = g.info()
    assert i["band_tiles"] == 0
    k = np.fft.fftfreq(64, 15.0 / 64)
    k2 = k[None, :] ** 2 + k[:, None] ** 2
    band, lap = k2 <= i["kmax"] ** 2, -4 * 3.14159 ** 2 * k2
    dz, lam, sig = i["dzFD"], i["wavelength"], i["sigma2"]
    al = 2 * 3.14159 * dz / lam
    pm, p0 = (g.get_wave(w).astype(np.complex128) for w in (1, 0))
    H = np.float32(i["MaximumZ"]) - np.float32(i["MinimumZ"])
    for it in range(first, first + 3):
        g.MultisliceStep(it)
        V = o.potential(2, float(H - np.float32(dz) * np.float32(it)), 1.0).real
        V = np.fft.ifft2(band * np.fft.fft2(V)).real
        u = 2 * p0 - dz ** 2 * np.fft.ifft2(lap * np.fft.fft2(p0)) - dz ** 2 * 4 * 3.14159 * sig * V / lam * p0
        pp = np.fft.ifft2(band * np.fft.fft2((u - (1 - 1j * al) * pm) / (1 + 1j * al)))
        pm, p0 = p0, pp
    assert _rel(g.get_wave(0), p0) < 1e-5
    g.close()
