"""The potential kernels' two launch forms (four waves sharing 64 pixels below
4096 patches of 8 x 8, one wave per patch from there on) and two table
sources (LDS up to four species, global memory beyond) against the oracle,
on grids that end inside a pixel tile."""
import numpy as np
import pytest

from cudamultislice_amd import structures as S
from oracle import oracle as O

pytestmark = pytest.mark.gpu

SPECIES = [14, 6, 79, 38, 8, 103]


def _pair(fp, nspec, box, n, seed):
    from cudamultislice_amd import MultisliceSimulation
    Z, x, y, z = S.jittered_atoms(n, box, seed=seed)
    Z = np.array([SPECIES[i % nspec] for i in range(Z.size)], np.int32)
    g = MultisliceSimulation()
    g.set_atoms(Z, x, y, z)
    g.GetParameterisation()
    g.UploadBinnedAtoms()
    o = O.OracleSim()
    o.set_atoms(Z, x, y, z)
    o.set_fparams(fp)
    o.bin()
    return g, o


def _setup(g, o, nx, ny, ps):
    g.ApplyMicroscopeParameters(300.0)
    g.SetCalculationVariables(ps, 0.0, nx, ny, 1, 1, 20.0, 1.0, 1.5)
    g.PreCalculateFrequencies()
    o.apply_microscope(300.0)
    o.set_calc(ps, 0.0, nx, ny, 1, 1, 20.0, 1.0, 1.5)


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("nx,ny,ps,nspec", [(37, 21, 0.3, 1), (96, 80, 0.13, 4), (90, 61, 0.13, 5),
                                            (520, 505, 0.03, 2), (505, 520, 0.03, 6)])
def test_potential_forms_match_the_oracle(fp, mode, nx, ny, ps, nspec):
    """Within 2e-5 of the largest value, the bound of the other potential
    tests (FP32 positions: 1e-6 A at 20 A, against a slope of up to 5 / A)."""
    g, o = _pair(fp, nspec, (12.0, 11.0, 9.0), 60, 5 + nspec)
    _setup(g, o, nx, ny, ps)
    g.set_potential_mode(mode)
    e = o.extents()
    H = np.float32(e[4] - e[5])
    top = 0.0
    for it, dz in ((1, 2.0), (4, 2.0), (9, 1.0)):
        zf = float(H - np.float32(np.float32(dz) * np.float32(it)))
        want = o.potential(3 if mode == 0 else 4, zf, dz).real
        got = g.potential_slice(it, dz, real=True)
        top = max(top, want.max())
        assert np.max(np.abs(got - want)) <= 2e-5 * np.max(np.abs(want))
    assert top > 1.0  # some slice holds atoms
    g.close()


def test_more_atoms_than_one_chunk_in_a_bin_window(fp):
    """1500 atoms in a 6 x 6 x 3 A box: a window of several 512-atom chunks
    and of more than 256 bin rows."""
    from cudamultislice_amd import MultisliceSimulation
    rng = np.random.default_rng(3)
    n = 1500
    Z = np.full(n, 6, np.int32)
    x, y = (rng.uniform(0.0, 6.0, n).astype(np.float32) for _ in range(2))
    z = rng.uniform(0.0, 3.0, n).astype(np.float32)
    g = MultisliceSimulation()
    g.set_atoms(Z, x, y, z)
    g.GetParameterisation()
    g.UploadBinnedAtoms()
    o = O.OracleSim()
    o.set_atoms(Z, x, y, z)
    o.set_fparams(fp)
    o.bin()
    _setup(g, o, 48, 40, 0.2)
    e = o.extents()
    want = o.potential(3, float(np.float32(e[4] - e[5]) - np.float32(4.0)), 2.0).real
    got = g.potential_slice(2, 2.0, real=True)
    # a sum of up to 1500 x 20 terms in FP32: 2e-5 as above
    assert np.max(np.abs(got - want)) <= 2e-5 * np.max(np.abs(want))
    g.close()


@pytest.mark.parametrize("n,ps", [(64, 0.3), (512, 0.035)])
def test_plane_potential_of_the_finite_difference_step(fp, n, ps):
    """The point potential of MultisliceStep in both launch forms, through
    three steps in the middle of the specimen (exit wave within 1e-5)."""
    g, o = _pair(fp, 3, (12.0, 11.0, 6.0), 40, 11)
    _setup(g, o, n, n, ps)
    g.InitialiseWavefunctions()
    o.init_plane_fd()
    e = o.extents()
    first = int(0.5 * (e[4] - e[5]) / o.scalars()["dzFD"])
    for it in range(first, first + 3):
        g.MultisliceStep(it)
        o.step_fd(it)
    w, want = g.get_wave(0), o.wave(0)
    assert np.max(np.abs(want - 1.0)) > 1e-5
    assert np.linalg.norm(w - want) / np.linalg.norm(want) < 1e-5
    g.close()
