"""The potential kernel's pixel tiles, on launches large enough to take them
(4096 patches of 8 x 8 pixels), and the tuner on launches that are not."""
import numpy as np
import pytest

from cudamultislice_amd import MultisliceSimulation
from cudamultislice_amd import structures as S
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _handle(fp, nspec, nx, ny, ps):
    Z, x, y, z = S.jittered_atoms(60, (12.0, 11.0, 9.0), seed=21)
    Z = np.array([(14, 38, 8, 22, 79, 6)[i % nspec] for i in range(Z.size)], np.int32)
    g = MultisliceSimulation()
    o = O.OracleSim()
    g.set_atoms(Z, x, y, z)
    o.set_atoms(Z, x, y, z)
    g.GetParameterisation()
    o.set_fparams(fp)
    g.UploadBinnedAtoms()
    o.bin()
    g.ApplyMicroscopeParameters(300.0)
    o.apply_microscope(300.0)
    g.SetCalculationVariables(ps, 0.0, nx, ny, 1, 1, 20.0, 1.0, 1.5)
    o.set_calc(ps, 0.0, nx, ny, 1, 1, 20.0, 1.0, 1.5)
    g.PreCalculateFrequencies()
    return g, o


@pytest.mark.parametrize("nspec", [3, 6])  # tables in LDS, in memory
@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("nx,ny", [(520, 505), (505, 520)])
def test_every_tile_matches_the_oracle(fp, nx, ny, mode, nspec):
    """The same atoms in the same order for every pixel: the same bits, and
    within 2e-5 of the largest value (as the other potential tests)."""
    g, o = _handle(fp, nspec, nx, ny, 0.03)
    g.set_potential_mode(mode)
    e = o.extents()
    top = 0.0
    for it in (2, 4):
        want = o.potential(3 if mode == 0 else 4, float(np.float32(e[4] - e[5]) - np.float32(2 * it)), 2.0).real
        top = max(top, want.max())
        outs = []
        for tile in range(4):
            g.set_potential_tile(tile)
            outs.append(g.potential_slice(it, 2.0, real=True))
            assert np.array_equal(outs[tile], outs[0]), tile
        assert np.max(np.abs(outs[0] - want)) <= 2e-5 * want.max()
    assert top > 1.0  # some slice holds atoms
    g.close()


def test_every_tile_in_the_plane_of_a_finite_difference_step(fp):
    waves = []
    for tile in range(4):
        g, o = _handle(fp, 3, 512, 512, 0.03)
        g.set_potential_tile(tile)
        g.InitialiseWavefunctions()
        o.init_plane_fd()
        e = o.extents()
        it = int(0.5 * (e[4] - e[5]) / o.scalars()["dzFD"])
        g.MultisliceStep(it)
        waves.append(g.get_wave())
        assert np.array_equal(waves[tile], waves[0]), tile
        if tile == 0:
            o.step_fd(it)
            assert np.linalg.norm(waves[0] - o.wave()) < 1e-5 * np.linalg.norm(o.wave())
        g.close()


def test_the_tuner_keeps_the_tile_where_tiles_have_no_part(fp):
    g, _ = _handle(fp, 3, 96, 96, 0.15)
    for tile in (0, 3, 1, 2):
        g.set_potential_tile(tile)
        best, ms = g.autotune_potential(2.0, nslices=4)
        assert best == tile and min(ms) > 0
    # 144 patches a slice: 29 slices are 4176
    best, ms = g.autotune_potential(0.5, nslices=29)
    assert best == int(np.argmin(ms)) and min(ms) > 0
    g.close()
