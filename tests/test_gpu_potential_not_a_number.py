"""Atoms whose position is no number add nothing to the potential: no distance
to them is below the cutoff."""
import numpy as np
import pytest

from cudamultislice_amd import MultisliceSimulation
from cudamultislice_amd import structures as S

pytestmark = pytest.mark.gpu


def _handle(atoms, n, ps):
    g = MultisliceSimulation()
    g.set_atoms(*atoms)
    g.GetParameterisation()
    g.ApplyMicroscopeParameters(200.0)
    g.SetCalculationVariables(ps, 0.0, n, n, 1, 1, 15.0, 2.0, 2.0)
    g.PreCalculateFrequencies()
    return g


def _specimen():
    """silicon, and its atom nearest to the centre (inside the extents)"""
    Z, x, y, z = S.silicon(2, 2, 2)
    k = int(np.argmin((x - x.mean()) ** 2 + (y - y.mean()) ** 2 + (z - z.mean()) ** 2))
    return (Z, x, y, z), k


# 64^2 shares each patch between four waves, 520^2 takes a patch per wave
@pytest.mark.parametrize("n", [64, 520])
@pytest.mark.parametrize("mode,axes", [(0, "xyz"), (1, "xy")])
def test_slices_ignore_it(n, mode, axes):
    atoms, k = _specimen()
    with _handle([np.delete(v, k) for v in atoms], n, 15.0 / n) as g:
        g.set_potential_mode(mode)
        g.UploadBinnedAtoms()
        want = [g.potential_slice(it, 2.0, real=True) for it in (1, 3, 5)]
    assert max(w.max() for w in want) > 1.0
    for axis in axes:
        with _handle(atoms, n, 15.0 / n) as g:
            g.set_potential_mode(mode)
            d = {a: np.zeros(atoms[0].size, np.float32) for a in "xyz"}
            d[axis][k] = np.nan
            g.upload_binned_atoms_displaced(d["x"], d["y"], d["z"])
            for w, it in zip(want, (1, 3, 5)):
                # the same atoms in the same order: at most their grouping differs
                assert np.max(np.abs(g.potential_slice(it, 2.0, real=True) - w)) < 1e-5 * w.max(), axis


@pytest.mark.parametrize("method", ["plane", "real space"])
def test_planes_and_real_space_slabs_ignore_it(method):
    atoms, k = _specimen()
    waves = []
    for case in range(2):
        with _handle([np.delete(v, k) for v in atoms] if case == 0 else atoms, 64, 0.235) as g:
            d = [np.zeros(atoms[0].size - (case == 0), np.float32) for _ in range(3)]
            if case == 1:
                d[1][k] = np.nan
            g.upload_binned_atoms_displaced(*d)
            g.InitialiseWavefunctions() if method == "plane" else g.InitialiseWavefunctions(1.0)
            i = g.info()
            depth = 0.5 * (i["MaximumZ"] - i["MinimumZ"])  # of the atom
            first = int(depth / (i["dzFD"] if method == "plane" else 1.0)) - 2
            for it in range(first, first + 5):
                g.MultisliceStep(it) if method == "plane" else g.MultisliceStepRS(it)
            waves.append(g.get_wave())
    assert np.linalg.norm(waves[1] - waves[0]) < 1e-5 * np.linalg.norm(waves[0])
