"""Parameter files other than the built-in table."""
import numpy as np
import pytest

from cudamultislice_amd import MultisliceSimulation
from cudamultislice_amd import structures as S
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [0, 1])
def test_a_file_with_unused_lorentzians(fp, tmp_path, mode):
    """a = b = 0 in one term: slices within 2e-5 of the oracle's largest
    value, the bound of the other potential tests."""
    par = fp.copy().reshape(103, 12)
    par[13, 4:6] = 0.0
    path = tmp_path / "params.dat"
    path.write_text("\n".join(" ".join(repr(float(v)) for v in row) for row in par))
    Z, x, y, z = S.silicon(2, 2, 2)
    o = O.OracleSim()
    o.set_atoms(Z, x, y, z)
    o.set_fparams(par)
    o.bin()
    o.apply_microscope(200.0)
    o.set_calc(0.2, 0.0, 64, 64, 1, 1, 15.0, 2.0, 2.0)
    with MultisliceSimulation() as g:
        g.set_atoms(Z, x, y, z)
        g.GetParameterisation(str(path))
        g.UploadBinnedAtoms()
        g.ApplyMicroscopeParameters(200.0)
        g.SetCalculationVariables(0.2, 0.0, 64, 64, 1, 1, 15.0, 2.0, 2.0)
        g.PreCalculateFrequencies()
        g.set_potential_mode(mode)
        e = o.extents()
        for it in (3, 4, 5):
            zf = float(np.float32(e[4] - e[5]) - np.float32(2 * it))
            want = o.potential(3 if mode == 0 else 4, zf, 2.0).real
            assert want.max() > 1.0
            assert np.max(np.abs(g.potential_slice(it, 2.0, real=True) - want)) <= 2e-5 * want.max()
