"""Undisplaced atoms far from the origin: the branch of the binning that waits
for the range check."""
import numpy as np
import pytest

from cudamultislice_amd import MultisliceSimulation

pytestmark = pytest.mark.gpu


def test_keys_are_those_of_the_same_atoms_at_the_origin():
    """3e5 A away FP32 resolves 0.031 A: positions on multiples of that."""
    x = np.arange(40, dtype=np.float32) * np.float32(0.5)
    keys = []
    for shift in (0.0, 3.0e5):
        s = np.float32(shift)
        with MultisliceSimulation() as g:
            g.set_atoms(np.full(40, 14, np.int32), x + s, x[::-1].copy() + s, x * np.float32(0.5) + s)
            g.UploadBinnedAtoms()
            keys.append(g.bin_keys())
    assert (keys[0] >= 0).all() and np.array_equal(keys[0], keys[1])
