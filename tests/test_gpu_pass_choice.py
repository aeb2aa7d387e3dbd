"""Pass variants read, set, tuned and put back: which of them the launches of a
single wave take, told by the bits of its result (plans differ in rounding)."""
import ctypes as C

import numpy as np
import pytest

from cudamultislice_amd import MultisliceSimulation
from cudamultislice_amd import structures as S
from cudamultislice_amd._lib import lib

pytestmark = pytest.mark.gpu


def _steps(n):
    with MultisliceSimulation() as g:
        g.set_atoms(*S.silicon(2, 2, 2))
        g.GetParameterisation()
        g.UploadBinnedAtoms()
        g.ApplyMicroscopeParameters(200.0)
        g.SetCalculationVariables(15.0 / n, 0.0, n, n, 1, 1, 15.0)
        g.PreCalculateFrequencies()
        g.InitialiseWavefunctions(1.0)
        for it in range(1, 7):
            g.MultisliceStepConv(it)
        return g.get_wave()


def _get(kind, n):
    v = C.c_int(-1)
    assert lib().msl_get_pass_variant(kind, n, C.byref(v)) == 0
    return v.value


def _defaults(n):
    """the defaults' numbers, with nothing pinned or tuned afterwards"""
    d = [_get(kind, n) for kind in (0, 1)]
    for kind in (0, 1):
        assert lib().msl_set_pass_variant(kind, n, d[kind]) == 0
    return d


# rows and columns of 64 and 256 have layouts of their own for one wave
@pytest.mark.parametrize("n", [64, 256])
def test_a_variant_read_and_set_again_changes_nothing(n):
    want = _steps(n)
    d = _defaults(n)
    assert np.array_equal(_steps(n), want)
    try:
        # a pinned variant takes every launch: another plan, other rounding
        assert lib().msl_set_pass_variant(0, n, 2) == 0 and _get(0, n) == 2
        pinned = _steps(n)
        assert not np.array_equal(pinned, want)
        assert np.linalg.norm(pinned - want) < 1e-5 * np.linalg.norm(want)
        assert lib().msl_set_pass_variant(0, n, _get(0, n)) == 0 and _get(0, n) == 2
        assert np.array_equal(_steps(n), pinned)
    finally:
        lib().msl_set_pass_variant(0, n, d[0])
    assert _get(0, n) == d[0]
    assert np.array_equal(_steps(n), want)


@pytest.mark.parametrize("n", [64, 256])
def test_the_tuner_leaves_the_layouts_of_one_wave(n):
    d = _defaults(n)
    want = _steps(n)
    try:
        r, c = C.c_int(-1), C.c_int(-1)
        assert lib().msl_autotune_passes(n, 256, 1, C.byref(r), C.byref(c), None) == 0
        assert (_get(0, n), _get(1, n)) == (r.value, c.value)
        assert np.array_equal(_steps(n), want)
    finally:
        for kind in (0, 1):
            lib().msl_set_pass_variant(kind, n, d[kind])
    assert [_get(0, n), _get(1, n)] == d
    assert np.array_equal(_steps(n), want)


def test_refused_variants_stay_refused():
    assert lib().msl_set_pass_variant(0, 64, -1) != 0
    assert lib().msl_set_pass_variant(0, 64, 5) != 0
    assert lib().msl_set_pass_variant(1, 64, 8) != 0
    assert lib().msl_set_pass_variant(0, 100, 0) != 0
