"""A run whose later job is refused: the earlier jobs' uploads have ended when
it returns, and the next run is unaffected."""
import numpy as np
import pytest

from cudamultislice_amd import MslError
from cudamultislice_amd import structures as S
from cudamultislice_amd.serve import Job, serve

pytestmark = pytest.mark.gpu


def _jobs():
    Z, x, y, z = S.jittered_atoms(60000, (98.0, 98.0, 120.0), seed=5)
    rng = np.random.default_rng(1)
    return [Job(1024, Z, x, y, z, 3),
            Job(128, *S.silicon(2, 2, 2), 3, 0, *(rng.integers(0, 128, 5).astype(np.int32) for _ in range(2)))]


def test_a_refused_job_behind_a_large_one():
    want = _jobs()
    serve(want)
    for _ in range(3):
        jobs = _jobs()
        bad = jobs[1].Z.copy()
        bad[3] = 0
        with pytest.raises(MslError):
            serve([jobs[0], Job(128, bad, jobs[1].x, jobs[1].y, jobs[1].z, 3)])
        got = _jobs()
        serve(got)
        assert np.array_equal(got[0].result["exit"], want[0].result["exit"])
        assert np.array_equal(got[1].result["adf"], want[1].result["adf"])
