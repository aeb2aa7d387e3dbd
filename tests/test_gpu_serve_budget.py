"""Batches of several classes in one run stay within the caller's budget."""
import numpy as np
import pytest
import torch

from cudamultislice_amd import structures as S
from cudamultislice_amd.serve import CONVENTIONAL, FD, Job, serve

pytestmark = pytest.mark.gpu

BUDGET = 2 << 30


def _jobs():
    """finite differences (five arrays of up to a fifth of the budget), then a
    conventional class that takes all of it in one array"""
    rng = np.random.default_rng(2)
    jobs = []
    for method, probes, ns in ((FD, 45, 3), (CONVENTIONAL, 240, 2)):
        atoms = S.jittered_atoms(500, (98.0, 98.0, 6.0), seed=method)
        jobs.append(Job(1024, *atoms, ns, method, *(rng.integers(0, 1024, probes).astype(np.int32) for _ in range(2))))
    jobs.append(Job(512, *S.jittered_atoms(200, (47.0, 47.0, 6.0), seed=9), 2, CONVENTIONAL,
                    *(rng.integers(0, 512, 30).astype(np.int32) for _ in range(2))))
    return jobs


@pytest.mark.parametrize("grouped", [False, True])
def test_a_mixed_run_fits_one_and_a_quarter_budgets(grouped):
    want = _jobs()
    serve(want, adf=(5.0, 25.0), group_sizes=grouped)
    torch.cuda.empty_cache()
    held = torch.empty(torch.cuda.mem_get_info()[0] - BUDGET * 5 // 4, dtype=torch.uint8, device="cuda")
    got = _jobs()
    stats = serve(got, adf=(5.0, 25.0), group_sizes=grouped, budget_bytes=BUDGET)
    del held
    torch.cuda.empty_cache()
    assert 0.8 * BUDGET < stats["largest_batch_bytes"] <= BUDGET
    for a, b in zip(got, want):
        assert b.result["adf"].min() > 0
        assert np.max(np.abs(a.result["adf"] - b.result["adf"]) / b.result["adf"]) < 1e-5
