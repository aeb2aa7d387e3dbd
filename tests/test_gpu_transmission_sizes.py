"""The transmissions of a differentiable forward, made in launches of fewer
than 2^32 threads."""
import pytest
import torch

from cudamultislice_amd.diff import DiffEngine

pytestmark = pytest.mark.gpu


def test_a_potential_of_2_32_values_off_the_alignment_of_wide_loads():
    """2048^2 x 1024 slices (16 GiB) one float past an allocation's start: the
    intensities of the same potential where it is aligned."""
    n, ns = 2048, 1024
    if torch.cuda.mem_get_info()[0] < 90 << 30:
        pytest.skip("needs 90 GiB of free device memory")
    V = torch.zeros(ns * n * n + 4, device="cuda")
    for i in (0, 511, 512, ns - 1):  # potential at the ends and around the middle
        g = torch.Generator("cuda").manual_seed(i)
        V[1 + i * n * n:1 + (i + 1) * n * n] = 20.0 * torch.rand(n * n, device="cuda", generator=g)
    psi = torch.ones(1, n, n, dtype=torch.complex64, device="cuda")
    eng = DiffEngine(n, n, 0.1, 300.0, 2.0, ns, 1, 64)
    got = eng.forward(V[1:-3].view(ns, n, n), psi, keep=False)
    want = eng.forward(V[1:-3].clone().view(ns, n, n), psi, keep=False)
    assert (want - 1.0).abs().max() > 1e-3
    assert torch.equal(got, want)
    eng.close()
