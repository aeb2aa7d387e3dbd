"""Gradients with the backward cut into chunks of probes."""
import pytest
import torch

from cudamultislice_amd.diff import DiffEngine

pytestmark = pytest.mark.gpu


# one probe of 64 columns and two of them are on two sides of a layout rule,
# as are 16 and 48 of 64 and 4 and 12 of 256
@pytest.mark.parametrize("n,probes,chunk", [(64, 2, 1), (64, 48, 16), (256, 12, 4), (512, 6, 2)])
def test_a_probe_has_the_same_adjoint_in_every_chunk(n, probes, chunk):
    """dL/dI is zero but for the probes of one chunk: the gradient is that of
    their adjoint waves alone, whose bits do not depend on the chunk."""
    g = torch.Generator("cuda").manual_seed(n)
    V = 20.0 * torch.rand(4, n, n, device="cuda", generator=g)
    psi = torch.view_as_complex(torch.randn(probes, n, n, 2, device="cuda", generator=g))
    eng = DiffEngine(n, n, 0.1, 300.0, 2.0, 4, probes, 0)
    eng.forward(V, psi)
    for k in range(0, probes, chunk):
        d = torch.zeros(probes, n, n, device="cuda")
        d[k] = 1.0
        eng.set_chunk(0)
        want = eng.backward(d).clone()
        eng.set_chunk(chunk)
        assert want.abs().max() > 0 and torch.equal(eng.backward(d), want), k
    eng.close()
