"""Rounding over many slices: the errors of the transforms' factors must not
add up from slice to slice beyond what rounding the waves costs."""
import numpy as np
import pytest
import torch

from cudamultislice_amd.diff import DiffEngine

pytestmark = pytest.mark.gpu

PS, KV, DZ, SLICES, PROBES = 0.1, 300.0, 2.0, 50, 2


def _exact(V, psi, n, sigma, lam, kmax):
    k = torch.from_numpy((np.where(np.arange(n) > n // 2, np.arange(n) - n, np.arange(n)).astype(np.float32)
                          / np.float32(np.float32(PS) * np.float32(n)))).cuda().double()
    k2 = k[None, :] ** 2 + k[:, None] ** 2
    P = (k2.sqrt() < kmax) * torch.exp(-1j * 3.14159265 * DZ * lam * k2)
    w = psi.to(torch.complex128)
    for v in V:
        w = torch.fft.ifft2(P * torch.fft.fft2(torch.exp(1j * sigma * v.double()) * w))
    return w.abs().square()


@pytest.mark.parametrize("n", [64, 128, 256, 512, 1024, 2048])
def test_fifty_slices_of_the_differentiable_forward(n):
    """A transform of n points in FP32 is right to about 3.5e-8 sqrt(log2 n)
    (half a unit in the last place per doubling, random signs).  50 slices are
    200 of them per wave, an intensity has twice a wave's relative error, and
    half as much again is allowed for the factors: 1.5 * 2 * 3.5e-8 *
    sqrt(200 log2 n)."""
    g = torch.Generator("cuda").manual_seed(n)
    x = torch.fft.fftfreq(n, PS, dtype=torch.float64, device="cuda")
    blur = torch.exp(-2 * (np.pi * 0.2) ** 2 * (x[None, :] ** 2 + x[:, None] ** 2)).float()
    V = torch.empty(SLICES, n, n, device="cuda")
    for i in range(SLICES):
        atoms = (torch.rand(n, n, device="cuda", generator=g) < 0.12 * PS ** 2).float()
        V[i] = torch.fft.ifft2(torch.fft.fft2(atoms * 2500.0) * blur).real.clamp_(min=0.0)
    eng = DiffEngine(n, n, PS, KV, DZ, SLICES, PROBES, 0)
    i = eng.info()
    ap = (x[None, :] ** 2 + x[:, None] ** 2).sqrt() < 0.025 / i["wavelength"]
    psi = torch.stack([torch.fft.ifft2(ap * torch.exp(-2j * np.pi * x[None, :] * n * PS * f)) for f in (0.3, 0.6)])
    psi = (psi / psi.abs().square().sum((1, 2), keepdim=True).sqrt()).to(torch.complex64)
    got = eng.forward(V, psi, keep=False).double()
    want = _exact(V, psi, n, i["sigma"], i["wavelength"], i["kmax"])
    assert (got - want).norm() / want.norm() < 1.5 * 2 * 3.5e-8 * np.sqrt(200 * np.log2(n))
    eng.close()
