"""The passes' transforms at every length, both directions, against numpy's in
64 bits: noise, and impulses whose spectra run through every factor of the
tables (also those whose cosine is zero)."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("inverse", [False, True])
@pytest.mark.parametrize("nx,ny", [(16, 2048), (32, 1024), (64, 512), (128, 256), (256, 128), (512, 64), (1024, 32),
                                   (2048, 16)])
def test_transforms_of_every_length(nx, ny, inverse):
    """log2(nx ny) <= 15 levels of butterflies whose sums and brackets round
    by at most 2^-24 each, random signs: 2^-24 sqrt(2 * 15) = 3.3e-7 rms; of
    an impulse, every value the product of at most 8 factors, each within
    2^-24 sqrt(2), and of its rounding: below 16 * 2^-24 = 9.6e-7."""
    import torch
    from cudamultislice_amd._lib import lib
    rng = np.random.default_rng(nx)
    a = (rng.standard_normal((4, ny, nx)) + 1j * rng.standard_normal((4, ny, nx))).astype(np.complex64)
    a[1:] = 0
    for b, (y, x) in enumerate(((0, 1), (1, 0), (ny // 2 - 1, nx // 4 + 1)), 1):
        a[b, y, x] = 1
    d = torch.from_numpy(a.copy()).cuda()
    torch.cuda.synchronize()
    s = torch.cuda.current_stream()
    assert lib().msl_fft2_device(nx, ny, 4, C.c_void_p(d.data_ptr()), int(inverse), C.c_void_p(s.cuda_stream)) == 0
    torch.cuda.synchronize()
    got = d.cpu().numpy()
    want = np.fft.ifft2(a.astype(np.complex128)) * (nx * ny) if inverse else np.fft.fft2(a.astype(np.complex128))
    assert np.linalg.norm(got[0] - want[0]) < 3.3e-7 * np.linalg.norm(want[0])
    assert np.abs(got[1:] - want[1:]).max() < 9.6e-7
