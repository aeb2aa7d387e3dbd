"""Transforms of large values."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("inverse", [False, True])
@pytest.mark.parametrize("nx,ny", [(16, 16), (32, 64), (256, 128), (512, 1024), (2048, 16)])
def test_values_of_1e26(nx, ny, inverse):
    """A power of two times the data is that power times the result, bit for
    bit: 2^86 = 7.7e25, whose partial sums stay below 2^97."""
    import torch
    from cudamultislice_amd._lib import lib
    g = torch.Generator("cuda").manual_seed(nx)
    a = torch.view_as_complex(torch.randn(2, ny, nx, 2, device="cuda", generator=g))
    b = a * 2.0 ** 86
    torch.cuda.synchronize()
    s = torch.cuda.current_stream()
    for d in (a, b):
        assert lib().msl_fft2_device(nx, ny, 2, C.c_void_p(d.data_ptr()), int(inverse), C.c_void_p(s.cuda_stream)) == 0
    torch.cuda.synchronize()
    a, b = a.cpu().numpy(), b.cpu().numpy()
    assert np.isfinite(b.view(np.float32)).all()
    assert np.array_equal(b, a * np.float32(2.0 ** 86))
