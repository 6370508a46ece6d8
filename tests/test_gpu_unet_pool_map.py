"""Pooling and 1x1 maps of the U-Net kernels at the edges of their vector
forms: every channel count, one point, the last block partly filled, arrays
that start on any element."""
import ctypes

import numpy as np
import pytest

torch = pytest.importorskip('torch')
pytestmark = pytest.mark.gpu

from gpaw_amd import _lib  # noqa: E402


def bf(n, offset, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(n + offset, generator=g).bfloat16().cuda()
    return x[offset:]


# one rounding to BF16 (2^-9 relative) and FP32 sums
@pytest.mark.parametrize('offset', [0, 1])
@pytest.mark.parametrize('c', [8, 16, 32])
@pytest.mark.parametrize('n,nb', [((2, 2, 2), 1), ((4, 6, 10), 3), ((6, 2, 34), 2)])
def test_pool(n, nb, c, offset):
    x = bf(nb * n[0] * n[1] * n[2] * c, offset, 1)
    m = tuple(k // 2 for k in n)
    out = torch.zeros(nb * m[0] * m[1] * m[2] * c + offset,
                      dtype=torch.bfloat16, device='cuda')[offset:]
    nc = np.array(n, np.int64)
    _lib.check(_lib.lib().gh_unet_pool2(
        c, nb, nc.ctypes.data_as(_lib.PI64), x.data_ptr(), out.data_ptr(),
        ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
    ref = x.double().reshape(nb, m[0], 2, m[1], 2, m[2], 2, c).mean((2, 4, 6))
    err = (out.double().reshape(ref.shape) - ref).abs()
    assert bool((err <= 2.0**-8 * ref.abs() + 1e-6).all())


@pytest.mark.parametrize('offset', [0, 1])
@pytest.mark.parametrize('ci,co', [(32, 16), (16, 8)])
@pytest.mark.parametrize('npts', [1, 255, 256, 1001])
def test_map(npts, ci, co, offset):
    x = bf(npts * ci, offset, 2)
    g = torch.Generator().manual_seed(3)
    W = torch.randn(ci, co, generator=g).cuda()
    b = torch.randn(co, generator=g).cuda()
    out = torch.zeros(npts * co + offset, dtype=torch.bfloat16,
                      device='cuda')[offset:]
    _lib.check(_lib.lib().gh_unet_map1(
        ci, co, npts, x.data_ptr(), W.data_ptr(), b.data_ptr(), out.data_ptr(),
        ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
    ref = x.double().reshape(npts, ci) @ W.double() + b.double()
    err = (out.double().reshape(ref.shape) - ref).abs()
    assert bool((err <= 2.0**-8 * ref.abs() + 1e-4).all())
