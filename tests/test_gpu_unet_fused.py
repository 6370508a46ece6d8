"""The marching convolution with a fused 1x1 map or correction: the same bits
as the two layers run one after the other, on grids of one and of several
y tiles and x runs, rows that are no multiple of 16 points, odd band counts,
and rows too long for the LDS (refused: the caller takes the two layers)."""
import numpy as np
import pytest

torch = pytest.importorskip('torch')

pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():
    pytest.skip('no GPU', allow_module_level=True)

from gpaw_amd import _lib  # noqa: E402
from gpaw_amd._arrays import dtype_code, stream_ptr  # noqa: E402
from gpaw_amd.learned.unet import HIPUNet, UNet3  # noqa: E402


def bits(shape, g):
    return torch.randn(shape, device='cuda', generator=g).to(
        torch.bfloat16).view(torch.int16)


@pytest.mark.parametrize('dtype', [torch.float32, torch.float64])
@pytest.mark.parametrize('n,nb', [((2, 2, 2), 1), ((4, 6, 10), 2),
                                  ((12, 40, 22), 3), ((34, 26, 98), 2),
                                  ((8, 8, 300), 1)])
def test_fused_layers_equal_separate(n, nb, dtype):
    L = _lib.lib()
    torch.manual_seed(2)
    net = HIPUNet(UNet3())
    g = torch.Generator(device='cuda')
    g.manual_seed(sum(n) + nb)
    npts = nb * int(np.prod(n))
    nc = np.ascontiguousarray(n, np.int64)
    ncp = nc.ctypes.data_as(_lib.PI64)
    scale = torch.rand(nb, device='cuda', generator=g) + 0.5

    inp, skip = bits((npts // 8, 16), g), bits((npts, 16), g)
    h = torch.empty((npts, 16), dtype=torch.int16, device='cuda')
    net._conv('c1u', 16, 16, 2, nb, n, h, inp=inp, skip=skip)
    ref = torch.empty((npts, 8), dtype=torch.int16, device='cuda')
    net._map('m1', 16, 8, npts, h, ref)
    out = torch.zeros_like(ref)
    W, b = net.conv['c1u']
    Wm, bm = net.map1['m1']
    rc = L.gh_unet_conv3_map1(nb, ncp, inp.data_ptr(), skip.data_ptr(),
                              W.data_ptr(), b.data_ptr(), Wm.data_ptr(),
                              bm.data_ptr(), out.data_ptr(), stream_ptr())
    if n[2] > 150:     # three rows of 16 channels no longer fit the LDS
        assert rc == _lib.GH_ERR_UNSUPPORTED
    else:
        _lib.check(rc)
        assert torch.equal(out, ref)

    inp, skip = bits((npts // 8, 8), g), bits((npts, 8), g)
    h = torch.empty((npts, 8), dtype=torch.int16, device='cuda')
    net._conv('c0u', 8, 8, 2, nb, n, h, inp=inp, skip=skip)
    ref = torch.empty((nb,) + n, dtype=dtype, device='cuda')
    Wh, _ = net.map1['head']
    _lib.check(L.gh_unet_head(8, dtype_code(dtype), nb, npts // nb,
                              h.data_ptr(), Wh.data_ptr(), net.head_bias,
                              scale.data_ptr(), ref.data_ptr(), stream_ptr()))
    out = torch.zeros_like(ref)
    W, b = net.conv['c0u']
    _lib.check(L.gh_unet_conv3_head(
        dtype_code(dtype), nb, ncp, inp.data_ptr(), skip.data_ptr(),
        W.data_ptr(), b.data_ptr(), Wh.data_ptr(), net.head_bias,
        scale.data_ptr(), out.data_ptr(), stream_ptr()))
    assert torch.equal(out, ref)


def test_long_rows_take_the_separate_layers():
    """800 points: the fused layers refuse, the network runs layer by layer;
    1000 points: the first layer's slab does not fit either, as before."""
    model = UNet3().cuda()
    net = HIPUNet(model)
    g = torch.Generator(device='cuda')
    g.manual_seed(4)
    scale = torch.ones(1, device='cuda')
    for n in ((4, 4, 800), (4, 4, 1000)):
        R = torch.randn((1,) + n, device='cuda', generator=g)
        v = torch.randn(n, device='cuda', generator=g)
        out = torch.empty_like(R)
        nc = np.ascontiguousarray(n, np.int64)
        rc = net._lib.gh_unet_conv3_head(
            dtype_code(R.dtype), 1, nc.ctypes.data_as(_lib.PI64), 1, 1, 1, 1,
            1, 0.0, 1, 1, None)
        assert rc == _lib.GH_ERR_UNSUPPORTED
        if n[2] == 1000:
            with pytest.raises(_lib.GPAWAMDError):
                net(R, v, scale, out)
            continue
        net(R, v, scale, out)
        x = torch.stack([R, 0.5 * v.expand(1, *n)], 1)
        with torch.no_grad():
            ref = model(x, bf16=True)[:, 0]
        assert float((out - ref).abs().mean()) < \
            3e-3 * float(ref.abs().mean())
