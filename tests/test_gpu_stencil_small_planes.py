"""Many grids of planes around one and two waves of 16-byte vectors, where the
stencil goes from the kernel without LDS to the ring, against the oracle.
Tolerances as in test_gpu_parity.py: 1e-12 of the largest value in FP64, 2e-5
in FP32."""
import numpy as np
import pytest

torch = pytest.importorskip('torch')

pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():
    pytest.skip('no GPU', allow_module_level=True)

from gpaw_amd.fd_operators import Laplace  # noqa: E402
from gpaw_amd.grid_descriptor import GridDescriptor  # noqa: E402
from oracle import grid as og  # noqa: E402
from oracle import stencil as ost  # noqa: E402


# rows of a plane and their length in 8 bytes: whole vectors below and at 56 and
# 32 (complex64), others below and at 128
@pytest.mark.parametrize('ny,nz', [(11, 10), (14, 8), (7, 8), (8, 8),
                                   (14, 17), (16, 15)])
@pytest.mark.parametrize('dtype', [np.float64, np.complex64, np.float32,
                                   np.complex128])
def test_planes(dtype, ny, nz):
    size = np.dtype(dtype).itemsize
    nz = nz * 8 // size if size < 16 or nz % 2 == 0 else nz
    vectors = ny * -(-nz * size // 16)
    N_c = np.array((5, ny, nz))
    gd = GridDescriptor(N_c, N_c * 0.4, True)
    ogd = og.Grid(N_c, N_c * 0.4, True)
    nb = int(5.5 * 2**20 / (5 * ny * nz * size)) + 1
    rng = np.random.default_rng(5)
    cplx = np.dtype(dtype).kind == 'c'
    a = rng.standard_normal((nb, 5, ny, nz))
    if cplx:
        a = a + 1j * rng.standard_normal(a.shape)
    a = a.astype(dtype)
    ph = ogd.phase_cd((0.2, -0.1, 0.4)) if cplx else None
    ad = torch.from_numpy(a).cuda()
    out = torch.empty_like(ad)
    op = Laplace(gd, -0.5, 2, dtype)
    op.apply(ad, out, ph)
    torch.cuda.synchronize()
    with torch.profiler.profile(
            activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
        op.apply(ad, out, ph)
        torch.cuda.synchronize()
    names = ' '.join(e.key for e in prof.key_averages())
    ring = vectors >= (128 if nz * size % 16 else
                       32 if dtype == np.complex64 else 56)
    assert ('stencil_rows' if ring else 'stencil_direct') in names
    pick = [0, nb // 2, nb - 1]
    c, o = ost.laplace_stencil(ogd.h_cv, -0.5, 2)
    want = ost.fd_apply(c, o, a[pick].astype(complex if cplx else float),
                        ogd.pbc_c, ph)
    tol = 2e-5 if dtype in (np.float32, np.complex64) else 1e-12
    assert abs(out[pick].cpu().numpy() - want).max() < tol * abs(want).max()
