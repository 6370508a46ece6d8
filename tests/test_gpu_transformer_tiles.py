"""Restriction and interpolation over the tiles that the band count selects:
the tile rows and the x-run of a block follow from sizes and bands, the
values do not.  Every band of a call must be bit-equal to the same band
alone, and agree with the oracle."""
import numpy as np
import pytest

torch = pytest.importorskip('torch')
pytestmark = pytest.mark.gpu

from gpaw_amd.grid_descriptor import GridDescriptor  # noqa: E402
from gpaw_amd.transformers import Transformer  # noqa: E402

from oracle import grid as og  # noqa: E402
from oracle import transformers as otr  # noqa: E402


# 16 roundings of sums of at most (2 K + 1)^3 terms of order one stay below
# 1e-14 in FP64; FP32 is larger by 2^29
@pytest.mark.parametrize('dtype,tol', [(np.float64, 1e-14), (np.complex128, 1e-14),
                                       (np.float32, 5e-6), (np.complex64, 5e-6)])
@pytest.mark.parametrize('nn', [1, 3])
@pytest.mark.parametrize('N_c,pbc', [((20, 26, 34), True), ((8, 60, 10), True),
                                     ((36, 16, 130), False)])
@pytest.mark.parametrize('nb', [1, 7, 300])
def test_tiles(N_c, pbc, nn, dtype, tol, nb):
    rng = np.random.default_rng(31)
    N_c = np.array(N_c)
    gd = GridDescriptor(N_c, N_c * 0.3, (pbc,) * 3)
    ogd = og.Grid(N_c, N_c * 0.3, pbc_c=(pbc,) * 3)
    cplx = np.dtype(dtype).kind == 'c'
    ph = ogd.phase_cd((0.25, 0.1, 0)) if cplx and pbc else None
    for a, b, oa, ob in ((gd, gd.coarsen(), ogd, ogd.coarsen()),
                         (gd.coarsen(), gd, ogd.coarsen(), ogd)):
        x = rng.standard_normal((nb,) + tuple(a.n_c))
        if cplx:
            x = x + 1j * rng.standard_normal(x.shape)
        x = x.astype(dtype)
        T = Transformer(a, b, nn, dtype)
        xd = torch.from_numpy(x).cuda()
        out = T.apply(xd, phases=ph)
        for i in {0, nb // 2, nb - 1}:
            alone = T.apply(xd[i:i + 1].contiguous(), phases=ph)
            assert torch.equal(out[i:i + 1], alone)
        # zero boundaries of a complex grid: the oracle takes the real parts
        ref = otr.Transformer(oa, ob, nn)
        i = nb - 1
        wide = x[i:i + 1].astype(np.complex128 if ph is not None else np.float64) \
            if not (cplx and ph is None) else None
        if wide is not None:
            want = ref.apply(wide, ph)
        else:
            want = ref.apply(x[i:i + 1].real.astype(np.float64), None) + \
                1j * ref.apply(x[i:i + 1].imag.astype(np.float64), None)
        got = out[i:i + 1].cpu().numpy()
        assert abs(got - want).max() <= tol * abs(want).max()


# calls large enough for the staged kernels of the short filter: restriction
# of whole vectors, complex128 and odd FP64 rows interpolated; the same bits
# as a few bands alone, which take the other kernels (real data; complex128
# with phases: last bits)
@pytest.mark.parametrize('dtype,N_c,pbc,op,nb', [
    (np.float64, (48, 44, 40), True, 'r', 290), (np.float32, (48, 44, 40), True, 'r', 290),
    (np.complex64, (48, 44, 40), True, 'r', 290), (np.complex128, (48, 44, 36), True, 'i', 240),
    (np.float64, (48, 44, 40), False, 'i', 230)])
def test_large_calls(dtype, N_c, pbc, op, nb):
    N_c = np.array(N_c)
    gd = GridDescriptor(N_c, N_c * 0.3, (pbc,) * 3)
    ogd = og.Grid(N_c, N_c * 0.3, pbc_c=(pbc,) * 3)
    cplx = np.dtype(dtype).kind == 'c'
    ph = ogd.phase_cd((0.25, 0, 0)) if cplx and pbc else None
    a, b = (gd, gd.coarsen()) if op == 'r' else (gd.coarsen(), gd)
    g = torch.Generator(device='cuda').manual_seed(3)
    td = torch.from_numpy(np.zeros(1, dtype)).dtype
    x = torch.randn((nb,) + tuple(int(k) for k in a.n_c), generator=g, dtype=td, device='cuda')
    T = Transformer(a, b, 1, dtype)
    out = T.apply(x, phases=ph)
    for i in (0, nb // 2, nb - 1):
        alone = T.apply(x[i:i + 1].contiguous(), phases=ph)
        err = (out[i:i + 1] - alone).abs().max()
        assert err <= (1e-15 if dtype == np.complex128 else 0) * alone.abs().max()
