"""The two forms of the short-filter transformers: calls just above the sizes
from which the staged kernels serve them, the same bits as a few bands alone
(which take the other kernels); and planes around the block sizes of the
kernels without LDS, against the oracle (FP64 1e-14 of the largest value,
FP32 1e-6)."""
import numpy as np
import pytest

torch = pytest.importorskip('torch')
pytestmark = pytest.mark.gpu

from gpaw_amd.grid_descriptor import GridDescriptor  # noqa: E402
from gpaw_amd.transformers import Transformer  # noqa: E402

from oracle import grid as og  # noqa: E402
from oracle import transformers as otr  # noqa: E402


@pytest.mark.parametrize('dtype,N_c,pbc,op,nb', [
    (np.float64, (48, 44, 40), True, 'r', 400),
    (np.float64, (24, 20, 18), True, 'r', 4000),
    (np.float32, (48, 44, 40), True, 'r', 190),
    (np.float32, (16, 16, 100), True, 'r', 700),
    (np.complex64, (48, 44, 40), True, 'r', 600),
    (np.complex128, (48, 44, 36), True, 'i', 210),
    (np.complex128, (32, 30, 26), False, 'i', 800),
    (np.float64, (48, 44, 40), False, 'i', 1300),
    (np.float32, (48, 44, 40), False, 'i', 2600),
    (np.float32, (48, 44, 38), True, 'i', 2600)])
def test_staged_calls(dtype, N_c, pbc, op, nb):
    N_c = np.array(N_c)
    gd = GridDescriptor(N_c, N_c * 0.3, (pbc,) * 3)
    ogd = og.Grid(N_c, N_c * 0.3, pbc_c=(pbc,) * 3)
    cplx = np.dtype(dtype).kind == 'c'
    ph = ogd.phase_cd((0.25, 0, 0)) if cplx and pbc else None
    a, b = (gd, gd.coarsen()) if op == 'r' else (gd.coarsen(), gd)
    g = torch.Generator(device='cuda').manual_seed(3)
    td = torch.from_numpy(np.zeros(1, dtype)).dtype
    x = torch.randn((nb,) + tuple(int(k) for k in a.n_c), generator=g,
                    dtype=td, device='cuda')
    T = Transformer(a, b, 1, dtype)
    out = T.apply(x, phases=ph)
    for i in (0, 1, nb // 2, nb - 1):
        alone = T.apply(x[i:i + 1].contiguous(), phases=ph)
        err = (out[i:i + 1] - alone).abs().max()
        assert err <= (1e-15 if cplx else 0) * alone.abs().max()


# coarse planes of 49 to 288 points: one wave to four per block, one point
# less and more than a multiple of 64
@pytest.mark.parametrize('dtype', [np.float64, np.float32])
@pytest.mark.parametrize('n1,n2', [(7, 7), (8, 8), (5, 13), (9, 14), (16, 8),
                                   (3, 43), (12, 16), (16, 16), (4, 65),
                                   (16, 18)])
@pytest.mark.parametrize('pbc', [True, False])
@pytest.mark.parametrize('nb', [1, 500])
def test_block_sizes(n1, n2, pbc, nb, dtype):
    rng = np.random.default_rng(n1 * n2)
    N_c = 2 * np.array([6, n1 + (not pbc), n2 + (not pbc)])
    gd = GridDescriptor(N_c, N_c * 0.3, (pbc,) * 3)
    ogd = og.Grid(N_c, N_c * 0.3, pbc_c=(pbc,) * 3)
    tol = 1e-14 if dtype == np.float64 else 1e-6
    for a, b, oa, ob in ((gd, gd.coarsen(), ogd, ogd.coarsen()),
                         (gd.coarsen(), gd, ogd.coarsen(), ogd)):
        x = rng.standard_normal((nb,) + tuple(a.n_c)).astype(dtype)
        out = Transformer(a, b, 1, dtype).apply(torch.from_numpy(x).cuda())
        pick = [0, nb - 1]
        want = otr.Transformer(oa, ob, 1).apply(x[pick].astype(float), None)
        got = out[pick].cpu().numpy()
        assert abs(got - want).max() <= tol * abs(want).max()
