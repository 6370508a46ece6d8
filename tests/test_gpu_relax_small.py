"""Jacobi sweeps of small grids in one launch, around the size limit, and the
pieces of the multigrid's upward half: interpolation subtracted from a grid,
sweeps that start in the work array."""
import numpy as np
import pytest

torch = pytest.importorskip('torch')
pytestmark = pytest.mark.gpu

from gpaw_amd.fd_operators import Laplace  # noqa: E402
from gpaw_amd.grid_descriptor import GridDescriptor  # noqa: E402
from gpaw_amd.transformers import Transformer  # noqa: E402

from oracle import grid as og  # noqa: E402
from oracle import poisson as opo  # noqa: E402
from oracle import stencil as ost  # noqa: E402
from oracle import transformers as otr  # noqa: E402


# at most 8 sweeps of 8 terms of order one: 2e-14, FP32 2^29 of that
@pytest.mark.parametrize('dtype,tol', [(np.float64, 2e-14), (np.float32, 1e-5)])
@pytest.mark.parametrize('N_c,pbc,n', [
    ((2, 2, 2), False, 1), ((2, 4, 6), True, 1), ((6, 6, 7), False, 1),
    ((16, 16, 16), True, 1), ((16, 17, 16), True, 1), ((5, 4, 205), True, 1),
    ((3, 2, 1100), (True, True, False), 1), ((9, 65, 9), (False, True, False), 1),
    ((8, 9, 10), True, 2)])
@pytest.mark.parametrize('count', [1, 2, 5, 8])
def test_relax(N_c, pbc, n, count, dtype, tol):
    rng = np.random.default_rng(5)
    N_c = np.array(N_c)
    gd = GridDescriptor(N_c, N_c * 0.4, pbc)
    ogd = og.Grid(N_c, N_c * 0.4, pbc)
    f = rng.standard_normal(tuple(gd.n_c)).astype(dtype)
    s = rng.standard_normal(tuple(gd.n_c)).astype(dtype)
    L = Laplace(gd, -0.3, n, dtype)
    fd, sd = torch.from_numpy(f).cuda(), torch.from_numpy(s).cuda()
    c, o = ost.laplace_stencil(ogd.h_cv, -0.3, n)
    want = opo.relax_jacobi(c, o, f.astype(float), s.astype(float), count, 0.6,
                            ogd.pbc_c)
    start = fd.clone()
    L.relax(2, fd, sd, count, 0.6)
    scale = abs(want).max()
    assert abs(fd.cpu().numpy() - want).max() <= tol * scale
    out = torch.full_like(fd, float('nan'))
    L._relax_from(out, sd, start, count, 0.6)
    assert torch.equal(out, fd)


@pytest.mark.parametrize('inplace', [True, False])
@pytest.mark.parametrize('N_c,pbc', [((8, 10, 14), True), ((16, 12, 20), False)])
def test_subtract(N_c, pbc, inplace):
    rng = np.random.default_rng(6)
    N_c = np.array(N_c)
    gd = GridDescriptor(N_c, N_c * 0.4, pbc)
    ogd = og.Grid(N_c, N_c * 0.4, pbc)
    u = rng.standard_normal((1,) + tuple(gd.coarsen().n_c))
    base = rng.standard_normal((1,) + tuple(gd.n_c))
    T = Transformer(gd.coarsen(), gd, 1)
    bd = torch.from_numpy(base).cuda()
    out = bd if inplace else torch.empty_like(bd)
    T._subtract(torch.from_numpy(u).cuda()[0], bd[0], out[0])
    want = base - otr.Transformer(ogd.coarsen(), ogd, 1).apply(u, None)
    assert abs(out.cpu().numpy() - want).max() <= 1e-15 * abs(want).max()
