"""The upward half of the V-cycle in one pass per level (stencil of the
interpolated function) against the oracle: every type, boundary mixture and
radius, rows that end inside a vector, more tiles and runs than one, and a
grid whose rows that kernel refuses (float32 rows of 4 k + 2 points)."""
import numpy as np
import pytest

torch = pytest.importorskip('torch')
pytestmark = pytest.mark.gpu

from gpaw_amd.fd_operators import Laplace  # noqa: E402
from gpaw_amd.grid_descriptor import GridDescriptor  # noqa: E402
from gpaw_amd.preconditioner import Preconditioner  # noqa: E402

from oracle import grid as og  # noqa: E402
from oracle import precond as opc  # noqa: E402
from oracle import stencil as ost  # noqa: E402


# as the other tests of the cycle: some hundred roundings of terms of order
# one, 2e-13 in FP64 and 2^29 / 50 of that in FP32
@pytest.mark.parametrize('dtype,tol', [(float, 2e-13), (complex, 2e-13),
                                       (np.float32, 2e-6), (np.complex64, 2e-6)])
@pytest.mark.parametrize('N_c,pbc,n,nb', [
    ((16, 16, 16), (1, 1, 1), 3, 1),
    ((40, 20, 72), (1, 1, 1), 3, 37),
    ((20, 24, 28), (1, 1, 1), 2, 300),      # level 1: rows of 14 points
    ((24, 76, 20), (0, 0, 0), 3, 9),
    ((24, 20, 44), (0, 1, 0), 1, 5),
    ((20, 28, 136), (1, 0, 1), 2, 3),
])
def test_cycle(N_c, pbc, n, nb, dtype, tol):
    rng = np.random.default_rng(41)
    N_c = np.array(N_c)
    pbc = tuple(bool(p) for p in pbc)
    gd = GridDescriptor(N_c, N_c * 0.3, pbc)
    ogd = og.Grid(N_c, N_c * 0.3, pbc_c=pbc)
    cplx = np.dtype(dtype).kind == 'c'
    k_c = [q if p else 0 for q, p in zip((0.25, 0.1, -0.3), pbc)]
    R = rng.standard_normal((nb,) + tuple(gd.n_c))
    if cplx:
        R = R + 1j * rng.standard_normal(R.shape)
    R = R.astype(dtype)

    class K:
        phase_cd = ogd.phase_cd(k_c) if cplx else None
    P = Preconditioner(gd, Laplace(gd, -0.5, n, dtype), dtype)
    got = P(torch.from_numpy(R).cuda(), K).cpu().numpy()
    c0, o0 = ost.laplace_stencil(ogd.h_cv, -0.5, n)
    pick = sorted({0, nb // 2, nb - 1})
    want = opc.Preconditioner(ogd, c0, o0)(
        R[pick].astype(complex if cplx else float), K.phase_cd)
    assert abs(got[pick] - want).max() <= tol * abs(want).max()
