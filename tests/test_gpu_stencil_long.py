"""Stencils of radius 4 to 6 in both kernels: rows as short as the radius, one
point off a vector, several tiles and x-runs, every type and boundary, with
potential, source and shift, against the oracle.  Tolerances as in
test_gpu_parity.py: 1e-12 of the largest value in FP64, 2e-5 in FP32."""
import numpy as np
import pytest

torch = pytest.importorskip('torch')

pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():
    pytest.skip('no GPU', allow_module_level=True)

from gpaw_amd.fd_operators import FDOperator, Laplace  # noqa: E402
from gpaw_amd.grid_descriptor import GridDescriptor  # noqa: E402
from oracle import grid as og  # noqa: E402
from oracle import stencil as ost  # noqa: E402


@pytest.mark.parametrize('kernel', ['', 'rows', 'reg'])
@pytest.mark.parametrize('dtype', [np.float64, np.float32, np.complex128,
                                   np.complex64])
@pytest.mark.parametrize('n', [4, 5, 6])
@pytest.mark.parametrize('N_c,pbc,nb,k_c', [
    ((6, 6, 6), True, 2, (0.2, -0.1, 0.4)),
    ((7, 9, 8), True, 3, (0.2, 0, 0)),
    ((8, 8, 7), (True, False, True), 2, (0.2, 0, 0.3)),
    ((30, 44, 40), True, 9, (0.2, -0.1, 0.4)),
    ((26, 31, 46), False, 20, None)])
def test_radius(monkeypatch, N_c, pbc, nb, k_c, n, dtype, kernel):
    monkeypatch.setenv('GPAW_AMD_STENCIL', kernel)
    rng = np.random.default_rng(3)
    N_c = np.array(N_c)
    gd = GridDescriptor(N_c, N_c * 0.4, pbc)
    ogd = og.Grid(N_c, N_c * 0.4, pbc)
    cplx = np.dtype(dtype).kind == 'c'
    single = dtype in (np.float32, np.complex64)
    shape = (nb,) + tuple(gd.n_c)

    def rand():
        a = rng.standard_normal(shape)
        return (a + 1j * rng.standard_normal(shape) if cplx else a).astype(
            dtype)
    a, src = rand(), rand()
    vt = rng.standard_normal(shape[1:]).astype(np.float32 if single else float)
    eps = rng.uniform(-1, 1, nb)
    ph = ogd.phase_cd(k_c) if cplx and k_c is not None else None
    pick = sorted({0, nb - 1})
    wide = a[pick].astype(complex if cplx else float)
    tol = 2e-5 if single else 1e-12
    ad, vd, sd = (torch.from_numpy(x).cuda() for x in (a, vt, src))
    out = torch.empty_like(ad)

    def check(want):
        got = out[pick].cpu().numpy()
        assert abs(got - want).max() < tol * abs(want).max()
    c, o = ost.laplace_stencil(ogd.h_cv, -0.5, n)
    ref = ost.fd_apply(c, o, wide, ogd.pbc_c, ph)
    op = Laplace(gd, -0.5, n, dtype)
    op.apply(ad, out, ph, vt_g=vd, src_xg=sd, beta=-0.3)
    check(ref + vt * wide - 0.3 * src[pick])
    op.apply_shifted(ad, out, eps, ph, vt_g=vd)
    check(ref + (vt - eps[pick][:, None, None, None]) * wide)
    # different coefficients at +j and -j
    c = rng.uniform(-1, 1, len(c))
    op = FDOperator(c, o, gd, dtype)
    op.apply(ad, out, ph)
    check(ost.fd_apply(c, o, wide, ogd.pbc_c, ph))
