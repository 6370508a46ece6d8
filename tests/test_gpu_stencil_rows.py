"""Stencils on rows of any length and alignment (zero and periodic
boundaries, Bloch phases, every radius) against the oracle: rows shorter
than a vector of points, rows one point off a vector or a 16-byte multiple,
arrays that start one element off a 16-byte boundary, one point per axis,
grids split into several tiles and x-runs.  Tolerances as in
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


def off_by_one(a):
    """The array on the GPU, starting one element off its allocation."""
    t = torch.empty(a.size + 1, dtype=torch.from_numpy(a[:0]).dtype,
                    device='cuda')[1:].reshape(a.shape)
    t.copy_(torch.from_numpy(a))
    return t


CASES = [
    # N_c, pbc, nbands, n, dtype, k_c
    ((2, 2, 2), False, 1, 1, np.float64, None),
    ((2, 3, 4), False, 2, 1, np.float32, None),
    ((4, 3, 3), True, 2, 3, np.float32, None),
    ((5, 4, 3), True, 2, 3, np.float64, None),
    ((5, 4, 7), True, 3, 3, np.complex64, (0.2, -0.1, 0.4)),
    ((8, 9, 10), False, 3, 3, np.float64, None),
    ((12, 12, 131), True, 2, 3, np.float64, None),
    ((12, 10, 260), (False, True, False), 1, 3, np.float32, None),
    ((9, 20, 23), (True, False, True), 5, 3, np.complex64, (0.2, 0, -0.3)),
    ((11, 40, 21), True, 3, 3, np.complex128, (0.25, -0.125, 0.375)),
    ((40, 40, 40), False, 7, 3, np.float64, None),
    ((10, 13, 22), True, 2, 5, np.float32, None),
    ((13, 14, 30), False, 2, 6, np.float64, None),
    ((64, 64, 80), False, 60, 3, np.float64, None),
    ((64, 64, 76), (True, True, False), 60, 2, np.complex64, (0.3, 0.1, 0)),
    ((64, 60, 53), True, 60, 3, np.float32, None),
    ((40, 64, 45), True, 40, 3, np.complex128, (0.25, -0.125, 0.375)),
    ((40, 64, 45), True, 40, 1, np.complex128, (0.25, 0, 0)),
]


@pytest.mark.parametrize('kernel', ['', 'rows', 'reg'])
@pytest.mark.parametrize('N_c,pbc,nb,n,dtype,k_c', CASES)
def test_rows(monkeypatch, N_c, pbc, nb, n, dtype, k_c, kernel):
    monkeypatch.setenv('GPAW_AMD_STENCIL', kernel)
    rng = np.random.default_rng(3)
    N_c = np.array(N_c)
    gd = GridDescriptor(N_c, N_c * 0.4, pbc)
    ogd = og.Grid(N_c, N_c * 0.4, pbc)
    cplx = np.dtype(dtype).kind == 'c'
    shape = (nb,) + tuple(gd.n_c)

    def rand():
        a = rng.standard_normal(shape)
        return (a + 1j * rng.standard_normal(shape) if cplx else a).astype(
            dtype)
    single = dtype in (np.float32, np.complex64)
    a, src = rand(), rand()
    vt = rng.standard_normal(shape[1:]).astype(
        np.float32 if single else np.float64)
    eps = rng.uniform(-1, 1, nb)
    ph = None if k_c is None else ogd.phase_cd(k_c)
    c, o = ost.laplace_stencil(ogd.h_cv, -0.5, n)
    wide = np.complex128 if cplx else np.float64
    # the oracle on the first, a middle and the last band
    pick = sorted({0, nb // 2, nb - 1})
    ref = ost.fd_apply(c, o, a[pick].astype(wide), ogd.pbc_c, ph)
    tol = 2e-5 if single else 1e-12
    op = Laplace(gd, -0.5, n, dtype)

    def check(out, want):
        got = out[pick].cpu().numpy()
        assert abs(got - want).max() < tol * abs(want).max()
    for place in (lambda x: torch.from_numpy(x).cuda(), off_by_one):
        ad, vd, sd = place(a), place(vt), place(src)
        out = place(np.full_like(a, np.nan))
        op.apply(ad, out, ph)
        check(out, ref)
        op.apply(ad, out, ph, vt_g=vd, src_xg=sd, beta=-0.3)
        check(out, ref + vt * a[pick] - 0.3 * src[pick])
        # the source may be the result's own array
        op.apply(ad, sd, ph, src_xg=sd, beta=2.0)
        check(sd, ref + 2.0 * src[pick])
        op.apply_shifted(ad, out, eps, ph, vt_g=vd)
        check(out, ref + (vt - eps[pick][:, None, None, None]) * a[pick])
    for tile in ((1, 0), (3, 2), (0, 5)):
        op.set_tile(*tile)
        op.apply(ad, out, ph)
        check(out, ref)


@pytest.mark.parametrize('kernel', ['', 'rows', 'reg'])
@pytest.mark.parametrize('value', [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize('N_c', [(9, 10, 12), (9, 10, 11)])
def test_zero_boundary_keeps_infinities_apart(monkeypatch, N_c, value,
                                              kernel):
    """A point beyond a zero boundary contributes zero, not 0 * (a value of
    the grid): an infinity at a face reaches only the points whose stencil
    holds it."""
    monkeypatch.setenv('GPAW_AMD_STENCIL', kernel)
    N_c = np.array(N_c)
    gd = GridDescriptor(N_c, N_c * 0.4, False)
    a = np.ones((1,) + tuple(gd.n_c))
    a[0, 0, 0, 0] = value
    op = Laplace(gd, -0.5, 3)
    d = torch.from_numpy(a).cuda()
    out = torch.empty_like(d)
    op.apply(d, out)
    bad = ~np.isfinite(out.cpu().numpy()[0])
    want = np.zeros(tuple(gd.n_c), bool)
    want[:4, 0, 0] = want[0, :4, 0] = want[0, 0, :4] = True
    assert (bad == want).all()


@pytest.mark.parametrize('kernel', ['', 'rows', 'reg'])
@pytest.mark.parametrize('N_c,pbc,nb,dtype,k_c', [
    ((10, 12, 14), True, 2, np.float64, None),
    ((64, 60, 53), False, 30, np.float64, None),
    ((64, 60, 52), True, 30, np.float32, None),
    ((40, 48, 45), True, 40, np.complex128, (0.25, -0.125, 0.375)),
    ((40, 48, 46), True, 40, np.complex64, (0.25, 0.1, 0.3))])
def test_unsymmetric_coefficients(monkeypatch, N_c, pbc, nb, dtype, k_c,
                                  kernel):
    """Different coefficients at +j and -j (a one-sided derivative)."""
    monkeypatch.setenv('GPAW_AMD_STENCIL', kernel)
    rng = np.random.default_rng(8)
    N_c = np.array(N_c)
    gd = GridDescriptor(N_c, N_c * 0.4, pbc)
    ogd = og.Grid(N_c, N_c * 0.4, pbc)
    offs = [(0, 0, 0)] + [tuple(s * j if c == d else 0 for d in range(3))
                          for c in range(3) for j in (1, 2) for s in (1, -1)]
    coef = rng.uniform(-1, 1, len(offs))
    cplx = np.dtype(dtype).kind == 'c'
    shape = (nb,) + tuple(gd.n_c)
    a = rng.standard_normal(shape)
    a = (a + 1j * rng.standard_normal(shape) if cplx else a).astype(dtype)
    ph = None if k_c is None else ogd.phase_cd(k_c)
    pick = sorted({0, nb // 2, nb - 1})
    ref = ost.fd_apply(coef, np.array(offs), a[pick].astype(
        np.complex128 if cplx else np.float64), ogd.pbc_c, ph)
    op = FDOperator(coef, offs, gd, dtype)
    d = torch.from_numpy(a).cuda()
    out = torch.empty_like(d)
    op.apply(d, out, ph)
    tol = 2e-5 if dtype in (np.float32, np.complex64) else 1e-12
    assert abs(out[pick].cpu().numpy() - ref).max() < tol * abs(ref).max()


@pytest.mark.parametrize('kernel', ['', 'rows', 'reg'])
@pytest.mark.parametrize('dtype', [np.complex128, np.complex64])
@pytest.mark.parametrize('N_c', [(9, 10, 12), (9, 10, 11), (40, 44, 46)])
@pytest.mark.parametrize('axis', [0, 1, 2])
def test_bloch_phases_keep_infinities_apart(monkeypatch, N_c, dtype, kernel,
                                            axis):
    """An infinite real part at a face gives the imaginary part nothing but
    through a Bloch phase: only the points that read it as a periodic image
    have both parts infinite."""
    monkeypatch.setenv('GPAW_AMD_STENCIL', kernel)
    N_c = np.array(N_c)
    gd = GridDescriptor(N_c, N_c * 0.4, True)
    at = [n // 2 for n in N_c]
    at[axis] = 0
    nb = 1 if N_c[0] < 40 else 10
    a = np.ones((nb,) + tuple(gd.n_c), dtype)
    a[(0,) + tuple(at)] = np.inf + 0j
    op = Laplace(gd, -0.5, 3, dtype)
    d = torch.from_numpy(a).cuda()
    out = torch.empty_like(d)
    op.apply(d, out, gd.phase_cd((0.2, 0.15, -0.1)))
    out = out.cpu().numpy()
    re, im = np.zeros(a.shape, bool), np.zeros(a.shape, bool)
    for c in range(3):
        for j in range(-3, 4):
            p = list(at)
            p[c] += j
            image = p[c] < 0
            p[c] %= N_c[c]
            re[(0,) + tuple(p)] = True
            if image:
                im[(0,) + tuple(p)] = True
    assert (~np.isfinite(out.real) == re).all()
    assert (~np.isfinite(out.imag) == im).all()
