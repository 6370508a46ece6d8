"""Stencils whose radius along one axis exceeds the points of another,
periodic one (accepted by gh_stencil_create, which compares every offset
with its own axis): no neighbour along the short axis may be read.  Against
a NumPy sum over the stencil's points; tolerances as in test_gpu_parity.py."""
import ctypes

import numpy as np
import pytest

torch = pytest.importorskip('torch')

pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():
    pytest.skip('no GPU', allow_module_level=True)

from gpaw_amd import _lib  # noqa: E402
from gpaw_amd._arrays import dtype_code, stream_ptr  # noqa: E402


def create(coefs, offs, n_c, pbc, dtype):
    h = ctypes.c_void_p()
    _lib.check(_lib.lib().gh_stencil_create(
        ctypes.byref(h), len(coefs), _lib.f64(coefs)[1],
        _lib.i64(np.ravel(offs))[1], _lib.i64(n_c)[1], _lib.i32(pbc)[1],
        dtype_code(dtype)))
    return h


def reference(coefs, offs, a, pbc, ph):
    out = np.zeros_like(a)
    for c, off in zip(coefs, offs):
        b = a
        for ax in range(3):
            n, o = a.shape[1 + ax], off[ax]
            i = np.arange(n) + o
            b = np.take(b, i % n, 1 + ax)
            f = np.ones(n, a.dtype)
            f[i < 0] = ph[ax, 1] if pbc[ax] else 0
            f[i >= n] = ph[ax, 0] if pbc[ax] else 0
            shape = [1] * 4
            shape[1 + ax] = n
            b = b * f.reshape(shape)
        out += c * b
    return out


@pytest.mark.parametrize('dtype', [np.float64, np.complex128, np.float32,
                                   np.complex64])
@pytest.mark.parametrize('n_c,axis,R,nb', [
    ((12, 1, 4), 0, 3, 3), ((12, 4, 1), 0, 3, 2), ((12, 2, 2), 0, 3, 1),
    ((1, 12, 16), 1, 3, 2), ((2, 9, 16), 1, 6, 2), ((4, 1, 16), 2, 2, 3),
    ((2, 2, 40), 2, 3, 4000)])
def test_short_periodic_axis(n_c, axis, R, nb, dtype):
    rng = np.random.default_rng(4)
    cplx = np.dtype(dtype).kind == 'c'
    single = dtype in (np.float32, np.complex64)
    offs = [(0, 0, 0)] + [tuple(s * j if c == axis else 0 for c in range(3))
                          for j in range(1, R + 1) for s in (1, -1)]
    coefs = rng.uniform(-1, 1, len(offs))
    pbc = [1, 1, 1]
    shape = (nb,) + n_c
    a = rng.standard_normal(shape)
    if cplx:
        a = a + 1j * rng.standard_normal(shape)
    a = a.astype(dtype)
    vt = rng.standard_normal(n_c).astype(np.float32 if single else float)
    eps = rng.uniform(-1, 1, nb)
    ph = np.ones((3, 2), complex)
    if cplx:
        p = np.exp(2j * np.pi * np.array([0.2, -0.1, 0.4]))
        ph[:, 0], ph[:, 1] = p, p.conj()
    wide = a.astype(complex if cplx else float)
    ref = reference(coefs, offs, wide, pbc, ph if cplx else ph.real)
    tol = 2e-5 if single else 1e-12
    # the array in the middle of NaN: a value read from outside it shows
    n = a.size
    pool = torch.full((n + 8192,), float('nan'),
                      dtype=torch.from_numpy(a[:0]).dtype, device='cuda')
    ad = pool[4096:4096 + n].reshape(shape)
    ad.copy_(torch.from_numpy(a))
    vd, ed = torch.from_numpy(vt).cuda(), torch.from_numpy(eps).cuda()
    out = torch.empty_like(ad)
    L = _lib.lib()
    h = create(coefs, offs, n_c, pbc, dtype)
    keep, php = _lib.phase_arg(ph) if cplx else (None, None)

    def check(want):
        got = out.cpu().numpy()
        assert abs(got - want).max() < tol * abs(want).max()
    _lib.check(L.gh_stencil_apply(h, ad.data_ptr(), out.data_ptr(), nb, php,
                                  None, None, 0.0, stream_ptr()))
    check(ref)
    _lib.check(L.gh_stencil_apply_shifted(
        h, ad.data_ptr(), out.data_ptr(), nb, php, vd.data_ptr(),
        ed.data_ptr(), stream_ptr()))
    check(ref + (vt - eps[:, None, None, None]) * wide)
    if not cplx:
        work = torch.empty_like(vd)
        f, s = ad[0].clone(), torch.from_numpy(vt).cuda()
        _lib.check(L.gh_stencil_relax(
            h, 2, f.data_ptr(), s.data_ptr(), work.data_ptr(), 1, 0.7,
            stream_ptr()))
        want = wide[0] + 0.7 / coefs[0] * (vt - ref[0])
        assert abs(f.cpu().numpy() - want).max() < tol * abs(want).max()
    L.gh_stencil_destroy(h)


@pytest.mark.parametrize('dtype', [np.float64, np.float32])
def test_batch_with_a_short_axis(dtype):
    """One cell of a batch with a radius beyond its periodic axis."""
    rng = np.random.default_rng(6)
    R = 3
    offs = [(0, 0, 0)] + [(s * j, 0, 0) for j in range(1, R + 1)
                          for s in (1, -1)]
    coefs = rng.uniform(-1, 1, len(offs))
    cells = [((12, 2, 4), 3), ((10, 8, 12), 2)]
    L = _lib.lib()
    hs = [create(coefs, offs, n_c, [1, 1, 1], dtype) for n_c, nb in cells]
    nbs = [nb for n_c, nb in cells]
    b = ctypes.c_void_p()
    _lib.check(L.gh_stencil_batch_create(
        ctypes.byref(b), 2, (_lib.P * 2)(*[h.value for h in hs]),
        _lib.i64(nbs)[1], None, None, 1))
    a = [rng.standard_normal((nb,) + n_c).astype(dtype) for n_c, nb in cells]
    v = [rng.standard_normal(n_c).astype(dtype) for n_c, nb in cells]
    ad = [torch.from_numpy(x).cuda() for x in a]
    vd = [torch.from_numpy(x).cuda() for x in v]
    od = [torch.full_like(x, float('nan')) for x in ad]
    ptrs = [(_lib.P * 2)(*[x.data_ptr() for x in t]) for t in (ad, od, vd)]
    _lib.check(L.gh_stencil_batch_apply(b, *ptrs, stream_ptr()))
    tol = 2e-5 if dtype == np.float32 else 1e-12
    for x, y, o in zip(a, v, od):
        x = x.astype(float)
        want = reference(coefs, offs, x, [1, 1, 1], np.ones((3, 2))) + y * x
        assert abs(o.cpu().numpy() - want).max() < tol * abs(want).max()
    L.gh_stencil_batch_destroy(b)
    for h in hs:
        L.gh_stencil_destroy(h)
