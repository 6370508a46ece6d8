"""Rotation of wave functions at the edges of its 16 x 16 x 4 tiles and at
the largest sizes, against a product in FP64 on the CPU; infinities stay in
the rows of the functions that hold them."""
import pytest

torch = pytest.importorskip('torch')
pytestmark = pytest.mark.gpu

from gpaw_amd import _lib, blas  # noqa: E402
from gpaw_amd._arrays import stream_ptr  # noqa: E402


# k products of order one: k roundings of 1.1e-16 of at most k
@pytest.mark.parametrize('m,k', [(1, 1), (3, 5), (16, 16), (17, 15), (48, 33),
                                 (64, 64), (10, 64), (64, 1), (65, 64)])
@pytest.mark.parametrize('n', [1, 15, 17, 4096 * 16 + 3])
def test_rotate(m, k, n):
    g = torch.Generator().manual_seed(m * 100 + k)
    U = torch.randn(m, k, generator=g, dtype=torch.float64)
    psi = torch.randn(k, n, generator=g, dtype=torch.float64)
    out = blas.rotate(U.cuda(), psi.cuda()).cpu()
    want = U @ psi
    assert out.shape == want.shape
    assert (out - want).abs().max() <= 1.1e-16 * k * (k + 12)


def test_transposed_and_infinite():
    g = torch.Generator().manual_seed(7)
    U = torch.randn(20, 30, generator=g, dtype=torch.float64)
    psi = torch.randn(20, 50, generator=g, dtype=torch.float64)
    psi[19, 7] = float('inf')
    out = blas.rotate(U.T.cuda(), psi.cuda()).cpu()
    want = U.T @ psi
    assert torch.equal(torch.isinf(out), torch.isinf(want))
    assert bool((torch.isinf(out).sum(0) == 30 * (torch.arange(50) == 7)).all())


def rotate_kernel(U, psi):
    out = torch.full((U.shape[0], psi.shape[1]), float('nan'),
                     dtype=torch.float64, device='cuda')
    U, psi = U.contiguous().cuda(), psi.cuda()
    _lib.check(_lib.lib().gh_rotate(*U.shape, psi.shape[1], U.data_ptr(),
                                    psi.data_ptr(), out.data_ptr(),
                                    stream_ptr()))
    return out.cpu()


@pytest.mark.parametrize('m,k', [(1, 1), (2, 2), (3, 5), (16, 16), (17, 15),
                                 (48, 33), (64, 64), (10, 64), (64, 1)])
@pytest.mark.parametrize('n', [1, 15, 17, 8191, 300007])
def test_kernel(m, k, n):
    """The kernel itself, also where rotate() takes the library's product."""
    g = torch.Generator().manual_seed(m * 100 + k)
    U = torch.randn(m, k, generator=g, dtype=torch.float64)
    psi = torch.randn(k, n, generator=g, dtype=torch.float64)
    out, want = rotate_kernel(U, psi), U @ psi
    assert (out - want).abs().max() <= 1.1e-16 * k * (k + 12)


@pytest.mark.parametrize('n', [100, 10000])
def test_other_devices_are_refused(n):
    """A matrix or functions in host memory: an error, as for U @ psi."""
    U = torch.ones(4, 4, dtype=torch.float64)
    psi = torch.ones(4, n, dtype=torch.float64)
    for a, b in ((U, psi.cuda()), (U.cuda(), psi)):
        with pytest.raises(RuntimeError):
            blas.rotate(a, b)


@pytest.mark.parametrize('n', [100, 10000])
def test_negated_views(n):
    """Views that carry a pending sign (the imaginary part of a conjugate)."""
    g = torch.Generator().manual_seed(3)
    z = torch.randn(1, 1, generator=g, dtype=torch.complex128).cuda()
    U = z.conj().imag
    psi = torch.randn(1, n, generator=g, dtype=torch.float64).cuda()
    assert torch.equal(blas.rotate(U, psi), -z.imag * psi)
