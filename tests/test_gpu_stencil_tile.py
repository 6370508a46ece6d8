"""Tiles that set_tile asks for and no block can hold: the largest that fits,
not another kernel."""
import numpy as np
import pytest

torch = pytest.importorskip('torch')

pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():
    pytest.skip('no GPU', allow_module_level=True)

from gpaw_amd.fd_operators import Laplace  # noqa: E402
from gpaw_amd.grid_descriptor import GridDescriptor  # noqa: E402


def kernels(f):
    with torch.profiler.profile(
            activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
        f()
        torch.cuda.synchronize()
    return [e.name for e in prof.events()]


@pytest.mark.parametrize('N_c,nb,dtype', [
    ((40, 60, 64), 12, np.float64), ((24, 70, 90), 40, np.float32),
    ((40, 44, 45), 20, np.complex128)])
@pytest.mark.parametrize('tile', [(0, 0), (1, 0), (3, 7), (64, 0), (500, 500)])
def test_tile(N_c, nb, dtype, tile):
    rng = np.random.default_rng(2)
    gd = GridDescriptor(N_c, np.array(N_c) * 0.4)
    a = rng.standard_normal((nb,) + N_c)
    if np.dtype(dtype).kind == 'c':
        a = a + 1j * rng.standard_normal(a.shape)
    a = torch.from_numpy(a.astype(dtype)).cuda()
    want, out = torch.empty_like(a), torch.empty_like(a)
    Laplace(gd, -0.5, 3, dtype).apply(a, want)
    op = Laplace(gd, -0.5, 3, dtype)
    op.set_tile(*tile)
    names = kernels(lambda: op.apply(a, out))
    assert any('stencil_rows_kernel' in n for n in names), names
    assert torch.equal(out, want)
