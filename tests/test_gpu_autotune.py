"""The tuners time the kernels whose tiles they choose: single grids over row
counts only, the cells of a batch in the batched kernel."""
import numpy as np
import pytest

torch = pytest.importorskip('torch')
pytestmark = pytest.mark.gpu

from gpaw_amd import autotune  # noqa: E402
from gpaw_amd.fd_operators import FDOperator, Laplace  # noqa: E402
from gpaw_amd.grid_descriptor import GridDescriptor  # noqa: E402


def operator(N_c=(24, 20, 28), dtype=np.float32):
    return Laplace(GridDescriptor(N_c, np.array(N_c) * 0.3), -0.5, 3, dtype)


@pytest.fixture(autouse=True)
def no_memory(monkeypatch):
    for name in ('_CACHE', '_CELL_CACHE', '_BATCH_CACHE'):
        monkeypatch.setattr(autotune, name, {})


def test_single_grid_rows_only(monkeypatch):
    """Every row count once: a prefetch depth would only repeat the tile."""
    op, tiles = operator(), []
    set_tile = FDOperator.set_tile
    monkeypatch.setattr(FDOperator, 'set_tile',
                        lambda self, rows=0, planes=0, depth=0:
                        tiles.append(rows) or set_tile(self, rows, planes,
                                                       depth))
    rows, depth, ms = autotune.tune_stencil(op, 3, with_v=True)
    tried = tiles[:-1]
    assert len(tried) == len(set(tried)) and tiles[-1] == rows in tried
    assert ms > 0 and autotune.tune_stencil(op, 3, with_v=True)[0] == rows


def test_cells_in_the_batched_kernel(monkeypatch):
    """No single-grid launch decides a batch's tiles."""
    ops = [operator(), operator((32, 24, 16))]

    def refuse(*args, **kwargs):
        raise AssertionError('single-grid launch')
    monkeypatch.setattr(FDOperator, 'apply', refuse)
    own = [autotune.tune_cell(op, 4) for op in ops]
    assert all(rows >= 1 and depth in (2, 3) for rows, depth, ms in own)
    rows, depths, ms, label = autotune.tune_batch(ops, [4, 2])
    assert len(rows) == len(depths) == 2 and ms > 0


def test_cells_no_batch_takes():
    assert autotune.tune_cell(operator((12, 10, 7)), 2) is None
