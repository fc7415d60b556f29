"""A field read out into its ghosted host box: every interior value unchanged,
every ghost the boundary cell's, over boxes that one thread writes and boxes that
several do (from 8 MiB), rows that fit the staging halves of 4 MiB and one that
does not."""
import numpy as np
import pytest

from conftest import load_lsmp

pytestmark = pytest.mark.gpu

SHAPES = [(5, 4, 6, 3), (33, 9, 37, 3), (131, 77, 101, 3), (257, 130, 64, 3), (70, 67, 1, 2), (1100, 700, 1, 2),
          (530000, 4, 1, 2)]


@pytest.mark.parametrize("nx,ny,nz,dim", SHAPES)
@pytest.mark.parametrize("precision", [0, 1])
def test_readout_box(nx, ny, nz, dim, precision):
    lsmp = load_lsmp()
    s = lsmp.Solver(lsmp.make_params(nx, dim=dim, ny=ny, nz=nz if dim == 3 else None, precision=precision))
    inner = np.random.default_rng(nx).standard_normal((nz, ny, nx))
    if precision:
        inner = inner.astype(np.float32).astype(np.float64)
    box = np.full((nz + 6, ny + 6, nx + 6), np.nan)
    box[3:-3, 3:-3, 3:-3] = inner
    s.upload_phi(box)
    for _ in range(2):
        got = s.download_phi()
        assert np.array_equal(got, np.pad(inner, 3, mode="edge"))
    s.close()
