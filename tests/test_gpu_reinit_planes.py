"""The 3D reinitialisation over more planes than a grid dimension takes blocks of
sixteen (65,535 of them): a field that repeats along z must come out as on a short
grid, bit for bit, at both ends and, repeated, in between."""
import numpy as np
import pytest

from conftest import load_lsmp

pytestmark = pytest.mark.gpu

PERIOD = 1000


def run(nz, btn):
    lsmp = load_lsmp()
    p = lsmp.make_params(4, ny=4, nz=nz, precision=lsmp.FP32)
    h = p.dx
    p.dy = p.dz = h
    p.dt = p.rdt = 0.1 * h
    k = np.clip(np.arange(-3, nz + 3), 0, nz - 1) % PERIOD
    i = np.clip(np.arange(-3, 7), 0, 3)
    z = np.minimum(k, PERIOD - k) / PERIOD * 6 * h          # a zigzag of slope 0.012
    phi = 0.8 * h * (i[None, None, :] - 1.3) + 0.3 * h * i[None, :, None] - z[:, None, None]
    with lsmp.Solver(p) as s:
        s.upload_phi(np.ascontiguousarray(phi))
        assert s.reinit(btn, 1.5 * p.rdt)[1] == 2
        return s.download_phi()[3:-3, 3:-3, 3:-3].astype(np.float32)


@pytest.mark.parametrize("btn", [0, 1])
def test_planes_without_bound(btn):
    ref = run(20 * PERIOD, btn)
    long = run(1049 * PERIOD, btn)       # 65,563 blocks of sixteen planes
    assert np.isfinite(long).all()
    assert np.array_equal(long[:10 * PERIOD], ref[:10 * PERIOD])
    assert np.array_equal(long[-10 * PERIOD:], ref[-10 * PERIOD:])
    inner = long[10 * PERIOD:-10 * PERIOD].reshape(-1, PERIOD, 4, 4)
    assert (inner == inner[0]).all()
