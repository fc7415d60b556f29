"""The narrow band in FP32 keeps its roundings whatever solve a line takes.

Beyond the tube's edge phi is +-W up to the rounding of the advection, and a tile
with a cell |phi| < W belongs to the tube, so that other roundings move the tube's
edge by a tile here and there (0.2 dx in its flat cells): a tolerance on phi cannot
tell.  The digests are those of the full reduction over normalised rows and of the
reinitialisation with expanded indicators (the library at commit a3d2939), after
three advections and after four pseudo-steps behind them.  The input takes
products, sums and square roots only, which round the same everywhere."""
import hashlib

import numpy as np
import pytest

from conftest import load_lsmp

pytestmark = pytest.mark.gpu

DIGESTS = {
    (40, 42, 44): ("39764f01a1e8668b", "0bd46a9e8163ef67"),   # a wave per line
    (66, 65, 64): ("105e9287408b23c6", "3023467646980c1e"),
    (40, 40, 300): ("b7aafdee2f99e346", "351df2b4b9ffe249"),   # sixteen rows a lane
    (30, 28, 26): ("c6fbc37d0996d859", "e0473501a3d50e02"),   # paired and twisted solves: short lines
    (530, 36, 38): ("11ed1d2c8bf498bd", "f120b1801e970c1c"),   # tiles of long lines along x
    (38, 530, 36): ("1d12c310e310782f", "b1f070845f7c706f"),   # and along y
    (36, 38, 530): ("da304395188386c9", "88910a1ec8694ac2"),   # the twisted solve along z
    (1030, 20, 22): ("63331d6b0a1aa49c", "cbb4804c30dab99f"),   # paired and twisted solves: long lines
    (20, 1030, 22): ("983798956c9b58f6", "d10074be25f66c44"),
    (20, 22, 1030): ("33e290496a3e49b8", "48246d826e1e751d"),
}


def fields(nx, ny, nz):
    """An ellipsoid, long along the grid's long side, and a smooth velocity."""
    n, least = (nx, ny, nz), min(nx, ny, nz)
    h = 1.0 / max(n)
    x, y, z = ((np.arange(-3, m + 3) + 0.5) * h for m in n)
    x, y, z = x[None, None, :], y[None, :, None], z[:, None, None]
    sx, sy, sz = (least / m for m in n)
    phi = 0.31 * least * h - np.sqrt(((x - 0.5 * nx * h) * sx) ** 2 + ((y - 0.5 * ny * h) * sy) ** 2 +
                                     ((z - 0.5 * nz * h) * sz) ** 2)
    phi = phi * (1 + 0.2 * (x - 0.5 * nx * h) / (nx * h))
    u = (1 - 2 * y) * x * (1 - x) + 0 * z
    v = (2 * x - 1) * y * (1 - y) + 0.3 * z
    w = 0.5 * (x - y) + 0.2 * z * (1 - z)
    return h, [np.ascontiguousarray(np.broadcast_to(f, phi.shape)) for f in (phi, u, v, w)]


def digest(s):
    phi = s.download_phi()[3:-3, 3:-3, 3:-3].astype(np.float32)
    assert np.isfinite(phi).all()
    return hashlib.sha256(np.ascontiguousarray(phi).tobytes()).hexdigest()[:16]


@pytest.mark.parametrize("grid", list(DIGESTS), ids=lambda g: "x".join(map(str, g)))
def test_narrow_band_fp32_bits(grid):
    lsmp = load_lsmp()
    h, (phi, u, v, w) = fields(*grid)
    p = lsmp.make_params(grid[0], ny=grid[1], nz=grid[2], precision=lsmp.FP32)
    p.dx = p.dy = p.dz = h
    p.dt = p.rdt = 0.1 * h
    p.ls_wid = 1.5 * h
    with lsmp.Solver(p) as s:
        s.upload_phi(phi)
        s.set_velocity(u, v, w)
        s.set_narrow_band(5.0)
        for _ in range(3):
            s.rk3_advect()
        got = [digest(s)]
        assert s.reinit(1, 3.5 * p.rdt)[1] == 4
        got.append(digest(s))
    print(grid, got, flush=True)
    assert tuple(got) == DIGESTS[grid]
