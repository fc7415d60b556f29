"""The CCD solve on both sides of the line count, which grows with the length, up to
which every line takes 32 lanes: the energy integrals against the oracle's, to
the tolerances of tests/test_gpu_energy.py."""
import pytest

from test_gpu_energy import run

pytestmark = pytest.mark.gpu

# y lines of 20 cells: 220 a cell in FP64, 340 in FP32; of 240 cells (eight rows a lane): 16,000
CASES = [
    (dict(nx=60, ny=20, nz=73, dim=3), 0), (dict(nx=60, ny=20, nz=75, dim=3), 0),
    (dict(nx=60, ny=20, nz=112, dim=3), 1), (dict(nx=60, ny=20, nz=115, dim=3), 1),
    (dict(nx=125, ny=240, nz=128, dim=3), 0), (dict(nx=126, ny=240, nz=128, dim=3), 0),
    # 42,000 x lines of 130 cells, which have no limit
    (dict(nx=130, ny=210, nz=200, dim=3), 0),
]


@pytest.mark.parametrize("case,precision", CASES,
                         ids=["{nx}x{ny}x{nz}_".format(**c) + ("fp32" if p else "fp64") for c, p in CASES])
def test_energy_lines(case, precision):
    e_o, e_g, vscale = run(case, precision)
    for k in e_o:
        tol = (1e-5 if precision else 1e-12) * (vscale if k in ("px", "py", "pz") else abs(e_o[k]))
        assert abs(e_g[k] - e_o[k]) <= tol + 1e-300, (k, e_g[k], e_o[k])
