"""The CCD solve on both sides of the rule that gives a line 32 lanes or one
(40,960 lines along y or z; x lines always 32), and of the one that keeps a large
coefficient table in LDS (512 workgroups): the energy integrals, which
solve every line of three fields, to 1e-12 of the oracle's, and the mass
correction on every line against the one on band lines."""
import numpy as np
import pytest

from test_gpu_energy import run
from test_gpu_parity import TOL, pair, rel_err

pytestmark = pytest.mark.gpu

CASES = [
    dict(nx=66, ny=65, nz=64, dim=3),
    dict(nx=200, ny=8, nz=204, dim=3),   # 40,800 y lines
    dict(nx=200, ny=8, nz=205, dim=3),   # 41,000
    dict(nx=11, ny=210, nz=200, dim=3),  # 42,000 x lines
    dict(nx=700, ny=40, nz=40, dim=3),   # a table of 73 KB in LDS: 400 workgroups
    dict(nx=700, ny=52, nz=40, dim=3),   # and in memory: 520
]


def ids(c):
    return "x".join(str(c[k]) for k in ("nx", "ny", "nz"))


@pytest.mark.parametrize("case", CASES, ids=ids)
def test_energy_lines(case):
    e_o, e_g, vscale = run(case, 0)
    for k in e_o:
        tol = TOL * (vscale if k in ("px", "py", "pz") else abs(e_o[k]))
        print(f"{ids(case)} {k}: oracle {e_o[k]:.15e} gpu {e_g[k]:.15e}", flush=True)
        assert abs(e_g[k] - e_o[k]) <= tol + 1e-300, k


@pytest.mark.parametrize("case", CASES, ids=ids)
def test_mass_every_line(case):
    boxes = []
    for mode in (0, 2):
        o, s = pair(**case)
        o.initial_phi(2, 0)
        o.store_initial()
        s.upload_phi(o.field("PHI") + 0.1 * o.p.dx)
        s.set_band_lines(mode)
        s.mass_fix(o.get("imass"))
        boxes.append(s.download_phi())
        s.close()
    e = rel_err(boxes[0], boxes[1])
    print(f"{ids(case)}: rel {e:.2e}", flush=True)
    assert e <= TOL
    assert np.isfinite(boxes[0]).all()
