"""The advection line solves where the rows a lane takes change: lines of 34, 65,
97, 128 .. 130, 257 and 258 cells through the tiled solve (4096 lines or more), and
few lines through the partitioned one; smooth fields, where the cyclic reduction
ends early, and noise, where neighbouring interfaces stay coupled."""
import numpy as np
import pytest

from test_gpu_parity import TOL, load_state, pair, rel_err

pytestmark = pytest.mark.gpu

CASES = [
    dict(nx=34, ny=130, nz=65, dim=3),
    dict(nx=129, ny=97, nz=64, dim=3),
    dict(nx=128, ny=66, nz=98, dim=3),
    dict(nx=258, ny=36, nz=130, dim=3),
    dict(nx=33, ny=34, dim=2),
    dict(nx=257, ny=258, dim=2),
    dict(nx=65, ny=129, dim=2),
]


def ids(c):
    return "x".join(str(c[k]) for k in ("nx", "ny", "nz") if k in c)


@pytest.mark.parametrize("case", CASES, ids=ids)
@pytest.mark.parametrize("noise", [False, True])
def test_advection_rows(case, noise):
    o, s = pair(**case)
    load_state(o, s, shape=2 if case["dim"] == 3 else 1, perturb=True, field=2 if case["dim"] == 3 else 1)
    if noise:
        phi = o.field("PHI")
        phi += 0.5 * np.random.default_rng(case["nx"]).choice([-1.0, 0.0, 1.0], phi.shape)
        o.bc_field("PHI")
        s.upload_phi(phi)
    o.rk3_advect()
    s.rk3_advect()
    e = rel_err(s.download_phi(), o.field("PHI"))
    print(f"{ids(case)} noise={noise}: rel {e:.2e}", flush=True)
    assert e <= TOL
    s.close()


@pytest.mark.parametrize("case", CASES[:4] + CASES[5:6], ids=ids)
def test_advection_rows_fp32(case):
    """FP32 bulk against the FP64 path: one step moves phi (|phi| < 1) by less than
    a cell, so it stays within some FP32 roundings of the field."""
    boxes = []
    for precision in (0, 1):
        o, s = pair(precision=precision, **case)
        load_state(o, s, shape=2 if case["dim"] == 3 else 1, perturb=True, field=2 if case["dim"] == 3 else 1)
        s.rk3_advect()
        boxes.append(s.download_phi())
        s.close()
    diff = np.max(np.abs(boxes[0] - boxes[1]))
    print(f"{ids(case)} fp32: max diff {diff:.2e}", flush=True)
    assert diff <= 1e-5


@pytest.mark.parametrize("case", [dict(nx=129, ny=97, nz=64, dim=3), dict(nx=40, ny=36, nz=45, dim=3),
                                  dict(nx=258, ny=36, nz=130, dim=3)], ids=ids)
@pytest.mark.parametrize("precision", [0, 1])
def test_advection_rows_listed(case, precision):
    """Every line listed (a narrow band wider than the domain) against the plain
    pass: FP64 to the drop-in tolerance, FP32, whose listed lines take every
    step of the reduction over normalised rows, to some roundings of the field."""
    boxes = []
    for band in (0.0, 1000.0):
        o, s = pair(precision=precision, **case)
        load_state(o, s, shape=2, perturb=True, field=2)
        s.set_narrow_band(band)
        s.rk3_advect()
        boxes.append(s.download_phi())
        s.close()
    diff = np.max(np.abs(boxes[0] - boxes[1])) / np.max(np.abs(boxes[0]))
    print(f"{ids(case)} precision {precision}: diff {diff:.2e}", flush=True)
    assert diff <= (1e-5 if precision else TOL)
