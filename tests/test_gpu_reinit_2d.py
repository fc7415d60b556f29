"""The 2D reinitialisation stage at the edges of its columns (56 a wave with
lambda, 58 without), of its rows (2, 6 and 14 a workgroup with lambda, 4 and 8
without) and of the rule that picks them (2^14 and 2^17 cells)."""
import numpy as np
import pytest

from test_gpu_parity import TOL, load_state, pair, rel_err

pytestmark = pytest.mark.gpu

SIZES = [(4, 4), (56, 5), (57, 6), (58, 9), (59, 8), (113, 7), (117, 13), (128, 128), (129, 127),
         (128, 129), (300, 61), (512, 256), (512, 257), (447, 295), (465, 305)]


@pytest.mark.parametrize("nx,ny", SIZES)
@pytest.mark.parametrize("btn", [0, 1])
def test_reinit_2d_edges(nx, ny, btn):
    o, s = pair(nx, ny=ny, dim=2)
    load_state(o, s, shape=1, perturb=True, field=1)
    T = 2.5 * s.params.rdt
    n_o = o.redis(btn, T)
    err, n_g = s.reinit(btn, T)
    assert n_g == n_o == 3
    rel = rel_err(s.download_phi(), o.field("PHI"))
    print(f"{nx}x{ny} btn={btn}: rel {rel:.2e}", flush=True)
    assert rel <= TOL
    assert abs(err - o.get("red_error")) <= TOL * max(1.0, err)


@pytest.mark.parametrize("nx,ny", [(59, 8), (300, 61), (512, 257)])
@pytest.mark.parametrize("btn", [0, 1])
def test_reinit_2d_fp32(nx, ny, btn):
    """FP32 bulk against the FP64 path: three pseudo-steps of 0.1 dx keep the
    difference at some FP32 roundings of the field (|phi| < 1)."""
    boxes = []
    for precision in (0, 1):
        o, s = pair(nx, ny=ny, dim=2, precision=precision)
        load_state(o, s, shape=1, perturb=True, field=1)
        s.reinit(btn, 2.5 * s.params.rdt)
        boxes.append(s.download_phi())
    diff = np.max(np.abs(boxes[0] - boxes[1]))
    print(f"{nx}x{ny} btn={btn} fp32: max diff {diff:.2e}", flush=True)
    assert diff <= 1e-5
