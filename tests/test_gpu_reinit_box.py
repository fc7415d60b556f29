"""The 3D reinitialisation stage that forms lambda in the same launch, at the edges
of its columns (56 a wave), rows (2 or 6 a workgroup) and planes (1 to 3), on
both sides of the rules that choose it, and against the two-kernel stage, which
a narrow band wider than the domain runs over every cell."""
import numpy as np
import pytest

from test_gpu_parity import TOL, load_state, pair, rel_err

pytestmark = pytest.mark.gpu

SIZES = [(4, 4, 4), (16, 16, 16), (24, 25, 23), (56, 9, 11), (57, 8, 7), (113, 5, 6), (40, 41, 39), (48, 48, 48),
         (49, 47, 50), (56, 56, 56), (110, 40, 40), (57, 57, 57)]


@pytest.mark.parametrize("nx,ny,nz", SIZES)
def test_reinit_box_parity(nx, ny, nz):
    o, s = pair(nx, ny=ny, nz=nz, dim=3)
    load_state(o, s, perturb=True)
    T = 2.5 * s.params.rdt
    n_o = o.redis(1, T)
    err, n_g = s.reinit(1, T)
    assert n_g == n_o == 3
    rel = rel_err(s.download_phi(), o.field("PHI"))
    print(f"{nx}x{ny}x{nz}: rel {rel:.2e}", flush=True)
    assert rel <= TOL
    assert abs(err - o.get("red_error")) <= TOL * max(1.0, err)


@pytest.mark.parametrize("nx,ny,nz", [(16, 16, 16), (57, 8, 7), (48, 48, 48), (56, 56, 56)])
@pytest.mark.parametrize("precision", [0, 1])
def test_reinit_box_against_two_kernels(nx, ny, nz, precision):
    """Ten pseudo-steps: FP64 to the drop-in tolerance, FP32 to some roundings of
    the field (|phi| < 1)."""
    boxes = []
    for band in (0.0, 1000.0):
        o, s = pair(nx, ny=ny, nz=nz, dim=3, precision=precision)
        load_state(o, s, perturb=True)
        s.set_narrow_band(band)
        s.reinit(1, 9.5 * s.params.rdt)
        boxes.append(s.download_phi())
        s.close()
    diff = np.max(np.abs(boxes[0] - boxes[1])) / np.max(np.abs(boxes[1]))
    print(f"{nx}x{ny}x{nz} precision {precision}: diff {diff:.2e}", flush=True)
    assert diff <= (1e-5 if precision else TOL)
