"""The 3D reinitialisation on grids that cut its z march differently: one
plane a workgroup, short marches with a remainder, and marches of eight."""
import numpy as np
import pytest

from test_gpu_parity import TOL, load_state, pair, rel_err

pytestmark = pytest.mark.gpu

# nx, ny, nz, planes per workgroup that the grid gets
SPLITS = [
    (33, 9, 37, 1),       # 4 tiles: one plane each
    (64, 64, 66, 2),      # 16 tiles, whole marches
    (100, 100, 53, 3),    # 52 tiles, a remainder of two planes
    (250, 132, 40, 6),    # 136 tiles, a remainder of four planes
    (512, 256, 20, 8),    # 512 tiles: more than one round of workgroups
]


@pytest.mark.parametrize("nx,ny,nz,planes", SPLITS)
@pytest.mark.parametrize("btn", [0, 1])
def test_reinit_split_parity(nx, ny, nz, planes, btn):
    o, s = pair(nx, ny=ny, nz=nz, dim=3)
    load_state(o, s, perturb=True)
    steps = 3 if nx * ny * nz < 1000000 else 1
    T = (steps - 0.5) * s.params.rdt
    n_o = o.redis(btn, T)
    err, n_g = s.reinit(btn, T)
    assert n_g == n_o == steps
    rel = rel_err(s.download_phi(), o.field("PHI"))
    print(f"{nx}x{ny}x{nz} ({planes} planes) btn={btn}: rel {rel:.2e}", flush=True)
    assert rel <= TOL
    assert abs(err - o.get("red_error")) <= TOL * max(1.0, err)


@pytest.mark.parametrize("nx,ny,nz,planes", SPLITS[:4])
def test_reinit_split_fp32(nx, ny, nz, planes):
    """FP32 bulk against the FP64 path: three pseudo-steps of 0.1 dx keep the
    difference at some FP32 roundings of the field (|phi| < 1)."""
    boxes = []
    for precision in (0, 1):
        o, s = pair(nx, ny=ny, nz=nz, dim=3, precision=precision)
        load_state(o, s, perturb=True)
        s.reinit(1, 2.5 * s.params.rdt)
        boxes.append(s.download_phi())
    diff = np.max(np.abs(boxes[0] - boxes[1]))
    print(f"{nx}x{ny}x{nz} ({planes} planes) fp32: max diff {diff:.2e}", flush=True)
    assert diff <= 1e-5
