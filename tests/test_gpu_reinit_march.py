"""The two-kernel 3D stage where a march is one plane: a grid too wide for the
one-launch stage (300 workgroups of it), of 120 tiles over 8 planes (960 marches).
Steps and tolerances as in tests/test_gpu_reinit_split.py."""
import numpy as np
import pytest

from test_gpu_parity import TOL, load_state, pair, rel_err

pytestmark = pytest.mark.gpu

CASE = dict(nx=256, ny=120, nz=8, dim=3)


@pytest.mark.parametrize("btn", [0, 1])
def test_one_plane_march(btn):
    o, s = pair(**CASE)
    load_state(o, s, perturb=True)
    T = 2.5 * s.params.rdt
    n_o = o.redis(btn, T)
    err, n_g = s.reinit(btn, T)
    assert n_g == n_o == 3
    rel = rel_err(s.download_phi(), o.field("PHI"))
    print(f"btn={btn}: rel {rel:.2e}", flush=True)
    assert rel <= TOL
    assert abs(err - o.get("red_error")) <= TOL * max(1.0, err)
    s.close()


def test_one_plane_march_fp32():
    boxes = []
    for precision in (0, 1):
        o, s = pair(precision=precision, **CASE)
        load_state(o, s, perturb=True)
        s.reinit(1, 2.5 * s.params.rdt)
        boxes.append(s.download_phi())
        s.close()
    assert np.max(np.abs(boxes[0] - boxes[1])) <= 1e-5
