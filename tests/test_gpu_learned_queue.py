"""The learned reinitialisation runs the sweeps it is asked for, whatever the
solver ran before: a plain reinitialisation of one and of five pseudo-steps must
not shorten it, and the field must be a fresh solver's, bit for bit."""
import numpy as np
import pytest

from conftest import load_lsmp
from test_gpu_learned import sphere_box

pytestmark = pytest.mark.gpu


# the one-launch stage, the two-kernel stage, 2D
@pytest.mark.parametrize("n,dim", [(24, 3), (72, 3), (48, 2)])
@pytest.mark.parametrize("precision", [0, 1])
def test_sweeps_after_a_plain_run(n, dim, precision):
    lsmp = load_lsmp()
    p = lsmp.make_params(n, dim=dim, precision=precision)
    box = sphere_box(n, dim=dim, warp=0.3)
    with lsmp.Net(seed=3) as net:
        for use in (net, None):
            for steps in (1, 5):
                for sweeps in (2, 8):
                    out = []
                    for before in (0, steps):
                        with lsmp.Solver(p) as s:
                            s.upload_phi(box)
                            if before:
                                assert s.reinit(1, (before - 0.5) * p.rdt)[1] == before
                                s.upload_phi(box)
                            # no residual is above the tolerance: no continuation
                            res, fallback, n_pseudo = s.reinit_learned(use, sweeps=sweeps, residual_tol=1e9)
                            assert n_pseudo == sweeps and not fallback
                            out.append((res, s.download_phi()))
                    assert out[0][0] == out[1][0] and np.array_equal(out[0][1], out[1][1])
