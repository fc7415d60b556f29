"""Pseudo-steps queued ahead of the host's look at the control words: as many as
the last run took.  A queue longer than the run, shorter than it, and one whose
run stops at its first step must leave what a fresh solver leaves."""
import numpy as np
import pytest

from test_gpu_parity import load_state, pair

pytestmark = pytest.mark.gpu

CASES = [dict(nx=33, ny=9, nz=37, dim=3), dict(nx=70, ny=67, dim=2)]


@pytest.mark.parametrize("case", CASES, ids=["3d", "2d"])
@pytest.mark.parametrize("precision", [0, 1])
def test_reinit_queue_length_changes_nothing(case, precision):
    o, s = pair(precision=precision, **case)
    load_state(o, s, shape=2 if case["dim"] == 3 else 1, perturb=True, field=case["dim"] - 1)
    box = o.field("PHI").copy()
    rdt = s.params.rdt
    for steps in (3, 40, 1, 70, 17):   # shorter, longer, past the queue's cap
        s.upload_phi(box)
        err, n = s.reinit(0, (steps - 0.5) * rdt)
        _, f = pair(precision=precision, **case)
        f.upload_phi(box)
        assert f.reinit(0, (steps - 0.5) * rdt) == (err, n) and n == steps
        assert np.array_equal(s.download_phi(), f.download_phi())
        f.close()
    # phi = 0 has no sign (0/0, as in the oracle) and stops after one step, whatever is queued
    zero = np.zeros_like(box)
    o.field("PHI")[:] = zero
    assert o.redis(0, 50.5 * rdt) == 1 and np.isnan(o.field("PHI")).all()
    _, f = pair(precision=precision, **case)
    f.upload_phi(zero)
    s.upload_phi(zero)
    assert s.reinit(0, 50.5 * rdt) == f.reinit(0, 50.5 * rdt) == (0.0, 1)
    assert np.array_equal(s.download_phi(), f.download_phi(), equal_nan=True)
    f.close()
    s.upload_phi(box)
    _, n = s.reinit(0, 4.5 * rdt)
    assert n == 5
    s.close()
