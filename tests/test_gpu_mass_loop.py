"""The mass correction's iterations queued ahead of the host: the stop test is
taken on the device, so a queue that is longer or shorter than the iterations
needed, and an error within it, must leave what a loop of single iterations
leaves.  The grids lie on both sides of the rules that let the update form the
totals (at most 256 block sums and 2^19 cells)."""
import numpy as np
import pytest

from conftest import load_lsmp
from test_gpu_parity import TOL, pair, rel_err

pytestmark = pytest.mark.gpu

CASES = [
    dict(nx=33, ny=9, nz=37, dim=3),       # 42 sums: totals in the update
    dict(nx=66, ny=65, nz=64, dim=3),      # 537 sums: a launch of their own, every line updated
    dict(nx=1024, ny=512, dim=2),          # 2^19 cells
    dict(nx=1024, ny=513, dim=2),          # one row more
    dict(nx=5, ny=4, dim=2),
]


def ids(c):
    return "x".join(str(c[k]) for k in ("nx", "ny", "nz") if k in c)


@pytest.mark.parametrize("case", CASES, ids=ids)
def test_mass_iterations_queued(case):
    o, s = pair(**case)
    o.initial_phi(2 if case["dim"] == 3 else 1, 0)
    o.store_initial()
    imass = o.get("imass")
    # one solver through corrections of different lengths: each queue is as long
    # as the correction before it
    for shift in (0.1, 0.0, 0.3, 1e-6):
        o.field("PHI")[:] += shift * o.p.dx
        s.upload_phi(o.field("PHI"))
        no = o.mass_fix()
        mass, ng = s.mass_fix(imass)
        e = rel_err(s.download_phi(), o.field("PHI"))
        print(f"{ids(case)} shift {shift}: iterations {no}/{ng} rel {e:.2e}", flush=True)
        assert abs(ng - no) <= 1 and e <= TOL
        assert abs(mass - imass) <= 1e-13 * imass   # of the last iteration's field
    s.close()


@pytest.mark.parametrize("case", CASES[:4], ids=ids)
def test_queue_length_changes_nothing(case):
    """FP32 bulk and FP64: a fresh solver and one whose queue is long give the
    same bits, the same mass and the same iteration count."""
    for precision in (0, 1):
        out = []
        for before in ((), (0.9, 0.9)):
            o, s = pair(precision=precision, **case)
            o.initial_phi(2 if case["dim"] == 3 else 1, 0)
            o.store_initial()
            box = o.field("PHI").copy()
            for shift in before:
                s.upload_phi(box + shift * o.p.dx)
                s.mass_fix(o.get("imass"))
            s.upload_phi(box + 1e-4 * o.p.dx)
            mass, n = s.mass_fix(o.get("imass"))
            out.append((s.download_phi(), mass, n))
            s.close()
        print(f"{ids(case)} precision {precision}: {out[0][2]} iterations", flush=True)
        assert out[0][1:] == out[1][1:]
        assert np.array_equal(out[0][0], out[1][0])


@pytest.mark.parametrize("case", CASES[:2], ids=ids)
def test_empty_band_within_a_queue(case):
    """No cell in the band is an error, leaves phi as it was, and the next
    correction on the same solver is a first one's."""
    lsmp = load_lsmp()
    o, s = pair(**case)
    o.initial_phi(2, 0)
    o.store_initial()
    imass = o.get("imass")
    good = o.field("PHI") + 0.3 * o.p.dx
    s.upload_phi(good)
    first = s.mass_fix(imass)
    ref = s.download_phi()
    far = np.ones_like(good)
    s.upload_phi(far)
    with pytest.raises(lsmp.LsmpError, match="-4"):
        s.mass_fix(imass)
    assert np.array_equal(s.download_phi(), far)
    s.upload_phi(good)
    assert s.mass_fix(imass) == first
    assert np.array_equal(s.download_phi(), ref)
    s.close()
