"""The gradient sums of a training step over numbers of workgroups (64 samples
each) below, at and past the update kernel's 16 waves, with a remainder."""
import numpy as np
import pytest

from conftest import load_lsmp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 64 * 15, 64 * 16, 64 * 16 + 1, 64 * 37 + 5])
def test_gradient_sums(n):
    """The loss and its gradient are means over the samples: n copies of one
    sample have that sample's, up to the rounding of n FP32 terms (2^-24 each,
    of gradients below 1)."""
    lsmp = load_lsmp()
    rng = np.random.default_rng(n)
    x1 = rng.normal(size=(1, 128)).astype(np.float32)
    y1 = np.array([0.3], np.float32)
    net = lsmp.Net(capacity=0, seed=3)
    l1, g1 = net.eval_grad(x1, y1)
    ln, gn = net.eval_grad(np.repeat(x1, n, axis=0), np.repeat(y1, n))
    # dZ is rounded to BF16 before the weight gradients (2^-9 relative, the
    # same for every copy but for the factor 1/n, which may round differently)
    tol = 2.0 ** -8 * np.abs(g1).max()
    print(n, l1, ln, np.abs(gn - g1).max(), tol, flush=True)
    assert abs(ln - l1) <= 1e-5 * abs(l1)
    assert np.abs(gn - g1).max() <= tol
