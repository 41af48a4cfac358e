"""The sums of the training pass (over a workgroup's wavefronts, then over the
workgroups' partials) against the FP64 oracle, at the ends of what they
cover: one sample (three of the four wavefronts without any), one tile and a
bit, fewer partials than the reduction has rows, a ragged last row of them, and
every wavefront with several tiles."""
import numpy as np
import pytest

from oracle import warm_start as W

from helpers import gpu_world
from test_gpu_warm_start import _net, _samples

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 17, 320, 33 * 64 + 5, 16 * 1024 * 2 + 3])
def test_gradient_sums_match_oracle(n):
    w = gpu_world()
    p = _net(n % 7)
    assert w.set_warm_start_net(p)
    X, t = _samples(n, n)
    y, g, loss = w.debug_warm_net(X, t)
    lo, go, yo = W.loss_and_grad(p.astype(np.float64), X, t, emulate=True)
    # A tile or a wavefront left out or taken twice is off by its share of the
    # batch (1/2049 at the largest), and shows in every parameter.  What is
    # allowed: FP32 sums and, where FP32 rounds an activation to the other
    # BF16 neighbour, 2^-8 of that sample's share; 5e-3 for a handful of
    # samples, and 1e-4 (a wavefront's share over 4) from a thousand on, where
    # such roundings are few and of either sign.
    tol = 5e-3 if n < 1000 else 1e-4
    assert np.abs(g - go).max() <= tol * np.abs(go).max()
    assert abs(loss - lo) <= tol * lo
    # The same again: a sum that depends on timing would differ.
    _, g2, loss2 = w.debug_warm_net(X, t)
    assert np.array_equal(g, g2) and loss == loss2
