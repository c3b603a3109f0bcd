"""sph_mlp_eval's kept buffer: calls of growing, shrinking and very large sizes
on one handle (tiles of 64 points; above 64 MiB the buffer is given back) give
the bits of a call on a fresh handle."""
import numpy as np
import pytest

import cudasphnew_amd as S

pytestmark = pytest.mark.gpu


def test_sizes_in_any_order():
    lo, hi = [-0.05] * 3, [1.05] * 3
    pts = np.random.default_rng(3).uniform(-0.05, 1.05, (2500001, 3)).astype(np.float32)
    net = S.NeuralSDF(lo, hi, seed=1, out_scale=0.5)
    want = S.NeuralSDF(lo, hi, seed=1, out_scale=0.5).eval(pts[:100003])
    for n in (1, 64, 65, 100003, 63, 2500001, 3, 100003):
        got = net.eval(pts[:n])
        assert got.shape == (n, 4)
        m = min(n, 100003)
        assert np.array_equal(got[:m], want[:m]), n
    # the last points of the largest call, from their own call
    assert np.array_equal(net.eval(pts)[-1000:], net.eval(pts[-1000:]))
