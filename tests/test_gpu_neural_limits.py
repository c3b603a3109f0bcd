"""SiLU of the learned boundary at its limits: a network whose weights are 0 but
for one unit of the last hidden layer, y = w4 silu(b3), evaluated at biases
where the sigmoid leaves the normal numbers, underflows to 0 and meets
infinities and NaN.  The exponential's relative error grows with its argument
(about 88 roundings there, 1e-5); quotients below the normal numbers are exact
to 2^-149, 6e-39 of them to 2e-7.  And the sigmoid against the correctly rounded
quotient over its range: silu(z) / z and the quotient of the same exponential
differ by their own roundings."""
import math

import numpy as np
import pytest

import cudasphnew_amd as S

pytestmark = pytest.mark.gpu

W4 = 2.0 ** 100
OB3 = 128 * 64 + 64 + 2 * (64 * 64) + 64      # b3 in the flat parameters
NPARAMS = OB3 + 64 + 64 + 1


def _silu(z):
    net = S.NeuralSDF([0.0] * 3, [1.0] * 3, seed=1, out_scale=1.0)
    p = np.zeros(NPARAMS, np.float32)
    p[OB3], p[OB3 + 64] = z, W4
    net.set_params(p)
    return float(net.eval(np.full((3, 3), 0.25, np.float32))[1, 0]) / W4


@pytest.mark.parametrize("z", [-1.0, -30.0, -87.0, -87.5, -88.0, -88.5])
def test_silu_below_the_normal_numbers(z):
    want = z / (1.0 + math.exp(-z))
    assert abs(_silu(z) - want) <= 1e-4 * abs(want) + 89 * 2.0 ** -149


@pytest.mark.parametrize("z", [-89.0, -100.0, -1e4, -3e38])
def test_silu_underflows_to_zero(z):
    assert abs(_silu(z)) <= 89 * 2.0 ** -149


def test_silu_of_infinities_and_nan():
    assert math.isnan(_silu(-math.inf))       # -inf * 0
    assert _silu(math.inf) == math.inf
    assert math.isnan(_silu(math.nan))
