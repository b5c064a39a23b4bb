"""The inference sigmoid against FP64.  With W2 = 0 and one non-zero output
weight of 1 the network returns z sigmoid(z) of one second-layer bias z, all
of it in FP32: 1 ulp of the exponential and half of one each for its sum with
1, the quotient and the product, 2.5 * 2^-23 of the value."""
import numpy as np
import pytest

from oracle import mlp as omlp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("unit", [0, 17, 63])
def test_sigmoid_error(sph, unit):
    net = sph.Mlp(seed=1)
    norm = np.zeros(sph.MLP_NORM, np.float32)
    norm[12:24] = norm[25] = 1
    x = np.ones((1, 12), np.float32)
    for z in np.r_[np.linspace(-60, 60, 61), -0.37, 1e-3, -17.3].astype(np.float32):
        p = np.zeros(sph.MLP_PARAMS, np.float32)
        p[omlp.OFF_B2 + unit] = z
        p[omlp.OFF_W3 + unit] = 1
        net.set(p, norm)
        want = np.float64(z) / (1 + np.exp(-np.float64(z)))
        got = np.float64(net.forward(x)[0])
        assert abs(got - want) <= 2.51 * 2.0 ** -23 * abs(want), z
