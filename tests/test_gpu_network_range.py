"""The training kernels' SiLU over FP32's whole range: pre-activations far
below zero, where value and derivative are tiny but not zero, and infinite
ones."""
import numpy as np
import pytest

import femtech_amd as ft
from oracle import mlp as M

pytestmark = pytest.mark.gpu


def network(z):
    """Layer 1's pre-activations are `z` (its weights are zero); the other
    weights and biases are of order one and positive."""
    rng = np.random.default_rng(7)
    p = rng.uniform(0.05, 0.3, M.N_PARAMS)
    p[M.W_OFF[1]:M.B_OFF[1]] = 0.0
    p[M.B_OFF[1]:M.B_OFF[1] + M.HID] = z
    return p.astype(np.float32)


def data(n):
    rng = np.random.default_rng(8)
    x, t = rng.normal(size=(n, 16)).astype(np.float32), rng.normal(size=(n, 8)).astype(np.float32)
    x[:, 12:] = 0.0
    t[:, 6:] = 0.0
    return x, t


def weights(g, l):
    return g[M.W_OFF[l]:M.B_OFF[l]].astype(np.float64)


@pytest.mark.parametrize("z", [-30.0, -43.0, -46.0, -60.0, -75.0, -84.0, -88.0])
def test_far_below_zero(gpu_ready, z):
    """dW of layer 2 is its dZ times SiLU(z), dW and db of layer 1 are that
    layer's dA times SiLU'(z): each of z's size, e^z, against FP64.  Bar: the
    gradients' (1.5e-3) plus e^-z's relative error, half an ulp of z."""
    x, t = data(64)
    p = network(z)
    with ft.Mlp(seed=1) as net:
        net.set_params(p)
        loss, g = net.gradients(x, t)
    lref, gref = M.loss_and_grad(p.astype(np.float64), x, t)
    assert abs(loss / lref - 1) < 1e-4
    tol = 1.5e-3 + abs(z) * 2.0**-23
    for a, b in ((weights(g, 2), weights(gref, 2)), (weights(g, 1), weights(gref, 1)),
                 (g[M.B_OFF[1]:M.W_OFF[2]].astype(np.float64), gref[M.B_OFF[1]:M.W_OFF[2]])):
        scale = np.abs(b).max()
        assert scale > 0 and np.linalg.norm((a - b) / scale) <= tol * np.linalg.norm(b / scale)


@pytest.mark.parametrize("z", [-89.0, -200.0, -np.inf])
def test_beyond_the_exponential(gpu_ready, z):
    """e^-z overflows: the value is -0 (not a number at -inf, as z / (1 + e^-z) is)."""
    x, t = data(32)
    with ft.Mlp(seed=1) as net:
        net.set_params(network(z))
        loss, g = net.gradients(x, t)
    if np.isinf(z):
        assert np.isnan(loss)
    else:
        assert np.isfinite(loss) and np.all(weights(g, 2) == 0) and np.all(weights(g, 1) == 0)


def test_infinite_pre_activation(gpu_ready):
    """SiLU(+inf) = +inf: positive weights behind it carry it to the loss."""
    x, t = data(32)
    with ft.Mlp(seed=1) as net:
        net.set_params(network(np.inf))
        loss, _ = net.gradients(x, t)
    assert loss == np.inf
