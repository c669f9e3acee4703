"""Network training kernels at the sizes where their blocks can go wrong (one
sample, a block of 128 samples and its neighbours, a gradient chunk of 256 and
its neighbours), and what a training step leaves behind."""
import numpy as np
import pytest

import femtech_amd as ft
from oracle import mlp as M

pytestmark = pytest.mark.gpu


def data(n, seed):
    rng = np.random.default_rng(seed)
    x, t = rng.normal(size=(n, 16)).astype(np.float32), rng.normal(size=(n, 8)).astype(np.float32)
    x[:, 12:] = 0.0
    t[:, 6:] = 0.0
    return x, t


def rel(a, b):
    return float(np.linalg.norm(np.asarray(a, np.float64) - b) / max(np.linalg.norm(b), 1e-300))


@pytest.mark.parametrize("n", [1, 2, 63, 127, 128, 129, 255, 257, 511, 513, 1025])
def test_gradients_at_block_edges(gpu_ready, n):
    """Bars of the larger batches (1e-5 on the loss, 1.5e-3 on a gradient)
    plus one activation rounded to the other BF16 neighbour, 2^-8 of itself,
    which a mean over few samples does not average out."""
    x, t = data(n, 40 + n)
    with ft.Mlp(seed=6) as net:
        p = net.params().astype(np.float64)
        loss, g = net.gradients(x, t)
        again = net.gradients(x, t)
    assert again[0] == loss and np.array_equal(again[1], g)  # fixed sum order
    lref, gref = M.loss_and_grad(p, x, t)
    assert abs(loss / lref - 1) < 1e-5 + 2.0**-8 / n
    for l in range(M.LAYERS):
        for part in (slice(M.W_OFF[l], M.B_OFF[l]), slice(M.B_OFF[l], M.B_OFF[l] + M.layer_out(l))):
            assert rel(g[part], gref[part]) < 1.5e-3 + 2.0**-8 / n, (l, part, rel(g[part], gref[part]))


@pytest.mark.parametrize("batch", [1, 127, 129, 256, 300])
def test_one_step_moves_every_parameter_by_its_gradient(gpu_ready, batch):
    """Adam's first step moves a parameter by lr g / (|g| + eps): by lr in the
    direction against g where |g| is well above eps.  The data hold one sample,
    so a batch's mean gradient is that sample's.  The network that the step
    leaves is the one its parameters make."""
    x, t = data(1, 3)
    lr = 1e-3
    with ft.Mlp(seed=8) as net, ft.Mlp(seed=9) as copy:
        p0 = net.params()
        net.train(x, t, steps=1, batch=batch, lr=lr, seed=1)
        p1 = net.params()
        xs, _ = data(300, 5)
        y = net.forward(xs)
        copy.set_params(p1)
        assert np.array_equal(y, copy.forward(xs))
        gx, gt = np.repeat(x, batch, axis=0), np.repeat(t, batch, axis=0)
        after = net.gradients(gx, gt)
        same = copy.gradients(gx, gt)
        assert after[0] == same[0] and np.array_equal(after[1], same[1])
    _, g = M.loss_and_grad(p0.astype(np.float64), x, t)
    big = np.abs(g) > 1e-2 * np.abs(g).max()
    assert big.sum() > 500
    # the step itself, FP32 round-off of p (|p| < 2: 1.2e-7) and eps / |g|
    np.testing.assert_allclose((p1 - p0)[big], -lr * np.sign(g[big]), atol=2.4e-7 + lr * 1e-3)
