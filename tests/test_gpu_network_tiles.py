"""Network gradients at the edges of the training kernel's 32-sample blocks."""
import numpy as np
import pytest

import femtech_amd as ft
from oracle import mlp as M
from test_gpu_network_sizes import data, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [31, 32, 33, 64, 65, 95, 97])
def test_gradients_at_tile_edges(gpu_ready, n):
    """Bars of the block-edge test of the larger counts: 1e-5 on the loss and
    1.5e-3 on a gradient, plus one activation rounded to the other BF16
    neighbour (2^-8 of itself, over n samples)."""
    x, t = data(n, 140 + n)
    with ft.Mlp(seed=6) as net:
        p = net.params().astype(np.float64)
        loss, g = net.gradients(x, t)
    lref, gref = M.loss_and_grad(p, x, t)
    assert abs(loss / lref - 1) < 1e-5 + 2.0**-8 / n
    for l in range(M.LAYERS):
        for part in (slice(M.W_OFF[l], M.B_OFF[l]), slice(M.B_OFF[l], M.B_OFF[l] + M.layer_out(l))):
            assert rel(g[part], gref[part]) < 1.5e-3 + 2.0**-8 / n, (l, part, rel(g[part], gref[part]))


@pytest.mark.parametrize("batch", [31, 32, 33])
def test_padding_samples_count_for_nothing(gpu_ready, batch):
    """A step over copies of one sample is that sample's, whatever the block holds beyond the batch."""
    x, t = data(1, 3)
    with ft.Mlp(seed=8) as net:
        one = net.gradients(x, t)
        many = net.gradients(np.repeat(x, batch, axis=0), np.repeat(t, batch, axis=0))
    assert many[0] == pytest.approx(one[0], rel=1e-6)
    assert rel(many[1], one[1].astype(np.float64)) < 2.0**-8  # dZ / n rounds to BF16 elsewhere for each n
