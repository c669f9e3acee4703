"""Calls whose device allocation fails (more than the card holds) report it and
leave nothing behind: the next call works, and as if the failed one had not been."""
import numpy as np
import pytest

import femtech_amd as ft
from femtech_amd import workloads as W

pytestmark = pytest.mark.gpu


def test_network_after_a_failed_step(gpu_ready):
    """A batch of 2^30 samples needs 1.1 TB of activations."""
    rng = np.random.default_rng(1)
    x, t = rng.normal(size=(2000, 16)).astype(np.float32), rng.normal(size=(2000, 8)).astype(np.float32)
    with ft.Mlp(seed=3) as net:
        y, g = net.forward(x), net.gradients(x, t)
        with pytest.raises(ft.FemTechError):
            net.train(x, t, steps=3, batch=2**30)
        assert np.array_equal(net.forward(x), y)
        again = net.gradients(x, t)
        assert again[0] == g[0] and np.array_equal(again[1], g[1])


def test_training_after_a_failed_step(gpu_ready):
    """Adam's step count (its bias corrections) does not move with a step that
    never ran."""
    rng = np.random.default_rng(1)
    x, t = rng.normal(size=(2000, 16)).astype(np.float32), rng.normal(size=(2000, 8)).astype(np.float32)
    out = []
    for failed in (False, True):
        with ft.Mlp(seed=3) as net:
            if failed:
                p = net.params()
                with pytest.raises(ft.FemTechError):
                    net.train(x, t, steps=3, batch=2**30)
                assert np.array_equal(net.params(), p)
            net.train(x, t, steps=20, batch=512)
            out.append(net.params())
    assert np.array_equal(*out)


def test_engine_after_a_failed_reserve(gpu_ready):
    w = W.impact_block(n=4, slab=1, seed=1)
    u = 1e-6 * np.random.default_rng(2).normal(size=w["X"].size)
    with ft.Engine(w["X"], w["conn"], w["pid"], w["material_id"], w["props"], ft.FT_FP64) as e:
        f = e.get_force(u, 1e-7)
        with pytest.raises(ft.FemTechError) as ei:
            e.surrogate_reserve(10**11)
        assert ei.value.code == 12
        assert np.array_equal(e.get_force(u, 1e-7), f)
