"""Nodal arrays to and from the device on both sides of the node counts at
which their path changes (host or device transposition, pinned buffer or the
caller's pages), and the constrained DOFs at the start of a run."""
import numpy as np
import pytest

import femtech_amd as ft
from femtech_amd import workloads as W
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx", [1, 4095, 4096, 10921, 10922, 20000])  # 4 (nx + 1) nodes
@pytest.mark.parametrize("precision", [ft.FT_FP64, ft.FT_FP32])
def test_state_round_trip_and_start(gpu_ready, nx, precision):
    X, conn = ft.mesh_block(nx, 1, 1, 1e-3, jitter=0.1, seed=2)
    nn, ne = X.size // 3, conn.size // 8
    rng = np.random.default_rng(nx)
    u, v = 1e-6 * rng.normal(size=3 * nn), rng.normal(size=3 * nn)
    dofs = rng.integers(0, 3 * nn, size=min(40, nn))
    dofs = np.unique(np.concatenate([dofs, [0, 3 * nn - 1]]))
    motions = np.stack([W.motion(W.MOTION_FIXED), W.motion(W.MOTION_LINEAR, 3.0)])
    dof_motion = np.full(3 * nn, -1, np.int32)
    dof_motion[dofs] = np.arange(dofs.size) % 2
    with ft.Engine(X, conn, np.zeros(ne, np.int32), np.array([1], np.int32),
                   W.props_row(1000.0, 1e6, 1e7)[None], precision) as e:
        e.set_boundary(dof_motion, motions)
        e.set_state(u, v)
        e.lumped_mass()
        s = e.state()
        assert np.array_equal(s[0], u) and np.array_equal(s[1], v)
        assert np.array_equal(e.get_force(u, 1e-7), e.get_force(None, 1e-7))
        e.run_init(1.0, 0.5, 0.0)
        s = e.state()
    free = np.ones(3 * nn, bool)
    free[dofs] = False
    assert np.array_equal(s[0][free], u[free]) and np.array_equal(s[1][free], v[free])
    for i in dofs:
        ub, vb, _ = O.motion_eval(motions[dof_motion[i]], X.reshape(-1, 3)[i // 3], 0.0)
        assert s[0][i] == pytest.approx(ub[i % 3], rel=1e-12, abs=1e-18)
        assert s[1][i] == pytest.approx(vb[i % 3], rel=1e-12, abs=1e-18)
