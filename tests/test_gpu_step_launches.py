"""Launches that a step shares: the surrogate laws' one element launch against
launches of their own, and the motion states and corner-pair extras of batches
with more node tiles than the tiles evaluate by themselves."""
import numpy as np
import pytest

import femtech_amd as ft
from femtech_amd import workloads as W

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


def run_surrogate(w, box, tiles, steps=20):
    """(u, stats, Gauss points of the surrogate laws); box None: the plain run."""
    with ft.Engine(w["X"], w["conn"], w["pid"], w["material_id"], w["props"], ft.FT_FP32) as e, ft.Mlp(seed=4) as net:
        e.set_fibres(w["fibres"])
        e.set_boundary(w["dof_motion"], w["motions"])
        segs = e.segments()
        for k, s in enumerate(segs):
            if s[0] in tiles:
                e.set_segment_shape(k, 0, tiles[s[0]])
        e.lumped_mass()
        e.run_init(1e9, 0.9, 1e-11)
        if box is not None:
            norm = np.zeros(80, np.float32)
            norm[16:32], norm[72:80] = 1.0, 100.0
            norm[32:48], norm[48:64] = -box, box
            e.surrogate_set(net.params(), norm)
            e.surrogate_enable(True, 1000, 1)
        assert e.run_steps(steps) == steps
        stats = e.surrogate_stats() if box is not None else None
        return e.state()[0], stats, 8 * sum(int(s[2] - s[1]) for s in segs if s[0] in (7, 8))


@pytest.mark.parametrize("laws", ["both", "only 7", "only 8"])
@pytest.mark.parametrize("tiles", [{}, {7: 64, 8: 64}, {8: 64}, {7: 128}])
def test_surrogate_laws_share_launches(gpu_ready, laws, tiles):
    """Every surrogate Gauss point of both laws is evaluated once per step,
    whatever the tile sizes.  With an empty box all take the analytic law: the
    plain run up to FP32 round-off (20 steps of 24-term force sums: 5e-5);
    with an endless one the tile sizes change round-off only."""
    w = W.ellipsoid_head(n=13, peak=7.0e4, duration=2.0e-3)
    if laws != "both":
        core = w["pid"] > 0
        w["pid"][core] = 1 if laws == "only 7" else 2
    plain, _, _ = run_surrogate(w, None, {})
    u, st, n = run_surrogate(w, -1.0, tiles)
    assert n > 0 and st[4] == 20 * n and st[2] == 1.0
    assert rel(u, plain) < 5e-5
    u0, s0, _ = run_surrogate(w, 1e30, {})
    u1, s1, _ = run_surrogate(w, 1e30, tiles)
    assert s0[2] == s1[2] == 0.0 and s1[4] == 20 * n
    assert rel(u1, u0) < 5e-5


@pytest.mark.parametrize("precision", [ft.FT_FP64, ft.FT_FP32])
def test_many_node_tiles_match_few(gpu_ready, precision):
    """1,030 instances (a node tile each at least: motion states and extras in
    one launch before the node update) against the first six of them alone
    (motion states in the node tiles): round-off of 30 steps."""
    base = [W.ellipsoid_head(n=6, peak=4e5, duration=2e-3), W.ellipsoid_head(n=5, peak=2e5, duration=3e-3),
            W.impact_block(n=3, slab=1, seed=11)]

    def run(count):
        m, no, eo = W.concatenate([base[i % 3] for i in range(count)])
        with ft.Engine(m["X"], m["conn"], m["pid"], m["material_id"], m["props"], precision) as e:
            e.set_instances(no, eo)
            e.set_fibres(m["fibres"])
            e.set_boundary(m["dof_motion"], m["motions"])
            e.set_state(None, m["v0"])
            e.lumped_mass()
            e.run_init(1e9, 0.9, 1e-11)
            e.run_steps(30)
            return e.state()[0][:3 * no[6]], np.stack([e.instance(i) for i in range(6)])

    u0, i0 = run(6)
    u1, i1 = run(1030)
    tol = 1e-10 if precision == ft.FT_FP64 else 1e-5
    assert rel(u1, u0) < tol
    np.testing.assert_allclose(i1[:, :3], i0[:, :3], rtol=1e-6 if precision == ft.FT_FP32 else 1e-10)
