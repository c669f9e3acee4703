"""The surrogate's audit tallies when the element tiles change after they were
made: one row per tile, so smaller tiles or another force layout need more."""
import numpy as np
import pytest

import femtech_amd as ft
from femtech_amd import workloads as W

pytestmark = pytest.mark.gpu


def engine():
    w = W.ellipsoid_head(n=12, peak=7e4, duration=2e-3)
    e = ft.Engine(w["X"], w["conn"], w["pid"], w["material_id"], w["props"], ft.FT_FP32)
    e.set_fibres(w["fibres"])
    e.set_boundary(w["dof_motion"], w["motions"])
    e.lumped_mass()
    return e


def enable(e):
    # no input lies in the empty training box: every evaluation falls back, so the counts are known
    norm = np.zeros(80, np.float32)
    norm[16:32] = norm[72:80] = 1.0
    norm[32:48] = 1e30
    e.surrogate_set(np.zeros(52744, np.float32), norm)
    e.surrogate_enable(True, 2, 1000)


def points(e):
    return 8 * sum(b - a for mat, a, b, _, _ in e.segments() if mat in (7, 8))


@pytest.mark.parametrize("change", ["shape", "layout", "autotune"])
def test_tallies_follow_the_tiles(gpu_ready, change):
    """The counts of the steps before and after the change, as many as the
    segments' Gauss points each."""
    with engine() as e:
        if change == "layout":  # corner pairs take 63 elements to a wavefront, node slots 64
            e.set_layout(ft.LAYOUT_NODE_SLOTS)
        enable(e)
        steps = 0
        if change != "layout":
            e.run_init(1e9, 0.9, 1e-11)
            steps += e.run_steps(3)
        if change == "shape":
            for s in range(len(e.segments())):
                e.set_segment_shape(s, 0, 64)
        elif change == "layout":
            e.set_layout(ft.LAYOUT_CORNER_PAIRS)
            for s in range(len(e.segments())):
                e.set_segment_shape(s, 0, 64)
        else:
            e.autotune(1)  # tries tiles of 64, 128 and 256 elements
        if change == "layout":
            e.run_init(1e9, 0.9, 1e-11)
        steps += e.run_steps(4)
        st = e.surrogate_stats()
        assert steps in (4, 7) and st[4] == st[5] == steps * points(e)
        assert np.all(np.isfinite(st))


def test_growth_leaves_the_run_as_it_is(gpu_ready):
    """Tiles of 64 set before the surrogate was enabled, or after: the same
    tiles, so the same run and the same tallies."""
    out = []
    for before in (True, False):
        with engine() as e:
            if not before:
                enable(e)
            for s in range(len(e.segments())):
                e.set_segment_shape(s, 0, 64)
            if before:
                enable(e)
            e.run_init(1e9, 0.9, 1e-11)
            assert e.run_steps(6) == 6
            out.append((e.state(), e.surrogate_stats()))
    (a, sa), (b, sb) = out
    assert all(np.array_equal(x, y) for x, y in zip(a, b)) and np.array_equal(sa, sb)
