"""The autotuner on segments that share an element launch: it leaves them in it
where that is the faster side, so tuning does not take it apart."""
import numpy as np
import pytest

import femtech_amd as ft
from femtech_amd import workloads as W
from test_gpu_merge_rule import problem

pytestmark = pytest.mark.gpu


def engine(sizes, precision):
    X, conn, pid, mat, props, dm, v0 = problem(sizes)
    e = ft.Engine(X, conn, pid, mat, props, precision)
    e.set_boundary(dm, ft.motion(ft.MOTION_FIXED)[None, :])
    e.set_state(None, v0)
    e.lumped_mass()
    e.run_init(1e9, 0.9, 1e-11)
    return e


def launches(e, steps=4):
    e.set_timing(1)
    assert e.run_steps(steps) == steps
    n = e.timing()[1][0] / steps
    e.set_timing(0)
    return n


@pytest.mark.parametrize("precision", [ft.FT_FP32, ft.FT_FP64])
@pytest.mark.parametrize("shaped", [False, True])
def test_small_segments_stay_together(gpu_ready, precision, shaped):
    """Five laws of 6,000 elements: one launch takes a third of five and less,
    before and after tuning, also where a segment had a shape of its own."""
    sizes = {m: 6000 for m in (1, 2, 3, 4, 5)}
    with engine(sizes, precision) as e, engine(sizes, precision) as plain:
        assert launches(plain) == 1
        if shaped:
            e.set_segment_shape(2, 3 if precision == ft.FT_FP32 else 0, 64)
        rep = e.autotune(3)
        seg = e.segments()
        assert np.all(seg[:, 3] == 0) and np.all(seg[:, 4] == 256)
        assert np.array_equal(rep[:, 2], seg[:, 3]) and np.array_equal(rep[:, 3], seg[:, 4])
        assert np.all(rep[:, 4] == rep[0, 4]) and np.all(rep[:, 5] == rep[:, 4]) and rep[0, 4] > 0
        assert launches(e) == 1
        assert all(np.array_equal(a, b) for a, b in zip(e.state(), plain.state()))


@pytest.mark.parametrize("precision", [ft.FT_FP32, ft.FT_FP64])
def test_a_large_segment_is_tuned_by_itself(gpu_ready, precision):
    with engine({1: 2000, 2: 2000, 4: 200000 if precision == ft.FT_FP64 else 280000}, precision) as e:
        n = launches(e)
        rep = e.autotune(2)
        seg = e.segments()
        assert np.all(seg[:2, 3] == 0) and np.all(seg[:2, 4] == 256)
        assert 0 < rep[2, 4] <= rep[2, 5] and rep[0, 4] == rep[1, 4] > 0
        assert launches(e) == n == 2
