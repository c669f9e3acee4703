"""Which FP64 segments share an element launch, on both sides of the rule's
sizes.  (The results are the same to the bit whichever they take.)"""
import pytest

import femtech_amd as ft
from test_gpu_merge_rule import problem

pytestmark = pytest.mark.gpu


def run(sizes, steps=3):
    X, conn, pid, mat, props, dm, v0 = problem(sizes)
    with ft.Engine(X, conn, pid, mat, props, ft.FT_FP64) as e:
        e.set_boundary(dm, ft.motion(ft.MOTION_FIXED)[None, :])
        e.set_state(None, v0)
        e.lumped_mass()
        e.run_init(1e9, 0.9, 1e-11)
        e.set_timing(1)
        assert e.run_steps(steps) == steps
        return e.timing()[1][0] / steps


@pytest.mark.parametrize("sizes,launches", [
    ({1: 2000, 2: 2000, 3: 2000}, 1),
    ({1: 24000, 2: 24000, 3: 24000}, 1),
    ({1: 58000, 2: 58000, 3: 58000}, 3),   # one launch of these takes 88 us, three of k_element 64
    ({1: 44000, 2: 44000}, 2),
    ({1: 70000, 2: 2000}, 2),
    ({5: 30000, 7: 30000}, 1),
    ({5: 58000, 7: 58000}, 2),
    ({1: 2000, 2: 2000, 3: 100000, 4: 2000, 5: 2000}, 3),  # two runs around a large segment
])
def test_launches(gpu_ready, sizes, launches):
    assert run(sizes) == launches
