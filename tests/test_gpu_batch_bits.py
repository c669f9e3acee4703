"""FP64: an instance of a batch follows the run of the same mesh alone to the
bit, also where the batch's segments are large enough for another element kernel
than the mesh's own (one Gauss point per wavefront)."""
import numpy as np
import pytest

import femtech_amd as ft
from femtech_amd import workloads as W
from test_gpu_small_segments import problem

pytestmark = pytest.mark.gpu


def workload(dims, mats, permute=False):
    X, conn, pid, mat, props, dm, v0, fib = problem(dims, mats, permute, 5)
    return dict(X=X, conn=conn, pid=pid, material_id=mat, props=props, dof_motion=dm,
                motions=ft.motion(ft.MOTION_FIXED)[None, :], v0=v0, fibres=fib)


def run(w, inst, layout, steps=12):
    with ft.Engine(w["X"], w["conn"], w["pid"], w["material_id"], w["props"], ft.FT_FP64) as e:
        if inst:
            e.set_instances(*inst)
        e.set_layout(layout)
        e.set_fibres(w["fibres"].reshape(-1))
        e.set_boundary(w["dof_motion"], w["motions"])
        u = 3e-4 * w["v0"]
        f, dt = e.get_force(u, 1e-6), e.stable_time_step(u)
        e.reset_history()
        e.set_state(None, w["v0"])
        e.lumped_mass()
        e.run_init(1e9, 0.9, 1e-11)
        assert e.run_steps(steps) == steps
        return f, dt, e.state()


def compare(w, copies, layout=ft.LAYOUT_AUTO):
    m, no, eo = W.concatenate([w] * copies)
    f, dt, state = run(w, None, layout)
    fb, dtb, stateb = run(m, (no, eo), layout)
    assert dt == dtb
    for i in (0, copies // 2, copies - 1):
        part = slice(3 * no[i], 3 * no[i + 1])
        assert np.array_equal(f, fb[part])
        for a, b in zip(state, stateb):
            assert np.array_equal(a, b[part]), i


@pytest.mark.parametrize("layout", [ft.LAYOUT_CORNER_PAIRS, ft.LAYOUT_NODE_SLOTS])
@pytest.mark.parametrize("mat", [1, 2, 3, 4, 5, 6, 7, 8])
def test_one_law(gpu_ready, mat, layout):
    """8,000 elements alone (a small segment) and 128,000 (176,000 of the Ogden laws) in the batch."""
    compare(workload((20, 20, 20), [mat]), 22 if mat in (6, 7) else 16, layout)


@pytest.mark.parametrize("permute", [False, True])
def test_laws_together(gpu_ready, permute):
    """Three laws that share a launch alone and have one each in the batch."""
    compare(workload((24, 24, 24), [2, 6, 8], permute), 40)
