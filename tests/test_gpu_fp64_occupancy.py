"""The FP64 element kernels of the two HGO laws on both sides of one wavefront
per SIMD (1,024 wavefronts of 63 elements, or 64 without corner pairs), where
another instance of the kernel takes over: forces and step size against the
oracle."""
import numpy as np
import pytest

import femtech_amd as ft
from conftest import rel
from oracle import oracle as O
from test_gpu_small_segments import problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layout", [ft.LAYOUT_CORNER_PAIRS, ft.LAYOUT_CORNER])
@pytest.mark.parametrize("mat", [4, 8])
@pytest.mark.parametrize("dims", [(63, 64, 16), (64, 64, 16), (41, 40, 40)])  # 64,512, 65,536 and 65,600 elements
def test_both_sides(gpu_ready, dims, mat, layout):
    X, conn, pid, mats, props, dm, v0, fib = problem(dims, [mat], False, 2)
    u = 1e-4 * v0
    with ft.Engine(X, conn, pid, mats, props, ft.FT_FP64) as e:
        e.set_layout(layout)
        e.set_boundary(dm, ft.motion(ft.MOTION_FIXED)[None, :])
        e.set_fibres(fib.reshape(-1))
        f = e.get_force(u, 1e-5)
        e.set_state(None, v0)
        e.lumped_mass()
        e.run_init(1e9, 0.9, 1e-11)
        assert e.run_steps(6) == 6
        ur, t = e.state()[0], e.time()
    o = O.Model(X, conn, pid, mats, props, threads=8)
    o.set_fibres(fib)
    o.set_bc(dm, ft.motion(ft.MOTION_FIXED)[None, :])
    assert rel(f, o.get_force(u, 1e-5)) < 1e-10
    o.set_initial(None, v0)
    r = o.run(6, 1e9, 0.9, 1e-11)
    assert rel(ur, r["u"]) < 1e-10 and t[0] == pytest.approx(r["time"][-1], rel=1e-12)
