"""ft_get_state with some of its arrays, or none (which waits for the engine's
queued work, as every read-back does)."""
import ctypes

import numpy as np
import pytest

import femtech_amd as ft
from femtech_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [6, 26, 36])  # pinned and pageable copies, host and device transposition
def test_any_of_the_arrays_may_be_null(gpu_ready, n):
    w = W.impact_block(n=n, slab=1, seed=4)
    with ft.Engine(w["X"], w["conn"], w["pid"], w["material_id"], w["props"], ft.FT_FP64) as e:
        e.set_boundary(w["dof_motion"], w["motions"])
        e.set_state(None, w["v0"])
        e.lumped_mass()
        e.run_init(1e9, 0.9, 1e-11)
        e.run_steps(5)
        full = e.state()
        for take in ([], [0], [1], [2], [3], [2, 3], [0, 1, 2]):
            out = [np.full(full[0].size, 7.0) for _ in range(4)]
            p = [out[k].ctypes.data_as(ctypes.POINTER(ctypes.c_double)) if k in take else None for k in range(4)]
            assert e._lib.ft_get_state(e._h, *p) == 0
            for k in range(4):
                assert np.array_equal(out[k], full[k]) if k in take else np.all(out[k] == 7.0)
        # whatever was read, the state is the same
        assert all(np.array_equal(x, y) for x, y in zip(full, e.state()))
