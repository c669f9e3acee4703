"""Which FP32 segments share an element launch in the run loop, on both sides of
the rule's sizes, and that runs on either side follow the oracle."""
import numpy as np
import pytest

import femtech_amd as ft
from conftest import rel
from femtech_amd import workloads as W
from oracle import oracle as O
from test_gpu_small_segments import ROWS

pytestmark = pytest.mark.gpu


def problem(sizes, seed=3):
    """A block whose elements are law 1's, then 2's, ...: sizes {law: count},
    the largest taking what the block has over."""
    total = sum(sizes.values())
    n = round(total ** (1 / 3))
    X, conn = ft.mesh_block(n, n, -(-total // (n * n)), 1e-3, jitter=0.15, seed=seed)
    ne = conn.size // 8
    big = max(sizes, key=sizes.get)
    pid = np.full(ne, list(sizes).index(big), np.int32)
    k = 0
    for j, (mat, count) in enumerate(sizes.items()):
        count += (ne - total) * (mat == big)
        pid[k:k + count] = j
        k += count
    Xr = X.reshape(-1, 3)
    dm = -np.ones(X.size, np.int32)
    base = np.nonzero(Xr[:, 2] < 1e-9)[0]
    for d in range(3):
        dm[3 * base + d] = 0
    z = Xr[:, 2] / Xr[:, 2].max()
    v0 = np.zeros(X.size)
    v0[0::3], v0[2::3] = np.sin(0.5 * np.pi * z), -0.4 * z
    mats = list(sizes)
    return X, conn, pid, np.array(mats, np.int32), np.stack([ROWS[m] for m in mats]), dm, v0


def run(sizes, steps):
    """Element launches per step, the problem and its displacement."""
    p = X, conn, pid, mat, props, dm, v0 = problem(sizes)
    with ft.Engine(X, conn, pid, mat, props, ft.FT_FP32) as e:
        e.set_boundary(dm, ft.motion(ft.MOTION_FIXED)[None, :])
        e.set_state(None, v0)
        e.lumped_mass()
        e.run_init(1e9, 0.9, 1e-11)
        e.set_timing(1)
        assert e.run_steps(steps) == steps
        launches = e.timing()[1][0] / steps
        return launches, p, e.state()[0]


@pytest.mark.parametrize("sizes,launches", [
    ({1: 2000, 2: 130000}, 1),
    ({1: 5000, 2: 176000}, 2),   # a second round of blocks at two wavefronts per SIMD for one launch's latency
    ({2: 176000, 8: 5000}, 2),
    ({1: 2000, 2: 100000, 3: 100000}, 1),
    ({1: 60000, 2: 60000, 3: 60000, 4: 60000}, 1),
    ({1: 80000, 2: 80000, 3: 80000, 4: 80000}, 2),  # the first three, within 250,000, then one
])
def test_launches(gpu_ready, sizes, launches):
    assert run(sizes, 3)[0] == launches


@pytest.mark.parametrize("sizes,launches", [
    ({1: 160000, 2: 900, 4: 1500}, 1),       # one run of three laws of very uneven size
    ({1: 300000, 2: 900, 4: 1500}, 2),       # a large segment first: the shared launch starts at a later tile
    ({1: 900, 2: 1500, 4: 300000}, 2),       # ... and last
    ({1: 900, 2: 300000, 4: 1500}, 3),       # none: the large one lies between the small ones
])
def test_runs_beside_a_large_segment(gpu_ready, sizes, launches):
    """Shared launches beside a segment's own, against the oracle (the FP32
    engine's displacement bar)."""
    n, (X, conn, pid, mat, props, dm, v0), u = run(sizes, 12)
    assert n == launches
    o = O.Model(X, conn, pid, mat, props, threads=8)
    o.set_bc(dm, ft.motion(ft.MOTION_FIXED)[None, :])
    o.set_initial(None, v0)
    assert rel(u, o.run(12, 1e9, 0.9, 1e-11)["u"]) < 1e-5
