"""The element launches of small segments (FP64: one Gauss point per wavefront;
FP32: several segments in one launch): runs against the oracle at the edges of
their 64-element blocks and the 63-element form behind a shadow lane, for every
law, both precisions and every force layout, and several laws in one launch."""
import numpy as np
import pytest

import femtech_amd as ft
from conftest import rel
from femtech_amd import workloads as W
from oracle import oracle as O

pytestmark = pytest.mark.gpu

MU, LAM = 2.0e4, 2.0e5
ROWS = {1: W.props_row(1000.0, MU, LAM), 2: W.props_row(1000.0, MU, LAM), 3: W.props_row(1000.0, MU, LAM),
        4: W.props_row(1000.0, MU, LAM, 3e4, 8.0), 5: W.props_row(1000.0, MU, LAM, 3e4, 8.0, 0.4, 2e-3, 0.3, 2e-2),
        6: W.props_row(1000.0, MU, LAM, -4.4), 7: W.props_row(1000.0, MU, LAM, 3.0, 0.0, 0.5, 2e-3, 0.3, 2e-2),
        8: W.props_row(1000.0, MU, LAM, 3e4, 8.0, 0.1), 0: W.props_row(1000.0, MU, LAM)}


def problem(dims, mats, permute, seed):
    X, conn = ft.mesh_block(*dims, 1e-3, jitter=0.15, seed=seed)
    ne = conn.size // 8
    if permute:
        conn = W.permute_elements(conn, seed)
    pid = (np.arange(ne) * len(mats) // ne).astype(np.int32)
    Xr = X.reshape(-1, 3)
    dm = -np.ones(X.size, np.int32)
    base = np.nonzero(Xr[:, 2] < 1e-9)[0]
    for d in range(3):
        dm[3 * base + d] = 0
    z = Xr[:, 2] / Xr[:, 2].max()
    v0 = np.zeros(X.size)
    v0[0::3] = np.sin(0.5 * np.pi * z)
    v0[2::3] = -0.4 * z
    fib = np.random.default_rng(seed).normal(size=(ne, 3))
    fib /= np.linalg.norm(fib, axis=1)[:, None]
    return X, conn, pid, np.array(mats, np.int32), np.stack([ROWS[m] for m in mats]), dm, v0, fib


def compare(dims, mats, fp32, layout=ft.LAYOUT_AUTO, permute=False, steps=40, seed=5):
    X, conn, pid, mat, props, dm, v0, fib = problem(dims, mats, permute, seed)
    motions = ft.motion(ft.MOTION_FIXED)[None, :]
    with ft.Engine(X, conn, pid, mat, props, ft.FT_FP32 if fp32 else ft.FT_FP64) as e:
        e.set_layout(layout)
        e.set_boundary(dm, motions)
        e.set_fibres(fib.reshape(-1))
        m = e.lumped_mass()
        f = e.get_force(1e-4 * v0, 1e-5)
        dt = e.stable_time_step(1e-4 * v0)
        e.reset_history()
        e.set_state(None, v0)
        e.run_init(1e9, 0.9, 1e-11)
        assert e.run_steps(steps) == steps
        u, v, a, fi = e.state()
        t = e.time()
        hist = e.visco_history()
        assert e.status() == 0
    o = O.Model(X, conn, pid, mat, props)
    o.set_fibres(fib)
    fo = o.get_force(1e-4 * v0, 1e-5)
    assert rel(f, fo) < (1e-4 if fp32 else 1e-10)  # strains of 1e-4: FP32 round-off relative to the strain
    o2 = O.Model(X, conn, pid, mat, props)
    o2.set_fibres(fib)
    o2.set_bc(dm, motions)
    o2.set_initial(None, v0)
    r = o2.run(steps, 1e9, 0.9, 1e-11)
    assert dt == pytest.approx(o2.stable_dt(1e-4 * v0, (dm >= 0).astype(np.int32)), rel=1e-12)
    # the step size comes from FP64 geometry in both precisions; the FP32 engine's displacement tolerance
    assert t[0] == pytest.approx(r["time"][-1], rel=1e-6 if fp32 else 1e-12)
    assert rel(u, r["u"]) < (1e-5 if fp32 else 1e-10)
    assert rel(v, r["v"]) < (1e-4 if fp32 else 1e-9)
    if 5 in mats or 7 in mats:
        ho = o2.history().reshape(-1, 8, 3, 9)[..., [0, 4, 8, 7, 6, 3]].reshape(-1)
        assert np.abs(hist.reshape(-1) - ho).max() <= (1e-4 if fp32 else 1e-9) * np.abs(ho).max()
    return m


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("mat", [1, 2, 3, 4, 5, 6, 7, 8])
@pytest.mark.parametrize("dims", [(9, 7, 1), (8, 8, 1), (13, 5, 1), (9, 7, 4)])
def test_one_law(gpu_ready, dims, mat, fp32):
    """63, 64, 65 and 252 elements: the last lane of a block, one beyond, whole tiles of 63."""
    compare(dims, [mat], fp32)


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("layout,permute", [(ft.LAYOUT_CORNER_PAIRS, False), (ft.LAYOUT_CORNER, False),
                                            (ft.LAYOUT_NODE_SLOTS, False), (ft.LAYOUT_ELL, False),
                                            (ft.LAYOUT_NODE_SLOTS, True), (ft.LAYOUT_ELL, True)])
def test_laws_in_one_launch(gpu_ready, layout, permute, fp32):
    """Eight laws and rigid elements over the parts of a ragged mesh, in one launch."""
    compare((11, 9, 17), [1, 2, 3, 4, 5, 6, 7, 8, 0], fp32, layout, permute)


def test_smallest_mesh(gpu_ready):
    compare((1, 1, 2), [1], False, steps=8)  # (the column inverts later, in the oracle as well)


@pytest.mark.parametrize("precision", [ft.FT_FP32, ft.FT_FP64])
def test_large_and_small_segments(gpu_ready, precision):
    """A segment beyond the small launches' range between two within it."""
    X, conn, pid, mat, props, dm, v0, fib = problem((72, 64, 64), [1, 2, 3], False, 3)
    ne = pid.size
    pid[:] = 1
    pid[:900] = 0
    pid[-1500:] = 2
    motions = ft.motion(ft.MOTION_FIXED)[None, :]
    with ft.Engine(X, conn, pid, mat, props, precision) as e:
        e.set_boundary(dm, motions)
        e.set_state(None, v0)
        e.lumped_mass()
        e.run_init(1e9, 0.9, 1e-11)
        assert e.run_steps(12) == 12
        u = e.state()[0]
    o = O.Model(X, conn, pid, mat, props, threads=8)
    o.set_bc(dm, motions)
    o.set_initial(None, v0)
    r = o.run(12, 1e9, 0.9, 1e-11)
    assert ne == 72 * 64 * 64 and rel(u, r["u"]) < (1e-5 if precision == ft.FT_FP32 else 1e-10)
