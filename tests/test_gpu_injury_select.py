"""The percentile search of the injury criteria (MPS-95, MPSxSR-95 and their
element lists) against the oracle at the sizes where its blocks and ranks can
go wrong: one element, few, a block and its neighbours, many; with parts left
out, repeated values and a second update below the first maximum."""
import numpy as np
import pytest

import femtech_amd as ft
from femtech_amd import workloads as W
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(1, 1, 1), (5, 2, 2), (17, 5, 3), (16, 4, 4), (257, 1, 1), (29, 17, 13)])
@pytest.mark.parametrize("case", ["all", "part", "uniform", "none"])
def test_percentiles_match_the_oracle(gpu_ready, dims, case):
    X, conn = ft.mesh_block(*dims, 1e-3, jitter=0.1, seed=3)
    ne = conn.size // 8
    pid = (np.arange(ne) % 3 == 1).astype(np.int32)
    mat, props = np.array([1, 1], np.int32), np.stack([W.props_row(1000.0, 1e6, 1e7)] * 2)
    include = {"all": None, "uniform": None, "part": np.array([0, 1], np.int32), "none": np.zeros(2, np.int32)}[case]
    rng = np.random.default_rng(1)
    if case == "uniform":  # every element strained alike, up to round-off (distinct stretches: with two equal ones
        # the oracle's principal values, as the reference's, can be NaN)
        shapes = [np.array([0.2, -0.05, -0.02]) * X.reshape(-1, 3)] * 3
    else:
        shapes = [s * rng.normal(size=(X.size // 3, 3)) * 1e-4 for s in (0.5, 1.5, 0.2)]
    o = O.Model(X, conn, pid, mat, props)
    o.injury_init(include)
    with ft.Engine(X, conn, pid, mat, props) as e:
        e.injury_enable(include)
        for k, u in enumerate(shapes):
            e.injury_update(u.reshape(-1), 1e-4 * (k + 1), 1e-4)
            o.injury_update(u.reshape(-1), 1e-4 * (k + 1), 1e-4)
        out, flags = e.injury_results()
    ro, fo = o.injury_results()
    np.testing.assert_allclose(out[12:16], ro[12:16], rtol=1e-9, atol=1e-15)
    np.testing.assert_allclose(out[[0, 2, 3, 5, 6, 8, 9, 11]], ro[[0, 2, 3, 5, 6, 8, 9, 11]], rtol=1e-9, atol=1e-15)
    if case != "uniform":  # (alike up to round-off: the lists follow the last bits)
        assert np.array_equal(flags, fo)
