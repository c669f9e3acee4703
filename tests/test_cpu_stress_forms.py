"""The closed stress forms of the element kernels (first Piola form of the
neo-Hookean and HGO laws; Ogden's isochoric stress by power series and, for
strains beyond it, by principal directions) against the oracle, one element at
a time, from strains near round-off to large stretches and under finite
rotations."""
import numpy as np
import pytest

from oracle import oracle as O
from test_cpu_kernel_math import elem, km  # noqa: F401 (km is a fixture)

MU, LAM = 2.0e4, 2.0e5
FIBRE = np.array([0.6, -0.48, 0.64])


def props(mat, alpha):
    p = np.zeros(9)
    p[:3] = [1000.0, MU, LAM]
    if mat in (6, 7):
        p[3] = alpha
        if mat == 7:
            p[5:9] = [0.5, 2e-3, 0.3, 2e-2]
    if mat in (4, 5):
        p[3:5] = [3.0e4, 8.0]
    if mat == 8:
        p[3:6] = [3.0e4, 8.0, 0.1]
    return p


def check(km, mat, fp32, strain, angle, alpha=-4.4, seed=0):
    rng = np.random.default_rng(seed)
    x = 1e-3 * (np.array([[0, 0, 0], [1, 0, 0], [1, 1, 0], [0, 1, 0], [0, 0, 1], [1, 0, 1], [1, 1, 1], [0, 1, 1]])
                + 0.1 * rng.uniform(-1, 1, (8, 3)))
    c, s = np.cos(angle), np.sin(angle)
    R = np.array([[c, -s, 0], [s, c, 0], [0, 0, 1.0]])
    # a homogeneous stretch plus node-wise parts of a tenth of it, then the rotation
    G = np.diag([1.0, -0.4, -0.3]) + 0.3 * rng.uniform(-1, 1, (3, 3))
    y = x + strain * (x @ G.T + 1e-4 * rng.uniform(-1, 1, (8, 3)))
    u = (y @ R.T - x).reshape(24)
    p = props(mat, alpha)
    f, _, flags = elem(km, fp32, x.reshape(24), u, mat, p, hist=np.zeros(144), fibre=FIBRE)
    o = O.Model(x.reshape(24), np.arange(8, dtype=np.int32), np.zeros(1, np.int32), np.array([mat], np.int32), p)
    o.set_fibres(FIBRE)
    fo = o.element_forces(u, 1e-5)
    assert flags == 0
    # a force of relative size `strain` comes from displacement gradients of size strain + angle, each rounded in
    # the element type; the oracle forms F^T F - I, whose FP64 round-off is relative to 1
    tol = (32 * 2.0 ** -24 if fp32 else 64 * 2.0 ** -53) * (1 + (angle + (0 if fp32 else 1)) / strain)
    tol += 64 * 2.0 ** -53 / strain
    assert np.linalg.norm(f - fo) <= tol * np.linalg.norm(fo)


@pytest.mark.parametrize("fp32", [0, 1])
@pytest.mark.parametrize("mat", [1, 4, 6, 7, 8])
@pytest.mark.parametrize("strain,angle", [(1e-5, 0.0), (1e-3, 0.0), (1e-3, 0.3), (0.05, 2.0), (0.2, 0.5), (0.6, 1.0)])
def test_forms_over_strain_and_rotation(km, mat, fp32, strain, angle):  # noqa: F811
    check(km, mat, fp32, strain, angle)


@pytest.mark.parametrize("fp32", [0, 1])
@pytest.mark.parametrize("alpha", [2.0, 4.0, -2.0, 20.0, -20.0, 0.5])
@pytest.mark.parametrize("strain", [1e-4, 0.03, 0.12, 0.4, 0.8])
def test_ogden_exponents(km, request, fp32, alpha, strain):  # noqa: F811
    """Exponents whose series ends (positive even), converges slowly or is
    left for the principal directions."""
    if fp32 and alpha == -20.0 and strain == 0.8:
        # the stretches' FP32 round-off comes out multiplied by |alpha|, which the bound leaves out: 3.9e-6 here
        # with the principal directions alone too, against 2.1e-6
        request.applymarker(pytest.mark.xfail(strict=True, reason="condition |alpha| of the FP32 stretches"))
    check(km, 7, fp32, strain, 0.1, alpha, seed=3)
