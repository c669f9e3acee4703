"""The Ogden law's choice between its power series and the principal directions:
the rule that takes the series never takes one that does not end (its terms
would be paid for beside the directions), and both give the same stress."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from conftest import HERE

SRC = os.path.join(HERE, "native", "ogden_host.cpp")
OUT = os.path.join(HERE, "native", "_build", "libogden.so")
_D = ctypes.POINTER(ctypes.c_double)
TERMS = {0: 40, 1: 24}
EPS = {0: 2.0**-53, 1: 2.0**-24}


@pytest.fixture(scope="module")
def both():
    os.makedirs(os.path.dirname(OUT), exist_ok=True)
    subprocess.run(["/opt/rocm/bin/hipcc", "-O2", "-std=c++17", "-fPIC", "-shared", "-x", "c++",
                    "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", SRC, "-o", OUT], check=True)
    lib = ctypes.CDLL(OUT)
    lib.oh_both.argtypes = [ctypes.c_int, _D, ctypes.c_double, _D, _D]

    def call(fp32, z, alpha):
        z = np.ascontiguousarray(z, np.float64)
        m, v = np.zeros(6), np.zeros(6)
        r = lib.oh_both(fp32, z.ctypes.data_as(_D), alpha, m.ctypes.data_as(_D), v.ctypes.data_as(_D))
        return bool(r & 1), bool(r & 2), m, v

    return call


DIRECTIONS = [(1.0, -0.4, -0.55), (1.0, 1.0, -1.5), (0.3, 0.2, -0.6)]


@pytest.mark.parametrize("fp32", [0, 1])
@pytest.mark.parametrize("alpha", [-50.0, -20.0, -12.3, -8.0, -4.4, -2.0, -1.0, -0.1, 0.5, 1.3, 2.0, 3.0, 4.0, 5.0, 6.0,
                                   7.5, 8.0, 12.7, 20.0, 30.5, 41.0, 50.0])
def test_the_rule_takes_series_that_end(both, fp32, alpha):
    taken = 0
    for d in DIRECTIONS:
        d = np.array(d) / np.linalg.norm(d)
        for rho in np.concatenate([np.geomspace(1e-6, 0.05, 12), np.linspace(0.06, 1.0, 95)]):
            if rho * d.min() <= -1:  # no deformation has it
                continue
            take, ends, _, _ = both(fp32, rho * d, alpha)
            assert ends or not take, (alpha, rho)
            taken += take
    whole = alpha > 0 and alpha / 2 == int(alpha / 2) and alpha / 2 < TERMS[fp32]
    assert taken == (3 * 107 if whole else taken) and taken > 3 * 14


@pytest.mark.parametrize("fp32", [0, 1])
@pytest.mark.parametrize("alpha", [-20.0, -4.4, -1.0, 0.5, 1.3, 2.0, 3.0, 4.0, 8.0, 12.7])
def test_both_ways_agree_where_the_series_is_taken(both, fp32, alpha):
    """Bound: a rounding per term of the series, whose terms sum to e^(2 |p| rho)
    of the result at most, and a few of log1p and expm1, whose argument p ln(1 +
    z) multiplies them."""
    p = abs(alpha / 2)
    for d in DIRECTIONS:
        d = np.array(d) / np.linalg.norm(d)
        for rho in (1e-4, 1e-2, 0.05, 0.1, 0.2, 0.3, 0.42, 0.6):
            take, _, m, v = both(fp32, rho * d, alpha)
            if not take:
                continue
            tol = EPS[fp32] * (TERMS[fp32] + 8 * (1 + p * rho)) * np.exp(2 * p * rho)
            assert np.linalg.norm(m - v) <= tol * np.linalg.norm(v), (alpha, rho, d)
