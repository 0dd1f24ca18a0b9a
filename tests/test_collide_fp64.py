"""The collision form that FP64 storage runs, compiled for the host, against the
oracle: all three cumulant operators and the Smagorinsky rate, with rho and u the
moments of the populations and, as on a first step, others."""
import ctypes
import os

import numpy as np
import pytest

from helpers import host_collide_lib, oracle_lib
from lb_amd import abi
from test_oracle import feq

_dp, _d = ctypes.POINTER(ctypes.c_double), ctypes.c_double


@pytest.fixture(scope="module")
def lib():
    L = ctypes.CDLL(os.path.join(os.path.dirname(__file__), "native", "libcollide_fp64_host.so"))
    L.host_fp64_collide.argtypes = [ctypes.c_int, ctypes.c_uint32, _dp, _d, _d, _d, _d, _d, _dp]
    L.host_fp64_collide.restype = None
    L.host_fp64_omega_les.argtypes = [_dp, _d, _d, _d, _d, _d, _d]
    L.host_fp64_omega_les.restype = _d
    return L


@pytest.mark.parametrize("first", [False, True], ids=["moments", "first_step"])
@pytest.mark.parametrize("compat", [0, abi.COMPAT_REFERENCE], ids=["published", "reference"])
@pytest.mark.parametrize("op", [abi.COLLISION_CUM2015, abi.COLLISION_CUM2017, abi.COLLISION_COMBINED],
                         ids=["2015", "2017", "combined"])
def test_fp64_collision_equals_the_oracle(lib, op, compat, first):
    O, rng = oracle_lib(), np.random.default_rng(21)
    worst = 0.0
    for it in range(200):
        f = feq(1 + 0.02 * rng.standard_normal(), 0.05 * rng.standard_normal(3)) * (1 + 0.02 * rng.standard_normal(27))
        om = (1.3, 1.9, 1.99)[it % 3]
        m = np.zeros(4)
        host_collide_lib().host_moments(1, abi.ptr(f), abi.ptr(m))
        if first:
            m = m + 1e-3 * rng.standard_normal(4)
        a, b = np.zeros(27), np.zeros(27)
        O.orc_cell_collide(op, compat, 1, abi.ptr(f), *m, om, 2, abi.ptr(a))
        lib.host_fp64_collide(op, compat, abi.ptr(f), *m, om, abi.ptr(b))
        worst = max(worst, np.abs(a - b).max())
    # populations up to 0.3 from sums of some 60 rounded terms: a few ulp of the
    # largest (5.6e-17 each)
    assert worst < 2e-15


@pytest.mark.parametrize("first", [False, True], ids=["moments", "first_step"])
def test_fp64_rate_equals_the_oracle(lib, first):
    O, rng = oracle_lib(), np.random.default_rng(22)
    for it in range(200):
        f = feq(1 + 0.02 * rng.standard_normal(), 0.05 * rng.standard_normal(3)) * (1 + 0.02 * rng.standard_normal(27))
        m = np.zeros(4)
        host_collide_lib().host_moments(1, abi.ptr(f), abi.ptr(m))
        if first:
            m = m + 1e-3 * rng.standard_normal(4)
        # with other rho and u than the moments the oracle's tensor (c c against the
        # equilibrium) is another one than the central moments: there the written-out
        # form of the fast arithmetic is the reference
        if first:
            a = host_collide_lib().host_omega_les(1, 1, 0, abi.ptr(f), *m, 0.5015, 0.173)
        else:
            a = O.orc_cell_omega_les(0, 1, abi.ptr(f), *m, 0.5015, 0.173)
        b = lib.host_fp64_omega_les(abi.ptr(f), *m, 0.5015, 0.173)
        # |Pi_neq| within some 1e-15, times d omega / d |Pi_neq| of at most 18 C omega^3 / 4
        assert abs(a - b) < 2e-14
