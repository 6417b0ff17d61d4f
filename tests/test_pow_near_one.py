"""The chain's power (mhm_amd/csrc/chain.h: pow_v) just above and below 1, where
y log x stays near 0 however large y is: no term of the size of y may be
rounded there.  The bound is the one pow_v states, (2 + 3 |y log x|) ulp, with
exponents up to the 65 that ordinary cells may have (1 + alpha, alpha < 64) and
bases on both sides of every table row that touches 1."""
import ctypes as C
import math
import os

import numpy as np
import pytest

mp = pytest.importorskip("mpmath")

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "tests", "native", "libmhmcheck.so")


@pytest.fixture(scope="module")
def power():
    if not os.path.exists(LIB):
        from mhm_amd import build
        build.build_check()
    f = C.CDLL(LIB).mhmhip_check_eval_host
    f.restype = C.c_int
    f.argtypes = [C.c_int] + [C.POINTER(C.c_double)] * 3 + [C.c_int64]

    def call(x, y):
        out = np.empty_like(x)
        p = [a.ctypes.data_as(C.POINTER(C.c_double)) for a in (x, y, out)]
        assert f(2, *p, x.shape[0]) == 0
        return out
    return call


def _bases(rng, n):
    """1 +- d: d spread over its logarithm, then evenly over the rows next to 1
    and out to where the exponent's part no longer cancels."""
    up = 1.0 + np.exp(rng.uniform(math.log(2.0**-52), math.log(0.05), n))
    even = rng.uniform(1.0, 1.05, n)
    rest = rng.uniform(1.05, 1.5, n // 2)
    down = 1.0 - np.exp(rng.uniform(math.log(2.0**-53), math.log(0.05), n // 2))
    edge = np.array([1.0 + k / 128.0 for k in range(1, 8)])
    edge = np.concatenate([edge, np.nextafter(edge, 0.0), np.nextafter(edge, 2.0)])
    return np.concatenate([up, even, rest, down, edge])


@pytest.mark.parametrize("y_lo,y_hi", [(0.1, 2.0), (2.0, 10.0), (10.0, 65.0)])
def test_power_next_to_one_keeps_its_bound(power, y_lo, y_hi):
    rng = np.random.default_rng(int(y_hi))
    x = _bases(rng, 6000)
    y = rng.uniform(y_lo, y_hi, x.shape[0])
    got = power(x, y)
    with mp.workprec(200):
        for g, a, b in zip(got, x, y):
            exact = mp.power(mp.mpf(float(a)), mp.mpf(float(b)))
            err = abs(mp.mpf(float(g)) - exact) / mp.mpf(math.ulp(float(exact)))
            assert err <= 2.0 + 3.0 * abs(b * math.log(a)), (a, b, float(err))


def test_one_to_any_power_is_one(power):
    y = np.concatenate([np.linspace(0.0, 65.0, 2001), -np.linspace(0.0, 65.0, 2001)])
    assert np.all(power(np.ones_like(y), y) == 1.0)
