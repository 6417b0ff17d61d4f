"""One step of the branch-free form of the cell chain beside its branches
(chain.h), on the device, over the ranges in which a cell may take it: weather,
parameters and states at random, many of them at an edge of their range or
where two branches meet.  And its power of the canopy's ratio (pow23_ratio)
against mpmath.

Bounds.  The two canopy powers are each within 3 ulp of the exact one, so the
canopy's evaporation differs by 8 ulp at most (the product rounds both once).
The other values come from the same operations on it, or, where two branches
meet, from the other branch's, one rounding of the store they meet at away: 32
roundings of the largest of the cell's stores and fluxes bound them all.  Away
from those meeting points they are as close as the canopy's: 19 of 20 cells
within 16 ulp of the value itself."""
import ctypes as C
import os
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "tests", "native", "libmhmcheck.so")
NH, EPS = 3, np.finfo(float).eps
OUT = (["thr", "ecan", "inter", "ddf", "melt", "peff", "rain", "snow", "pack", "rseal", "aseal",
        "seal"] + [f"{v}{h}" for v in ("infil", "aet", "sm") for h in range(NH)]
       + ["fast", "slow", "perc", "unsat", "sats", "bflow", "total"])


@pytest.fixture(scope="module")
def lib():
    if not os.path.exists(LIB):
        from mhm_amd import build
        build.build_check()
    h = C.CDLL(LIB)
    h.mhmhip_check_forms.argtypes = [C.c_int] + [C.c_void_p] * 4 + [C.c_int64]
    h.mhmhip_check_ratio.argtypes = [C.c_void_p] * 2 + [C.c_int64]
    return h


def _cells(rng, n):
    """(n, inputs), in the order of formcheck.hip's In."""
    def pick(random, *edges):
        v = np.array(random, dtype=float)
        for e in edges:
            sel = rng.random(n) < 0.08
            v[sel] = np.broadcast_to(e, (n,))[sel]
        return v

    prec = pick(rng.gamma(0.4, 4.0, n), 0.0, 0.0, 80.0)
    tth = pick(rng.uniform(-1.0, 2.0, n), 0.0)
    temp = pick(rng.normal(2.0, 8.0, n), tth, 0.0)
    pet = pick(rng.gamma(1.5, 1.0, n), 0.0, -0.2)
    maxi = pick(rng.uniform(0.05, 6.0, n), 0.0, EPS, 1e-12)
    evap = rng.uniform(0.5, 1.5, n)
    fs = pick(rng.random(n), 0.0, 0.0, 1.0)
    thrs = pick(rng.uniform(0.1, 5.0, n), 2e-15)
    incr = pick(rng.uniform(0.0, 1.0, n), 0.0)
    dmax = pick(rng.uniform(0.0, 8.0, n), 0.0)
    dnp = pick(rng.uniform(0.0, 4.0, n), 0.0, dmax)
    k0, k1 = pick(rng.uniform(0.0, 1.2, n), 0.0, 1.0), pick(rng.uniform(0.0, 0.5, n), 0.0)
    k2, kp = pick(rng.random(n), 0.0, 1.0), pick(rng.uniform(0.0, 1.2, n), 0.0, 1.0)
    karst, alpha = pick(rng.uniform(0.0, 1.5, n), 0.0), pick(rng.uniform(-0.5, 1.0, n), 0.0)
    thru, c1 = pick(rng.uniform(1.0, 60.0, n), 2e-15), pick(rng.uniform(0.05, 1.0, n), 1.0)
    sat = [pick(rng.uniform(20.0, 300.0, n), 1.0) for _ in range(NH)]
    fc = [pick(s * rng.uniform(0.3, 1.0, n), s) for s in sat]
    wp = [pick(f * rng.uniform(0.0, 0.95, n), 0.0, f * (1.0 - 1e-9)) for f in fc]
    fr = [pick(rng.random(n), 0.0) for _ in range(NH)]
    bexp = [pick(rng.uniform(1.0, 6.0, n), 1.0, 20.0) for _ in range(NH)]
    inter = pick(maxi * rng.random(n), 0.0, maxi)
    pack = pick(rng.gamma(0.7, 20.0, n), 0.0, 0.0)
    seal = pick(thrs * rng.random(n), 0.0, thrs)
    unsat = pick(rng.gamma(1.0, 20.0, n), 0.0, thru, EPS, np.maximum(thru - prec, 0.0))
    sats = pick(rng.gamma(1.0, 60.0, n), 0.0)
    sm = [pick(np.maximum(s * rng.random(n), EPS), EPS, s, f, np.maximum(w, EPS))
          for s, f, w in zip(sat, fc, wp)]
    cols = [prec, temp, pet, maxi, evap, fs, thrs, incr, dmax, dnp, tth, k0, k1, k2, kp, karst,
            alpha, thru, c1, *sat, *fr, *fc, *wp, *bexp, inter, pack, seal, unsat, sats, *sm]
    return np.ascontiguousarray(np.stack(cols, axis=1))


@pytest.mark.parametrize("jarvis,n", [(0, 200000), (1, 200000), (0, 1), (1, 255)])
def test_branch_free_step_equals_the_branches(lib, jarvis, n):
    print(f"case: forms of a step, jarvis={jarvis}, {n} cells", flush=True)
    sys.stdout.flush()
    cells = _cells(np.random.default_rng(90 + jarvis), n)
    ni, no = C.c_int(), C.c_int()
    lib.mhmhip_check_form_sizes(C.byref(ni), C.byref(no))
    assert (ni.value, no.value) == (cells.shape[1], len(OUT))
    a, b = np.empty((n, len(OUT))), np.empty((n, len(OUT)))
    ok = np.zeros(n, np.int32)
    assert lib.mhmhip_check_forms(jarvis, cells.ctypes.data, a.ctypes.data, b.ctypes.data,
                                  ok.ctypes.data, n) == 0
    sel = ok != 0
    if n > 1000:
        assert sel.mean() > 0.5
    a, b, cells = a[sel], b[sel], cells[sel]
    # the cell's largest store, flux or forcing
    size = np.maximum(np.abs(np.delete(cells, [1, 4, 10], axis=1)).max(axis=1, initial=0.0),
                      np.abs(a).max(axis=1, initial=0.0))
    for k, name in enumerate(OUT):
        diff = np.abs(a[:, k] - b[:, k])
        assert not np.isnan(diff).any(), name
        assert np.all(diff <= 32 * EPS * size), (name, float((diff / (EPS * size)).max()))
        if name == "ecan":
            assert np.all(diff <= 8 * np.spacing(np.abs(a[:, k]))), name
        if n > 1000:
            close = diff <= 16 * np.spacing(np.abs(a[:, k]))
            assert close.mean() >= 0.95, (name, float(close.mean()))


def test_device_ratio_power_within_three_ulp(lib):
    """pow23_ratio over the canopy's ratios, small ones through pow23; 0,
    negative and NaN ratios give NaN or -inf (the canopy's maximum with 0 drops
    both)."""
    mp = pytest.importorskip("mpmath")
    print("case: ratio power on the device", flush=True)
    rng = np.random.default_rng(91)
    n = 20000
    x = np.concatenate([rng.random(n), 2.0 ** rng.uniform(-40.0, 0.0, n),
                        np.exp(rng.uniform(-700.0, 0.0, n)),
                        2.0 ** rng.uniform(-33.0, -31.0, n),
                        np.array([1.0, 1.0 - 2**-53, 0.5, 2.0**-32, 2.0**-30, 2.0**-33, 2.0**-1000])])
    got = np.empty_like(x)
    assert lib.mhmhip_check_ratio(x.ctypes.data, got.ctypes.data, x.shape[0]) == 0
    with mp.workprec(120):
        for g, v in zip(got[::5], x[::5]):
            want = mp.power(mp.mpf(float(v)), mp.mpf(2) / 3)
            assert abs(mp.mpf(float(g)) - want) <= 3 * mp.mpf(float(np.spacing(float(want)))), v
    odd = np.array([0.0, -1.0, -1e-300, np.nan])
    got = np.empty_like(odd)
    assert lib.mhmhip_check_ratio(odd.ctypes.data, got.ctypes.data, 4) == 0
    assert np.all(np.isnan(got) | (got == -np.inf)), got
