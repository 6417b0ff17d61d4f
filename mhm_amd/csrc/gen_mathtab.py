"""Writes mathtab.h: the tables of the chain's logarithm, exponential and power
(chain.h, log_pos_v, exp_fin_v and pow_v).

Logarithm, F_j = j / 256 for j = 128..256 (F from 1/2 to 1, the nearest
point to the frexp mantissa m in [1/2, 1)): RN(1 / F_j) and log(F_j) split as
hi + lo, hi a multiple of 2^-42 (so e*ln2_hi + hi is exact for the exponents
of finite doubles) and lo = RN(log(F_j) - hi); a fourth entry of 0 pads each
row to 32 bytes.  F = 1/2 holds -(ln2_hi + ln2_lo) exactly, the split of
ln 2 that log_pos_v multiplies by the exponent, so that for x just above 1
(m near 1/2, e = 1) the two cancel without a rounding.

Exponential, 2^(j/256) for j = 0..255 as hi = RN(2^(j/256)) and
lo = RN(2^(j/256) - hi).

Power (pow_v in chain.h): base-2 logarithm rows {R, L} for j = 0..127, one per
interval [(128 + j)/256, (129 + j)/256) of the frexp mantissa m: R near the
reciprocal of the interval's middle, u = m R - 1 and log2(m) = L +
log2(1 + u).  R is searched next to that reciprocal so that L = -log2(R) lies
within 2^-66 of a multiple of 2^-42 (the accurate tables of Gal, in "Computing
elementary functions: a new approach for achieving high accuracy and good
performance", LNCS 235 (1986) 1-16): one double holds it, and e + L is exact
for the exponent e of every finite double, also where the two nearly cancel (x
just above 1).  The first row has R = 2 and the last R = 1, both with exact
logarithms, so that log2 x is 0 at x = 1.  These rows stand behind those of
2^(j/256), which the power uses too: the cell kernels copy both to LDS in one
piece.  And the coefficients of log2(1 + u) = u (c0 + ... + c5 u^5) on [-1/256, 1/128] and of
2^(r/256) = 1 + r (d0 + ... + d3 r^3) on [-1/2, 1/2], interpolated at Chebyshev
nodes; main() checks that log2(1 + u) and 2^(r/256) come out with relative
errors below 2^-51.8 and 2^-57.5.

Values from mpmath at 256 bits.
Run: python mhm_amd/csrc/gen_mathtab.py > mhm_amd/csrc/mathtab.h
"""
import math

import mpmath as mp

mp.mp.prec = 256
LOG_J0, LOG_J1 = 128, 256
EXP_N = 256
LN2_HI = float.fromhex("0x1.62e42fee00000p-1")  # chain.h kLn2Hi
LN2_LO = float.fromhex("0x1.a39ef35793c76p-33")  # chain.h kLn2Lo


def log_row(j):
    F = mp.mpf(j) / 256
    inv = float(1 / F)
    if j == 128:
        return inv, -LN2_HI, -LN2_LO
    L = mp.log(F)
    hi = math.ldexp(math.trunc(math.ldexp(float(L), 42)), -42)  # toward zero
    return inv, hi, float(L - mp.mpf(hi))


def exp_row(j):
    T = mp.power(2, mp.mpf(j) / EXP_N)
    hi = float(T)
    return hi, float(T - mp.mpf(hi))


def pow_row(j):
    if j == 0:
        return 2.0, -1.0
    if j == 127:
        return 1.0, 0.0
    # the grid's logarithms from the reciprocal's on, their powers of 2 a
    # factor apart: the first that a double meets to 2^-66 in the logarithm
    g = math.floor(mp.ldexp(-mp.log(mp.mpf(512) / (2 * (128 + j) + 1), 2), 42))
    want, step = mp.power(2, mp.ldexp(-g, -42)), mp.power(2, mp.ldexp(1, -42))
    with mp.workprec(128):
        while abs(mp.mpf(float(want)) / want - 1) * mp.log(mp.e, 2) > mp.ldexp(1, -66):
            g, want = g - 1, want * step
    R, L = float(want), math.ldexp(g, -42)
    assert abs(mp.log(mp.mpf(R), 2) + mp.mpf(L)) < mp.ldexp(1, -66) * 1.001
    return R, L


def chebyshev_fit(f, a, b, n):
    """Coefficients (constant first) of the degree n - 1 polynomial through f
    at the n Chebyshev nodes of [a, b]."""
    a, b = mp.mpf(a), mp.mpf(b)
    x = [(a + b) / 2 + (b - a) / 2 * mp.cos(mp.pi * (2 * k + 1) / (2 * n)) for k in range(n)]
    A = mp.matrix(n, n)
    y = mp.matrix(n, 1)
    for i in range(n):
        y[i] = f(x[i])
        for k in range(n):
            A[i, k] = x[i] ** k
    return [float(c) for c in mp.lu_solve(A, y)]


def worst_error(f, c, c0, a, b):
    """Largest relative error of c0 + t (c[0] + c[1] t + ...) against f over a
    grid of [a, b]."""
    worst = mp.mpf(0)
    for i in range(2001):
        t = a + (b - a) * i / 2000
        if f(t) != 0:
            p = c0 + t * mp.polyval([mp.mpf(v) for v in reversed(c)], t)
            worst = max(worst, abs(p / f(t) - 1))
    return worst


def main():
    assert LN2_HI + LN2_LO == float(mp.log(2))
    print("// mathtab.h -- generated by gen_mathtab.py; do not edit.")
    print("#pragma once")
    print("namespace mhmhip {")
    print("constexpr int kLogTabJ0 = %d;" % LOG_J0)
    print("constexpr int kLogTabN = %d;" % (LOG_J1 - LOG_J0 + 1))
    print("constexpr int kExpTabN = %d;" % EXP_N)
    print("constexpr int kPowLogN = 128;")
    print("constexpr int kExpTabOff = kLogTabN * 4;  // the exp rows' first element, then the power's")
    print("alignas(16) constexpr double kMathTab[kLogTabN * 4 + kExpTabN * 2 + kPowLogN * 2] = {")
    print("    // log: {RN(1/F), hi(log F), lo(log F), 0} for F = j/256, j = %d..%d"
          % (LOG_J0, LOG_J1))
    for j in range(LOG_J0, LOG_J1 + 1):
        inv, hi, lo = log_row(j)
        print("    %s, %s, %s, 0.0," % (inv.hex(), hi.hex(), lo.hex()))
    print("    // exp: {hi, lo} of 2^(j/%d), j = 0..%d" % (EXP_N, EXP_N - 1))
    for j in range(EXP_N):
        hi, lo = exp_row(j)
        print("    %s, %s," % (hi.hex(), lo.hex()))
    print("    // power: {R, L}, log2(m) = L + log2(m R), by interval of m")
    for j in range(128):
        print("    %s, %s," % tuple(v.hex() for v in pow_row(j)))
    print("};")
    half, u0, u1 = mp.mpf(1) / 2, -mp.mpf(1) / 256, mp.mpf(1) / 128
    c = chebyshev_fit(lambda u: mp.log(1 + u, 2) / u, u0, u1, 6)
    d = chebyshev_fit(lambda r: (mp.power(2, r / 256) - 1) / r, -half, half, 4)
    assert worst_error(lambda u: mp.log(1 + u, 2), c, 0, u0, u1) < mp.power(2, -51.8)
    assert worst_error(lambda r: mp.power(2, r / 256), d, 1, -half, half) < mp.power(2, -57.5)
    print("// log2(1 + u) / u and (2^(r/256) - 1) / r, constant term first")
    print("constexpr double kPowC[6] = {%s};" % ", ".join(v.hex() for v in c))
    print("constexpr double kPowD[4] = {%s};" % ", ".join(v.hex() for v in d))
    print("}  // namespace mhmhip")


if __name__ == "__main__":
    main()
