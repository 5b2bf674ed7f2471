#!/usr/bin/env python3
"""Generate boys_poly.inc: the device Boys function's polynomials, one row per
order and interval.

Order m = 0..4 (the orders of the Obara-Saika kernels), interval i = 0..800 of
width 1/16 about x_i = i / 16: a row of eight doubles

    c_0 .. c_6, e^{-x_i}     F_m(x_i + d) = sum_k c_k d^k,  |d| <= 1/32,

the polynomial that interpolates F_m at the seven Chebyshev points of the
interval, computed with 50-digit arithmetic (mpmath) and rounded to the nearest
double.  Its error is below (1/32)^7 / (7! 2^6) F_{m+7} = 9.1e-17 F_{m+7}, at most
3.6e-17 of F_m (m = 4; F_{m+7} <= 9/23 F_m there).  A row is one aligned half of a cache
line, so that a lane's gather touches one line; the FP32 rows (c_0 .. c_4, two
spare, e^{-x_i}) are a quarter.
"""
import os

import mpmath
import numpy as np

STEP_INV = 16
XMAX = 50
ROWS = XMAX * STEP_INV + 1
ORDERS = 5


def boys_orders(top, x):
    """F_0..F_top(x): gamma function at the top order, downward recursion."""
    out = [mpmath.mpf(0)] * (top + 1)
    if x == 0:
        return [mpmath.mpf(1) / (2 * m + 1) for m in range(top + 1)]
    a = mpmath.mpf(top) + mpmath.mpf(1) / 2
    # series of the lower incomplete gamma function; valid at either sign of x
    s, t, k = mpmath.mpf(0), 1 / (2 * a), 0
    while abs(t) > abs(s) * mpmath.mpf(10) ** (-mpmath.mp.dps):
        s += t
        k += 1
        t *= x / (a + k)
    ex = mpmath.exp(-x)
    out[top] = s * ex
    for m in range(top, 0, -1):
        out[m - 1] = (2 * x * out[m] + ex) / (2 * m - 1)
    return out


def cheb_points(n):
    h = mpmath.mpf(1) / (2 * STEP_INV)
    return [h * mpmath.cos(mpmath.pi * (2 * k + 1) / (2 * n)) for k in range(n)]


def interp_matrix(n):
    """Inverse Vandermonde of the n Chebyshev points."""
    p = cheb_points(n)
    return p, mpmath.matrix([[x ** k for k in range(n)] for x in p]) ** -1


def f32(v):
    r = np.float32(float(v))
    c = [np.nextafter(r, np.float32(-np.inf)), r, np.nextafter(r, np.float32(np.inf))]
    return float(min(c, key=lambda t: abs(mpmath.mpf(float(t)) - v))).hex() + "f"


def main():
    mpmath.mp.dps = 50
    out = os.path.join(os.path.dirname(os.path.abspath(__file__)), "boys_poly.inc")
    p7, m7 = interp_matrix(7)
    p5, m5 = interp_matrix(5)
    rows, rows32 = [[] for _ in range(ORDERS)], [[] for _ in range(ORDERS)]
    for i in range(ROWS):
        xi = mpmath.mpf(i) / STEP_INV
        ex = mpmath.exp(-xi)
        v7 = [boys_orders(ORDERS - 1, xi + d) for d in p7]
        v5 = [boys_orders(ORDERS - 1, xi + d) for d in p5]
        for m in range(ORDERS):
            c = m7 * mpmath.matrix([v[m] for v in v7])
            rows[m].append([float(c[k]).hex() for k in range(7)] + [float(ex).hex()])
            c = m5 * mpmath.matrix([v[m] for v in v5])
            rows32[m].append([f32(c[k]) for k in range(5)] + ["0.0f", "0.0f", f32(ex)])
    lines = ["// Generated by gen_boys_poly.py -- do not edit.",
             "#pragma once",
             "#define PK_BOYS_STEP_INV %d" % STEP_INV,
             "#define PK_BOYS_XMAX %d" % XMAX,
             "#define PK_BOYS_ROWS %d" % ROWS,
             "#define PK_BOYS_ORDERS %d" % ORDERS]
    for name, typ, tab, al in (("pk_boys_row", "double", rows, 64), ("pk_boys_row_f", "float", rows32, 32)):
        lines.append("alignas(%d) PK_BOYS_QUALIFIER %s %s[%d] = {" % (al, typ, name, ORDERS * ROWS * 8))
        for m in range(ORDERS):
            lines += ["  " + ", ".join(r) + "," for r in tab[m]]
        lines.append("};")
    with open(out, "w") as f:
        f.write("\n".join(lines) + "\n")
    print("wrote", out)


if __name__ == "__main__":
    main()
