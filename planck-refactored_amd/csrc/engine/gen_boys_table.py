#!/usr/bin/env python3
"""Generate boys_table.inc: F_m(x_i) on a grid, the table that the tests check
the large-argument branch, the recursions and the grid values against.

Grid x_i = i / 16, i = 0..BOYS_ROWS-1 (x <= 50), orders m = 0..BOYS_COLS-1, each
value the double nearest to F_m(x_i) = gamma_inc(m + 1/2, x_i) / (2 x_i^(m+1/2))
computed with 40-digit arithmetic (mpmath), and e^{-x_i}.  The kernels read the
polynomials of boys_poly.inc (gen_boys_poly.py) instead.
"""
import os

import mpmath

STEP_INV = 16
XMAX = 50
ROWS = XMAX * STEP_INV + 1
COLS = 24  # orders 0..23: Taylor top order up to 16 (L <= 16)


def F(m, x):
    if x == 0:
        return mpmath.mpf(1) / (2 * m + 1)
    return mpmath.gammainc(m + mpmath.mpf(1) / 2, 0, x) / (2 * x ** (m + mpmath.mpf(1) / 2))


def main():
    mpmath.mp.dps = 40
    out = os.path.join(os.path.dirname(os.path.abspath(__file__)), "boys_table.inc")
    lines = ["// Generated by gen_boys_table.py -- do not edit.",
             "// F_m(i/16), i < %d, m < %d (nearest doubles of 40-digit values)." % (ROWS, COLS),
             "#pragma once",
             "#define PK_BOYS_STEP_INV %d" % STEP_INV,
             "#define PK_BOYS_XMAX %d" % XMAX,
             "#define PK_BOYS_ROWS %d" % ROWS,
             "#define PK_BOYS_COLS %d" % COLS,
             "#ifndef PK_BOYS_QUALIFIER",
             "#define PK_BOYS_QUALIFIER static const",
             "#endif",
             "PK_BOYS_QUALIFIER double pk_boys_table[%d] = {" % (ROWS * COLS)]
    rows = []
    for i in range(ROWS):
        x = mpmath.mpf(i) / STEP_INV
        top = F(COLS - 1, x)
        ex = mpmath.exp(-x)
        vals = [mpmath.mpf(0)] * COLS
        vals[COLS - 1] = top
        for m in range(COLS - 1, 0, -1):
            vals[m - 1] = (2 * x * vals[m] + ex) / (2 * m - 1)
        rows.append(vals)
        lines.append("  " + ", ".join(float(v).hex() for v in vals) + ",")
    lines.append("};")
    lines.append("// e^{-x_i} on the same grid")
    lines.append("PK_BOYS_QUALIFIER double pk_boys_exp[%d] = {" % ROWS)
    lines.append("  " + ", ".join(float(mpmath.exp(-mpmath.mpf(i) / STEP_INV)).hex() for i in range(ROWS)))
    lines.append("};")
    with open(out, "w") as f:
        f.write("\n".join(lines) + "\n")
    print("wrote", out)


if __name__ == "__main__":
    main()
