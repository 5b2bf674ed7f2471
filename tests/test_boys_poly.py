"""The device Boys function's polynomial rows (boys_poly.inc), evaluated in the
order of the kernels (`boys<M>` in eri_prim.h) against the confluent
hypergeometric function of mpmath."""
import math
import os
import re

import mpmath
import numpy as np
import pytest

INC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "planck-refactored_amd", "csrc", "engine",
                   "boys_poly.inc")


def _table(name, typ):
    src = open(INC).read()
    body = src[src.index(name + "["):]
    body = body[body.index("{") + 1:body.index("}")]
    vals = [typ(float.fromhex(t.rstrip("f"))) if t[-1] == "f" and "x" in t and typ is np.float32 else typ(0)
            if t == "0.0f" else typ(float.fromhex(t)) for t in re.split(r"[,\s]+", body.strip(" ,\n"))]
    return np.array(vals, dtype=typ).reshape(5, 801, 8)


def _exact(m, T):
    return mpmath.hyp1f1(m + mpmath.mpf(1) / 2, m + mpmath.mpf(3) / 2, -T) / (2 * m + 1)


def _points():
    rng = np.random.default_rng(31)
    edges = [0.0, 1e-300, 1e-13, 1.0 / 32, np.nextafter(1.0 / 32, 0), 49.96875, np.nextafter(50.0, 0), 50.0, 50.03, 1e3]
    return [float(t) for t in np.concatenate([rng.uniform(0, 2, 40), rng.uniform(0, 55, 60)])] + edges


# Rounding u per operation: F_M carries 3 u (its leading coefficient, the last
# step and the rest), e^{-T} 4 u, each recursion step 3 u more (the error of a
# sum of positive terms is at most the larger of theirs): 4 u + 4 x 3 u = 16 u;
# above 50, 3 u and 4 u a step (1/2T twice rounded): 19 u.  The fits' own errors
# (4e-17; FP32 2e-11) are below 1 u.
@pytest.mark.parametrize("typ,u", [(np.float64, 2.0 ** -53), (np.float32, 2.0 ** -24)])
@pytest.mark.parametrize("M", range(5))
def test_boys_rows(M, typ, u):
    mpmath.mp.dps = 40
    f32 = typ is np.float32
    tab = _table("pk_boys_row_f" if f32 else "pk_boys_row", typ)
    for T in _points():
        T = typ(T)
        F = [typ(0)] * (M + 1)
        if T < 50:
            i = int(T * typ(16) + typ(0.5))
            assert 0 <= i < 801
            d = T - typ(i / 16.0)
            row = tab[M, i]
            deg = 4 if f32 else 6
            s = row[deg]
            for k in range(deg - 1, -1, -1):
                s = s * d + row[k]
            F[M] = s
            e = typ(0)
            for k in range(5 if f32 else 8, -1, -1):
                e = e * -d + typ(1.0 / math.factorial(k))
            eT = row[7] * e
            for m in range(M, 0, -1):
                F[m - 1] = (typ(2) * T * F[m] + eT) * typ(1.0 / (2 * m - 1))
        else:
            r = 1.0 / math.sqrt(float(T))
            f = 0.88622692545275801365 * r
            F[0] = typ(f)
            for m in range(1, M + 1):
                f = (2 * m - 1) * f * (0.5 * r * r)
                F[m] = typ(f)
        for m in range(M + 1):
            ex = _exact(m, mpmath.mpf(float(T)))
            assert abs(mpmath.mpf(float(F[m])) - ex) <= 19 * u * ex, (m, T)
