"""The expansion of J1 that neighbouring flux rows share (expand_j1 and
expanded_values in upc_flux.h), step by step in Python with its own tables and
limits (CPU only).  Against J1 to 40 digits its error stays within 4.9e-16 of
the envelope min(x / 2, sqrt(2 / (pi x))) wherever the kernel uses it: at the
ends of each term count's range of delta, up to the largest delta / x0 let
through (a group of rows beyond it evaluates its own nodes)."""
import os
import re
from fractions import Fraction

import pytest

mp = pytest.importorskip("mpmath")
mp.mp.dps = 40

SRC = open(os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "upcgen_amd", "csrc",
                        "upc_flux.h")).read()


def _numbers(name):
    return [float(v) for v in re.search(name + r"\[[^\]]*\] = \{([^}]*)\}", SRC).group(1).split(",")]


TERMS = [int(v) for v in _numbers("kExpandTerms")]
DELTA = _numbers("kExpandMax")
_ratio = re.search(r"kExpandRatio = ([0-9.e-]+);", SRC)
RATIO = float(_ratio.group(1)) if _ratio else 0.99  # no limit: delta < x0


def fma(a, b, c):
    return float(Fraction(a) * Fraction(b) + Fraction(c))


def coefficients(x0, q, T):
    j0, j1 = float(mp.besselj(0, x0)), float(mp.besselj(1, x0))
    r = 1.0 / x0
    r2 = r * r
    am2, am1, a, ap, qn = 0.0, 0.0, j1, fma(-j1, r, j0), q
    cf = [j1, ap * q]
    for n in range(T - 2):
        A, B, C = 1.0 / ((n + 1) * (n + 2)), (n - 1) / (n + 2), (2 * n + 1) / (n + 2)
        s = fma(fma(B, r2, A), a, A * fma(2.0 * r, am1, r2 * am2))
        an = -fma(C * r, ap, s)
        qn *= q
        cf.append(an * qn)
        am2, am1, a, ap = am1, a, ap, an
    return cf


def value(cf, db):
    T = len(cf)
    if T > 10:
        j = cf[-1]
        for c in cf[-2::-1]:
            j = fma(j, db, c)
        return j
    pw = [1.0]
    for _ in range(T - 1):
        pw.append(pw[-1] * db)
    j = 0.0
    for k in range(T - 1, -1, -1):
        j = fma(cf[k], pw[k], j)
    return j


@pytest.mark.parametrize("kind", range(1, len(TERMS)))
def test_expansion(kind):
    lo, hi = DELTA[kind - 1], DELTA[kind]
    worst = 0.0
    for delta in (hi, 0.5 * (lo + hi), lo + 0.01 * (hi - lo)):
        for ratio in (RATIO, 0.9 * RATIO, 0.5 * RATIO, 0.1 * RATIO, 0.003):
            for q in (0.013, 0.7):
                x0 = delta / ratio
                cf = coefficients(x0, q, TERMS[kind])
                for db in (delta / q, -delta / q, 0.6 * delta / q):
                    x = mp.mpf(x0) + mp.mpf(q) * mp.mpf(db)
                    envelope = min(x / 2, mp.sqrt(2 / (mp.pi * x)))
                    worst = max(worst, float(abs(mp.mpf(value(cf, db)) - mp.besselj(1, x)) / envelope))
    assert worst <= 4.9e-16, worst
