"""Coefficients of cs3d_theta.h.

The degree-15 Chebyshev interpolant of acos(t - 0.425) on |t| <= 0.275, computed
in 60-digit decimal arithmetic, converted to monomial coefficients in t and
rounded to double.  Prints the coefficients (constant term first) and the largest
absolute error of the rounded polynomial on a grid of 2001 points.

    python gen_theta_coeffs.py [degree]
"""
import math
import sys
from decimal import Decimal as D
from decimal import getcontext

getcontext().prec = 60
CENTRE, HALF = D("-0.425"), D("0.275")


def asin_series(s):
    """asin for |s| <= 0.75 from its power series."""
    s = D(s)
    tot, t, z = D(0), s, s * s
    for k in range(0, 2000):
        term = t / (2 * k + 1)
        tot += term
        if abs(term) < D(10) ** -58:
            break
        t = t * z * D(2 * k + 1) / D(2 * k + 2)
    return tot


PI = 6 * asin_series(D(1) / 2)


def acos_dec(x):
    return PI / 2 - asin_series(x)


def cos_dec(x):
    s, t, k = D(1), D(1), 0
    while abs(t) >= D(10) ** -59:
        k += 2
        t = -t * x * x / (k * (k - 1))
        s += t
    return s


def cheb(k, t):
    a, b = D(1), t
    for _ in range(k):
        a, b = b, 2 * t * b - a
    return a


deg = int(sys.argv[1]) if len(sys.argv) > 1 else 15
n = deg + 1
nodes = [cos_dec(PI * (2 * j + 1) / (2 * n)) for j in range(n)]
fx = [acos_dec(CENTRE + HALF * u) for u in nodes]
a = [sum(fx[j] * cheb(k, nodes[j]) for j in range(n)) * 2 / n for k in range(n)]
a[0] /= 2
# sum a_k T_k(u) with u = t / HALF as monomials of t
polys = [[D(1)], [D(0), 1 / HALF]]
for k in range(2, n):
    r = [D(0)] + [2 / HALF * v for v in polys[-1]]
    prev = polys[-2] + [D(0)] * (len(r) - len(polys[-2]))
    polys.append([x - y for x, y in zip(r, prev)])
c = [D(0)] * n
for k in range(n):
    for i, v in enumerate(polys[k]):
        c[i] += a[k] * v
for i, v in enumerate(c):
    print("    %s,  // t^%d" % (float(v).hex(), i))
cd = [D(float(v)) for v in c]
worst = D(0)
for j in range(2001):
    t = HALF * (D(j) / 1000 - 1)
    p = D(0)
    for v in reversed(cd):
        p = p * t + v
    worst = max(worst, abs(p - acos_dec(CENTRE + t)))
print("max abs err %.3e = 2^%.2f" % (float(worst), math.log2(float(worst))))
