"""Writes the reduction tables of i2_math.hpp.

i2_logtab.inc: entries j = 0..256 for the centres c_j = 1/2 + j/512 of the
mantissa range [1/2, 1): {invc_j, T_j hi, T_j lo} with invc_j = 1/c_j rounded
to double and T_j = -log(invc_j) split into a double hi part and a lo
remainder, so that log(m) = T_j + log1p(m invc_j - 1) to well below one ulp.

i2_atantab.inc: entries k = 0..32: {atan(k/32) hi, lo}.

It also prints the coefficients of atanh_over and atan_over of i2_math.hpp:
the interpolants of (atanh(sqrt s)/sqrt s - 1)/s on [0, 1/16] and
(atan(sqrt v)/sqrt v - 1)/v on [0, 0.003] at 8 and 5 Chebyshev nodes.

All values from 60-digit mpmath.  Run from this directory:
    python gen_math_tables.py
"""
import mpmath

mpmath.mp.dps = 60


def split(v):
    hi = float(v)
    return hi, float(v - mpmath.mpf(hi))


# ln 2 as the code splits it (LN2_HI to 32 significant bits, LN2_LO the rest)
LN2 = mpmath.log(2)
LN2_HI = float(mpmath.ldexp(mpmath.floor(mpmath.ldexp(LN2, 32)), -32))
LN2_LO = float(LN2 - mpmath.mpf(LN2_HI))
assert (LN2_HI, LN2_LO) == (0.69314718036912382, 1.9082149292705877e-10)

with open("i2_logtab.inc", "w") as f:
    f.write("// Generated by gen_math_tables.py: {invc, -log(invc) hi, lo} for c = 1/2 + j/512, j = 0..256\n")
    for j in range(257):
        c = mpmath.mpf(1) / 2 + mpmath.mpf(j) / 512
        invc = float(1 / c)
        hi, lo = split(-mpmath.log(mpmath.mpf(invc)))
        if j == 0:
            # T_0 = -ln 2 in the code's split, so that k = 1 cancels it exactly
            # and log(x) for x just above 1 is log1p(x - 1) alone
            hi, lo = -LN2_HI, -LN2_LO
        f.write("{%r, %r, %r},\n" % (invc, hi, lo))

with open("i2_atantab.inc", "w") as f:
    f.write("// Generated by gen_math_tables.py: {atan(k/32) hi, lo}, k = 0..32\n")
    for k in range(33):
        hi, lo = split(mpmath.atan(mpmath.mpf(k) / 32))
        f.write("{%r, %r},\n" % (hi, lo))


def interpolant(f, top, n):
    """Coefficients, ascending, of the degree-(n - 1) interpolant of (f(s) - 1)/s on [0, top]."""
    nodes = [top / 2 * (1 + mpmath.cos(mpmath.pi * (2 * k + 1) / (2 * n))) for k in range(n)]
    A = mpmath.matrix([[s ** j for j in range(n)] for s in nodes])
    return [float(c) for c in mpmath.lu_solve(A, mpmath.matrix([(f(s) - 1) / s for s in nodes]))]


print("atanh_over", interpolant(lambda s: mpmath.atanh(mpmath.sqrt(s)) / mpmath.sqrt(s), mpmath.mpf(1) / 16, 8))
print("atan_over", interpolant(lambda s: mpmath.atan(mpmath.sqrt(s)) / mpmath.sqrt(s), mpmath.mpf("0.003"), 5))
print("atanh_over, distant", interpolant(lambda s: mpmath.atanh(mpmath.sqrt(s)) / mpmath.sqrt(s), mpmath.mpf(1) / 144, 5))
print("atan_over, distant", interpolant(lambda s: mpmath.atan(mpmath.sqrt(s)) / mpmath.sqrt(s), mpmath.mpf("3.7e-5"), 3))
print("cos_turns, c", interpolant(lambda s: mpmath.cos(2 * mpmath.pi * mpmath.sqrt(s)), mpmath.mpf(1) / 64, 7))
print("cos_turns, s", interpolant(lambda s: 1 + mpmath.sqrt(s) * mpmath.sin(2 * mpmath.pi * mpmath.sqrt(s)), mpmath.mpf(1) / 64, 7))
