#!/usr/bin/env python3
"""Fits the arctangent polynomials of the direct-sum tile kernel (ds.hip).

atan(t) = t * P(t^2) with P of degree n, minimising the maximum relative
error on |t| <= a (Remez exchange on f(s) = atan(sqrt(s)) / sqrt(s),
s = t^2, weight 1/f), then rounds the coefficients to FP32:

* atan_unit (ds.hip): a = 1, degree 7;
* the paired small-angle series (ds.hip, short path): a = 16/63, degree 4.

The FP64 tile kernel's series (atan_short_f64) is atan(t) = t + t s Q(s) on
|t| <= tan(4 atan(1/16)), Q of degree 7 interpolated at Chebyshev nodes.  The
set printed here differs from the kernel's by 5e-8 of the highest coefficient and
by less in the others (the interpolation's own rounding); both are within 2.6e-17.

Usage: python fit_atan_poly.py  -- prints the coefficient sets (highest
degree first, as ds.hip evaluates them by Horner's rule) and their maximum
relative errors in exact arithmetic.
"""
import numpy as np


def _f(s):
    s = np.asarray(s, dtype=np.float64)
    r = np.sqrt(s)
    out = np.ones_like(s)
    nz = r > 1e-8
    out[nz] = np.arctan(r[nz]) / r[nz]
    small = ~nz  # series 1 - s/3 + s^2/5
    out[small] = 1.0 - s[small] / 3.0 + s[small] ** 2 / 5.0
    return out


def remez(a, degree, iters=60, grid=200001):
    """Coefficients c[0..degree] (lowest first) of P minimising
    max |t P(t^2) / atan(t) - 1| on 0 < t <= a."""
    b = a * a
    m = degree + 2
    # Chebyshev extrema as the first reference
    x = 0.5 * b * (1 - np.cos(np.pi * np.arange(m) / (m - 1)))
    s = np.linspace(0.0, b, grid)
    fs = _f(s)
    c = None
    for _ in range(iters):
        fx = _f(x)
        A = np.zeros((m, m))
        for j in range(degree + 1):
            A[:, j] = x ** j
        A[:, degree + 1] = ((-1.0) ** np.arange(m)) * fx
        sol = np.linalg.solve(A, fx)
        c = sol[: degree + 1]
        err = np.polyval(c[::-1], s) / fs - 1.0
        # new reference: the extremum of each run of constant sign
        sign = np.sign(err)
        sign[sign == 0] = 1
        idx, start = [], 0
        for k in range(1, len(s) + 1):
            if k == len(s) or sign[k] != sign[start]:
                seg = np.arange(start, k)
                idx.append(seg[np.argmax(np.abs(err[seg]))])
                start = k
        if len(idx) < m:
            break
        # keep m alternating extrema with the largest errors
        while len(idx) > m:
            drop = 0 if abs(err[idx[0]]) < abs(err[idx[-1]]) else len(idx) - 1
            idx.pop(drop)
        xn = s[idx]
        if np.allclose(xn, x, rtol=0, atol=1e-15 * b):
            break
        x = xn
    return c


def _tail(s):
    """(atan(t)/t - 1) / s for s = t^2 < 0.1, in extended precision."""
    out = np.zeros_like(s)
    for k in range(59, 0, -1):
        out = out * s + np.longdouble((-1) ** k) / (2 * k + 1)
    return out


def max_rel_error_f64(c, a):
    """Maximum relative error of t + t s Q(s) against atan(t) on |t| <= a, Q of
    the FP64 coefficients c (lowest first), in extended precision."""
    s = np.longdouble(a) ** 2 * np.linspace(0, 1, 100001)[1:].astype(np.longdouble)
    q = np.zeros_like(s)
    for v in c[::-1]:
        q = q * s + np.longdouble(v)
    return float(np.max(np.abs((q - _tail(s)) * s / (1 + s * _tail(s)))))


def interpolate_f64(a, degree):
    """Coefficients (lowest first, FP64) of Q in atan(t) = t + t s Q(s) on
    |t| <= a, and the maximum relative error of the result there."""
    b, m = np.longdouble(a) ** 2, degree + 1
    x = b / 2 * (1 - np.cos(np.longdouble(np.pi) * (2 * np.arange(m).astype(np.longdouble) + 1) / (2 * m)))
    d = _tail(x)  # Newton's divided differences
    for k in range(1, m):
        d[k:] = (d[k:] - d[k - 1:-1]) / (x[k:] - x[:-k])
    c = np.zeros(m, dtype=np.longdouble)  # to powers of s
    for k in range(m - 1, -1, -1):
        c[1:] = c[:-1] - x[k] * c[1:]
        c[0] = d[k] - x[k] * c[0]
    c = c.astype(np.float64)
    return c, max_rel_error_f64(c, a)


def max_rel_error(coef_high_first, a, n=400001, fp32=False):
    """Maximum relative error of t * P(t^2) against atan(t) on 0 < t <= a,
    in float64 arithmetic or emulating the kernel's FP32 Horner evaluation
    with fused multiply-adds; also the mean signed error (bias)."""
    t = np.linspace(a / n, a, n)
    if fp32:
        t32 = t.astype(np.float32)
        s = (t32 * t32).astype(np.float32)
        p = np.full_like(s, np.float32(coef_high_first[0]))
        for cf in coef_high_first[1:]:
            p = (p.astype(np.float64) * s.astype(np.float64) + np.float64(np.float32(cf))).astype(np.float32)
        v = (t32.astype(np.float64) * p.astype(np.float64)).astype(np.float32).astype(np.float64)
        ref = np.arctan(t32.astype(np.float64))
    else:
        s = t * t
        v = t * np.polyval(np.asarray(coef_high_first, dtype=np.float64), s)
        ref = np.arctan(t)
    rel = v / ref - 1.0
    return float(np.max(np.abs(rel))), float(np.mean(rel))


def main():
    for name, a, deg in (("atan_unit", 1.0, 7), ("small-angle series", 16.0 / 63.0, 4)):
        c = remez(a, deg)
        c32 = [float(np.float32(v)) for v in c[::-1]]
        e64, _ = max_rel_error(list(c[::-1]), a)
        e, bias = max_rel_error(c32, a)
        e32, _ = max_rel_error(c32, a, fp32=True)
        print(f"{name}: |t| <= {a:.6g}, degree {deg} in t^2")
        print("  coefficients (highest degree first):", ", ".join(f"{v:.17g}f" for v in c32))
        print(f"  max relative error: {e64:.3g} (FP64 coefficients), {e:.3g} (FP32 coefficients, mean signed "
              f"{bias:.2g}), {e32:.3g} (evaluated in FP32)")
    c, e = interpolate_f64(np.tan(4 * np.arctan(1 / 16)), 7)
    print("FP64 series, Q highest degree first:", ", ".join(repr(float(v)) for v in c[::-1]))
    print(f"  max relative error: {e:.3g}")


if __name__ == "__main__":
    main()
