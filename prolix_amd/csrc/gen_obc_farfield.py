"""Generate prx_obc_farfield.h: polynomial forms of the OBC2 pair integral in the far field.

When the descreening sphere of atom j lies wholly outside atom i's offset
sphere (r - s >= rho, with s = sr_j and rho = rho_i), the pair integral of
prolix's generalized_born.py:211-263 has L = r - s and U = r + s, and its
three terms collapse to

    I = (1 / 2r) [x / (1 - x^2) - atanh(x)],   x = s / r
      = (x^3 / 2r) h(x^2),   h(y) = sum_{k>=1} 2k / (2k+1) y^(k-1)

    dI/dr = -(x^3 / r^2) k(x^2),   k(y) = 2 h(y) + y h'(y) = sum_{k>=1} 2k(k+1) / (2k+1) y^(k-1)

The direct formula subtracts terms of size ~s/r^2 to get a result of size
~s^3/r^4, so in float32 it loses about log10((r/s)^2) digits; the series form
has only positive terms. h and k are fitted on y in [0, Y_MAX] and written out in
the power basis of y for Horner evaluation. The leading coefficients, all that
counts far away, are held at 2/3 and 4/3: the kernels scale them to 1 and -4 and put
the atom's s^3/3 in front, which is rounded once. What is left, (h(y) - 2/3) / y
and (k(y) - 4/3) / y, is fitted so that the largest relative error of the whole is as small as
it can be (Lawson's reweighted least squares). The errors written beside them
are those of the float32 coefficients that the kernels run: 3.1e-8 and 1.2e-8,
under float32's unit roundoff of 6e-8. Y_MAX = 0.25 (s <= r/2) rather than a
wider range keeps the degrees at 6 and 7: on compact proteins, r - s > rho
already implies s < 0.6 r, and s <= r/2 excludes under 0.5% of the pairs.

A second pair of fits covers y in [0, Y_MAX4] (s <= r/4) at degree 4 for
both (relative error 4.4e-9 and 1.3e-8): the pair kernels use them for work
items whose tiles are at least 4 s apart in every pair, where they save two
and three multiply-adds per direction. Two more pairs do the same further out:
degree 3 for s <= r/6.5 (4.7e-9 and 1.3e-8) and degree 2 for s <= r/14.5
(5.6e-9 and 1.4e-8), so with the distance of two tiles the polynomials get
shorter, and each stays a fourth of a unit roundoff at most from the series.

Run: python prolix_amd/csrc/gen_obc_farfield.py > prolix_amd/csrc/prx_obc_farfield.h
"""

import numpy as np

Y_MAX = 0.25  # x <= 0.5
DEG_H = 6
DEG_K = 7
Y_MAX4 = 0.0625  # x <= 0.25
DEG_H4 = 4
DEG_K4 = 4
# (suffix, smallest r / s, degree of h and of k)
SHORTER = ((3, 6.5, 3), (2, 14.5, 2))


def h_series(y):
    return sum(2 * k / (2 * k + 1) * y ** (k - 1) for k in range(1, 400))


def k_series(y):
    return sum(2 * k * (k + 1) / (2 * k + 1) * y ** (k - 1) for k in range(1, 400))


def fit(fn, deg, y_max, scale):
    """Coefficients of fn(0) + y g(y), and the relative error of their float32
    multiples by scale."""
    t = -np.cos(np.pi * (np.arange(2001) + 0.5) / 2001)  # Chebyshev nodes
    y = 0.5 * y_max * (1 + t)
    f, f0 = fn(y), float(fn(np.zeros(1))[0])
    basis = np.polynomial.chebyshev.chebvander(t, deg - 1) * (y / f)[:, None]
    w = np.ones_like(y)
    for _ in range(400):
        s = np.sqrt(w)
        c = np.linalg.lstsq(basis * s[:, None], (f - f0) / f * s, rcond=None)[0]
        w *= np.abs(basis @ c - (f - f0) / f)
        w = np.maximum(w / w.max(), 1e-12)
    g = np.polynomial.Polynomial(np.polynomial.chebyshev.cheb2poly(c))(np.polynomial.Polynomial([-1.0, 2.0 / y_max]))
    coef = np.concatenate([[f0], g.coef])
    yy = np.linspace(0.0, y_max, 40001)
    run = np.float32(scale * coef).astype(np.float64)
    err = float(np.max(np.abs(np.polynomial.polynomial.polyval(yy, run) / (scale * fn(yy)) - 1.0)))
    return coef, err


def fit_h(deg, y_max):
    return fit(h_series, deg, y_max, 1.5)


def fit_k(deg, y_max):
    return fit(k_series, deg, y_max, -3.0)


def main():
    ch, eh = fit_h(DEG_H, Y_MAX)
    ck, ek = fit_k(DEG_K, Y_MAX)
    ch4, eh4 = fit_h(DEG_H4, Y_MAX4)
    ck4, ek4 = fit_k(DEG_K4, Y_MAX4)
    fmt = lambda c: ", ".join(f"{v:.17g}" for v in c)
    print("// Generated by gen_obc_farfield.py -- do not edit by hand.")
    print("// Far-field OBC2 pair integral polynomials in y = (s/r)^2 on [0, %g]." % Y_MAX)
    print(f"// max relative error: h {eh:.2e}, k {ek:.2e}")
    print("#pragma once")
    print(f"#define PRX_OBC_FAR_YMAX {Y_MAX}f")
    print(f"#define PRX_OBC_FAR_XMAX {np.sqrt(Y_MAX):.9g}f")
    print(f"constexpr int kObcHDeg = {DEG_H};")
    print(f"__device__ constexpr double kObcH[{DEG_H + 1}] = {{{fmt(ch)}}};")
    print(f"constexpr int kObcKDeg = {DEG_K};")
    print(f"__device__ constexpr double kObcK[{DEG_K + 1}] = {{{fmt(ck)}}};")
    print("// The same on [0, %g] (s <= r/4); max relative error: h %.2e, k %.2e" % (Y_MAX4, eh4, ek4))
    print(f"#define PRX_OBC_FAR4_YMAX {Y_MAX4}f")
    print(f"#define PRX_OBC_FAR4_XMAX {np.sqrt(Y_MAX4):.9g}f")
    print(f"constexpr int kObcH4Deg = {DEG_H4};")
    print(f"__device__ constexpr double kObcH4[{DEG_H4 + 1}] = {{{fmt(ch4)}}};")
    print(f"constexpr int kObcK4Deg = {DEG_K4};")
    print(f"__device__ constexpr double kObcK4[{DEG_K4 + 1}] = {{{fmt(ck4)}}};")
    for n, ratio, deg in SHORTER:
        h, eh = fit_h(deg, 1.0 / ratio**2)
        k, ek = fit_k(deg, 1.0 / ratio**2)
        print("// The same for s <= r/%g; max relative error: h %.2e, k %.2e" % (ratio, eh, ek))
        print(f"#define PRX_OBC_FAR{n}_XMAX {1.0 / ratio:.9g}f")
        print(f"constexpr int kObcH{n}Deg = {deg}, kObcK{n}Deg = {deg};")
        print(f"__device__ constexpr double kObcH{n}[{deg + 1}] = {{{fmt(h)}}};")
        print(f"__device__ constexpr double kObcK{n}[{deg + 1}] = {{{fmt(k)}}};")


if __name__ == "__main__":
    main()
