// Frequency-domain interpolated sum: the stationary-phase approximation of
// every (mode, knot segment) evaluated at every frequency bin the segment's
// mode frequency sweeps over (get_waveform_generic_fd,
// src/few/cutils/interpolate.cu:1142-1563).
//
// Per bin f of item (mode q, segment j) -- interpolate.cu:1396-1500:
//   * the times where the mode frequency F(x) = m f_phi + k f_theta + n f_r
//     (cubic in x = t - t_j) equals f: Cardano's roots of
//     F3 x^3 + F2 x^2 + F1 x + (F0 - f), keeping the real part of each of the
//     three complex roots and every one that falls inside the segment;
//   * at such a time t: amplitude A(x), phase Phi(t) and its first two time
//     derivatives from the dense-output form, and
//       h(f) += Y+ A T(fdot, fddot) e^{i(2 pi f t - Phi)},
//       h(-f) += [m != 0] Y- conj(A T e^{...})      (bin 2 zero - i)
//     with T = -fdot/|fddot| (2/sqrt 3) SPA(x) / sqrt(x),
//     x = 2 pi fdot^3 / (3 fddot^2) and SPA(x) = i sqrt(x) e^{-ix} K_1/3(-ix).
//
// Layout of the work (summed output): bin-owned.  Each lane owns a bin and
// its mirror about the zero bin, a workgroup a tile of such owners; the
// segments that reach the tile are found per cell by binary search over the
// cell's segments sorted by first bin, and each lane adds every
// contribution to its bins itself, in a fixed order (cell, sorted segment,
// root): no atomics, and the result is the same on every run (the
// reference's kernel adds with atomic CAS loops in no fixed order).  With
// separate_modes every (mode, bin) has one writer already: the (mode,
// segment) items are flattened, their in-range bin counts prefix-summed on
// the device, and a persistent grid walks the flattened bins.
//
// The kernels evaluate fd_bin_fast, a shorter form of the reference's bin
// (interpolate.cu:1240-1500), with contraction off in the whole file.  The complex
// arithmetic of its rare branches and constants follows gcmplx::complex
// (src/few/cutils/cuda_complex.hpp, the libc++ <complex> algorithms) operation for
// operation, on the device's FP64 libm; the products keep their C99 Annex G NaN
// recovery.  cos and sin of one argument are taken with one sincos call, as an
// optimising compiler emits for gcmplx::exp / polar.
#include <math.h>

#include <algorithm>

#include "cells.hpp"
#include "fd.hpp"
#include "few_common.hpp"
#include "few_math.hpp"

#pragma clang fp contract(off)

namespace few {

struct fcx {
    double re, im;
};

__host__ __device__ inline fcx fcx_make(double re, double im)
{
    fcx z;
    z.re = re;
    z.im = im;
    return z;
}

// cuda_complex.hpp:440-498
__host__ __device__ inline fcx fcx_mul(fcx z, fcx w)
{
#pragma clang fp contract(off)
    double a = z.re, b = z.im, c = w.re, d = w.im;
    const double ac = a * c, bd = b * d, ad = a * d, bc = b * c;
    double x = ac - bd, y = ad + bc;
    if (isnan(x) && isnan(y)) {
        bool recalc = false;
        if (isinf(a) || isinf(b)) {
            a = copysign(isinf(a) ? 1.0 : 0.0, a);
            b = copysign(isinf(b) ? 1.0 : 0.0, b);
            if (isnan(c)) c = copysign(0.0, c);
            if (isnan(d)) d = copysign(0.0, d);
            recalc = true;
        }
        if (isinf(c) || isinf(d)) {
            c = copysign(isinf(c) ? 1.0 : 0.0, c);
            d = copysign(isinf(d) ? 1.0 : 0.0, d);
            if (isnan(a)) a = copysign(0.0, a);
            if (isnan(b)) b = copysign(0.0, b);
            recalc = true;
        }
        if (!recalc && (isinf(ac) || isinf(bd) || isinf(ad) || isinf(bc))) {
            if (isnan(a)) a = copysign(0.0, a);
            if (isnan(b)) b = copysign(0.0, b);
            if (isnan(c)) c = copysign(0.0, c);
            if (isnan(d)) d = copysign(0.0, d);
            recalc = true;
        }
        if (recalc) {
            x = INFINITY * (a * c - b * d);
            y = INFINITY * (a * d + b * c);
        }
    }
    return fcx_make(x, y);
}

// complex (*, /) real component-wise; real + complex adds to the real part
__host__ __device__ inline fcx fcx_scale(fcx z, double s) { return fcx_make(z.re * s, z.im * s); }
__host__ __device__ inline fcx fcx_divr(fcx z, double s) { return fcx_make(z.re / s, z.im / s); }
__host__ __device__ inline fcx fcx_add(fcx z, fcx w) { return fcx_make(z.re + w.re, z.im + w.im); }
__host__ __device__ inline fcx fcx_addr(double r, fcx z) { return fcx_make(z.re + r, z.im); }

// cuda_complex.hpp operator/(complex, complex): logb/scalbn-scaled quotient
__host__ __device__ inline fcx fcx_div(fcx z, fcx w)
{
#pragma clang fp contract(off)
    int ilogbw = 0;
    double a = z.re, b = z.im, c = w.re, d = w.im;
    const double logbw = logb(fmax(fabs(c), fabs(d)));
    if (isfinite(logbw)) {
        ilogbw = (int)logbw;
        c = scalbn(c, -ilogbw);
        d = scalbn(d, -ilogbw);
    }
    const double denom = c * c + d * d;
    double x = scalbn((a * c + b * d) / denom, -ilogbw);
    double y = scalbn((b * c - a * d) / denom, -ilogbw);
    if (isnan(x) && isnan(y)) {
        if ((denom == 0.0) && (!isnan(a) || !isnan(b))) {
            x = copysign(INFINITY, c) * a;
            y = copysign(INFINITY, c) * b;
        } else if ((isinf(a) || isinf(b)) && isfinite(c) && isfinite(d)) {
            a = copysign(isinf(a) ? 1.0 : 0.0, a);
            b = copysign(isinf(b) ? 1.0 : 0.0, b);
            x = INFINITY * (a * c + b * d);
            y = INFINITY * (b * c - a * d);
        } else if (isinf(logbw) && logbw > 0.0 && isfinite(a) && isfinite(b)) {
            c = copysign(isinf(c) ? 1.0 : 0.0, c);
            d = copysign(isinf(d) ? 1.0 : 0.0, d);
            x = 0.0 * (a * c + b * d);
            y = 0.0 * (b * c - a * d);
        }
    }
    return fcx_make(x, y);
}

__host__ __device__ inline double fcx_abs(fcx z) { return hypot(z.re, z.im); }
__host__ __device__ inline double fcx_arg(fcx z) { return atan2(z.im, z.re); }

// cuda_complex.hpp:864-893
__host__ __device__ inline fcx fcx_polar(double rho, double theta)
{
#pragma clang fp contract(off)
    if (isnan(rho) || signbit(rho)) return fcx_make(NAN, NAN);
    if (isnan(theta)) {
        if (isinf(rho)) return fcx_make(rho, theta);
        return fcx_make(theta, theta);
    }
    if (isinf(theta)) {
        if (isinf(rho)) return fcx_make(rho, NAN);
        return fcx_make(NAN, NAN);
    }
    double sn, cs;
    sincos(theta, &sn, &cs);
    double x = rho * cs;
    if (isnan(x)) x = 0;
    double y = rho * sn;
    if (isnan(y)) y = 0;
    return fcx_make(x, y);
}

__host__ __device__ inline fcx fcx_log(fcx z) { return fcx_make(log(fcx_abs(z)), fcx_arg(z)); }

// cuda_complex.hpp:914-930
__host__ __device__ inline fcx fcx_sqrt(fcx z)
{
    if (isinf(z.im)) return fcx_make(INFINITY, z.im);
    if (isinf(z.re)) {
        if (z.re > 0.0) return fcx_make(z.re, isnan(z.im) ? z.im : copysign(0.0, z.im));
        return fcx_make(isnan(z.im) ? z.im : 0.0, copysign(z.re, z.im));
    }
    return fcx_polar(sqrt(fcx_abs(z)), fcx_arg(z) / 2.0);
}

// cuda_complex.hpp:934-958
__host__ __device__ inline fcx fcx_exp(fcx z)
{
#pragma clang fp contract(off)
    double i = z.im;
    if (isinf(z.re)) {
        if (z.re < 0.0) {
            if (!isfinite(i)) i = 1.0;
        } else if (i == 0 || !isfinite(i)) {
            if (isinf(i)) i = NAN;
            return fcx_make(z.re, i);
        }
    } else if (isnan(z.re) && z.im == 0) {
        return z;
    }
    const double e = exp(z.re);
    double sn, cs;
    sincos(i, &sn, &cs);
    return fcx_make(e * cs, e * sn);
}

// cuda_complex.hpp:960-976: pow(x, y) = exp(complex(y) * log(x))
__host__ __device__ inline fcx fcx_pow(fcx x, double y)
{
    return fcx_exp(fcx_mul(fcx_make(y, 0.0), fcx_log(x)));
}

// The argument-independent factors of SPAFunc: exp(-2 pi i / 3), exp(-pi i / 3)
// and exp(-3 pi i / 4) sqrt(pi / 2), computed once per thread with the same
// operations the reference repeats on every call.
struct FdSpaConst {
    fcx e1, e2, pref_asym;
};

__host__ __device__ inline FdSpaConst fd_spa_const()
{
    const fcx II = fcx_make(0.0, 1.0);
    FdSpaConst k;
    k.e1 = fcx_exp(fcx_divr(fcx_scale(II, -2. * M_PI), 3.));
    k.e2 = fcx_exp(fcx_divr(fcx_scale(II, -M_PI), 3.));
    k.pref_asym = fcx_scale(fcx_exp(fcx_scale(fcx_scale(II, -0.75), M_PI)), sqrt(0.5 * M_PI));
    return k;
}

// SPAFunc (interpolate.cu:1041-1090): i sqrt(x) e^{-ix} K_1/3(-ix) by its
// small-argument series (|x| <= 7) or its asymptotic series.
__host__ __device__ inline fcx fd_spa(double x, const FdSpaConst &kc)
{
#pragma clang fp contract(off)
    const fcx II = fcx_make(0.0, 1.0);
    const double Gamp13 = 2.67893853470774763;   // Gamma(1/3)
    const double Gamm13 = -4.06235381827920125;  // Gamma(-1/3)
    if (fabs(x) <= 7.) {
        const fcx tmp_p = fcx_pow(fcx_make(x, 0.0), 1. / 6.);
        fcx pref1 = fcx_mul(kc.e1, tmp_p);
        pref1 = fcx_mul(pref1, tmp_p);
        pref1 = fcx_mul(pref1, tmp_p);
        pref1 = fcx_mul(pref1, tmp_p);
        pref1 = fcx_mul(pref1, tmp_p);
        pref1 = fcx_divr(fcx_scale(pref1, Gamm13), 1.2599210498948732);  // 2^(1/3)
        fcx pref2 = fcx_mul(kc.e2, tmp_p);
        pref2 = fcx_divr(fcx_scale(pref2, Gamp13), 1.5874010519681994748);  // 2^(2/3)
        const double x2 = x * x;
        // Taylor coefficients of the two Bessel-series factors (even powers)
        const double ser1 = 0.5 + x2 * (-0.09375 + x2 * (0.0050223214285714285714 + x2 * (-0.00012555803571428571429 + x2 * (1.8109332074175824176e-6 + x2 * (-1.6977498819539835165e-8 + x2 * (1.1169407118118312608e-10 + x2 * (-5.4396463237589184781e-13 + x2 * (2.0398673714095944293e-15 + x2 * (-6.0710338434809358015e-18 + x2 * (1.4687985105195812423e-20 + x2 * (-2.9454515585285720100e-23 + x2 * (4.9754249299469121790e-26 + x2 * -7.1760936489618925658e-29))))))))))));
        const double ser2 = 1. + x2 * (-0.375 + x2 * (0.028125 + x2 * (-0.00087890625 + x2 * (0.000014981356534090909091 + x2 * (-1.6051453429383116883e-7 + x2 * (1.1802539286311115355e-9 + x2 * (-6.3227889033809546546e-12 + x2 * (2.5772237377911499951e-14 + x2 * (-8.2603324929203525483e-17 + x2 * (2.1362928861000911763e-19 + x2 * (-4.5517604107246260858e-22 + x2 * (8.1281435905796894390e-25 + x2 * -1.2340298973552160079e-27))))))))))));
        const fcx ex = fcx_exp(fcx_scale(fcx_make(-II.re, -II.im), x));
        return fcx_mul(ex, fcx_add(fcx_scale(pref1, ser1), fcx_scale(pref2, ser2)));
    }
    const fcx y = fcx_make(1. / x, 0.0);
    const fcx pref = kc.pref_asym;
    // asymptotic series c_0 + y (c_1 + ... + y c_8): alternating imaginary/real terms
    fcx ser = fcx_add(fcx_make(-0.87766696951001691647, 0.0), fcx_mul(y, fcx_scale(II, 3.0794530301731669934)));
    ser = fcx_add(fcx_scale(II, -0.29159139923075051147), fcx_mul(y, ser));
    ser = fcx_add(fcx_make(0.11609906402551541102, 0.0), fcx_mul(y, ser));
    ser = fcx_add(fcx_scale(II, 0.057649190412669721333), fcx_mul(y, ser));
    ser = fcx_add(fcx_make(-0.037993059127800640146, 0.0), fcx_mul(y, ser));
    ser = fcx_add(fcx_scale(II, -0.037133487654320987654), fcx_mul(y, ser));
    ser = fcx_add(fcx_make(0.069444444444444444444, 0.0), fcx_mul(y, ser));
    ser = fcx_add(II, fcx_mul(y, ser));
    return fcx_mul(pref, ser);
}

__host__ __device__ inline fcx fd_xi()
{
    return fcx_divr(fcx_addr(-1., fcx_sqrt(fcx_make(-3., 0.0))), 2.);
}

__host__ __device__ inline double fd_phase(const double *r, double s, double s1)
{
#pragma clang fp contract(off)
    return r[0] + s * (r[1] + s1 * (r[2] + s * (r[3] + s1 * (r[4] + s * (r[5] + s1 * (r[6] + s * r[7]))))));
}

// ---------------------------------------------------------------- fast form
// What the kernels evaluate: the same roots, phase and stationary-phase factor
// as the reference's bin, without the complex library calls on numbers that are
// real or purely imaginary and with everything that depends on the segment alone
// formed once per segment.  The reference's operations one for one take ~2300
// instructions per bin, this form ~600.  What keeps the two close:
//   * the time of a root decides 2 pi f t - phase, of which an ulp of t is
//     ~1e-11 at 1e5 rad, so the roots are cube_roots' (interpolate.cu:1113-1134) own
//     values, 98 % of them bit for bit: Cardano's formula with the principal complex
//     cube root in the same operations, only that the discriminant is real
//     (its square root and, unless it is negative, the cube root need no hypot,
//     atan2 or sincos), that |C|^2 >= 1e-216 needs no scaling in D0 / C, and
//     that roots outside the segment (by a quotient shared by the three, with
//     a margin) are dropped before theirs is formed;
//   * s and the phases are the reference's values (s by a correctly rounded quotient);
//   * the frequency's derivatives enter the amplitude only, so they are
//     polynomials in s with fused steps.

// Everything an evaluation of one (cell or mode, segment) reads.  The first 40
// doubles depend on both, the last 32 on the segment only.
struct FdSeg {
    double tab[16];               // the cell's cubics: (Re C+, Im C+, Re C-, Im C-) of power 0..3
    double F0, b, D0, D03, D1c, a27;  // frequency cubic: F0, F2, Cardano's D0, 4 D0^3, D1 = D1c + a27 d
    double a;                     // -1 / (3 F3)
    double f[6], g[5];            // fdot and fddot as polynomials in s
    double mm, kk, nn;
    double theta;                 // 1: Phi_theta enters the phase
    double pad[2];
    double pp[8], pt[8], pr[8];   // dense-output phases
    double t0, t1, pt0, pw, rpw;  // segment bounds, phase segment start, width, 1 / width
    double pad2[3];
};
constexpr int FD_CELL_DOUBLES = 40, FD_SEG_DOUBLES = 32;
static_assert(sizeof(FdSeg) == sizeof(double) * (FD_CELL_DOUBLES + FD_SEG_DOUBLES), "FdSeg layout");

__host__ __device__ inline void fd_load_seg(const FdArgs &a, int q, int j, FdSeg &it)
{
    const long nb = (2L * a.K + 3) * a.L;
    const long np = (long)(a.L - 1) * 3;
    double fph[4], fth[4], frr[4], r[8];
    const int m = a.m[q], k = a.k[q], n = a.n[q];
    it.mm = m;
    it.kk = k;
    it.nn = n;
#pragma unroll
    for (int c = 0; c < 4; c++) {
        fph[c] = a.interp[c * nb + (long)(2 * a.K) * a.L + j];
        fth[c] = a.interp[c * nb + (long)(2 * a.K + 1) * a.L + j];
        frr[c] = a.interp[c * nb + (long)(2 * a.K + 2) * a.L + j];
    }
    double fin = 0.0;
#pragma unroll
    for (int c = 0; c < 8; c++) {
        it.pp[c] = a.pcoef[c * np + j];
        it.pt[c] = a.pcoef[c * np + (a.L - 1) + j];
        it.pr[c] = a.pcoef[c * np + 2 * (a.L - 1) + j];
        fin += 0.0 * it.pt[c];
        r[c] = it.mm * it.pp[c] + it.kk * it.pt[c] + it.nn * it.pr[c];
    }
    // k = 0: 0 * Phi_theta adds nothing unless it is not finite
    it.theta = k != 0 || fin != 0.0 ? 1.0 : 0.0;
    it.F0 = m * fph[0] + k * fth[0] + n * frr[0];
    const double F1 = m * fph[1] + k * fth[1] + n * frr[1];
    const double F2 = m * fph[2] + k * fth[2] + n * frr[2];
    const double F3 = m * fph[3] + k * fth[3] + n * frr[3];
    // the cubic (F3, F2, F1, F0 - f), what does not depend on f
    const double b2 = F2 * F2;
    const double b3 = b2 * F2;
    const double a2 = F3 * F3;
    it.b = F2;
    it.D0 = (b2 - 3 * F3 * F1);
    it.D03 = 4 * (it.D0 * it.D0 * it.D0);
    it.D1c = 2 * b3 - 9 * F3 * F2 * F1;
    it.a27 = 27 * a2;
    it.a = -(1. / (3 * F3));
    it.t0 = a.t_knots[j];
    it.t1 = a.t_knots[j + 1];
    it.pt0 = a.phase_t[j];
    it.pw = a.phase_t[j + 1] - a.phase_t[j];
    it.rpw = 1.0 / it.pw;
    // the second derivative of the phases over 2 pi by powers of s (interpolate.cu's
    // fdot), then its derivative over pw (fddot)
    const double w = 1.0 / (2. * M_PI * (it.pw * it.pw));
    it.f[0] = (2. * (r[3] - r[2] + r[4])) * w;
    it.f[1] = (6. * (r[5] + r[6] - r[3]) - 12. * r[4]) * w;
    it.f[2] = (12. * (r[4] + r[7]) - 24. * r[5] - 36. * r[6]) * w;
    it.f[3] = (20. * r[5] + 60. * (r[6] - r[7])) * w;
    it.f[4] = (90. * r[7] - 30. * r[6]) * w;
    it.f[5] = -42. * r[7] * w;
#pragma unroll
    for (int c = 0; c < 5; c++) it.g[c] = (c + 1) * it.f[c + 1] * it.rpw;
}

// The rare branches, kept out of line: inlined, their library calls set the
// kernel's registers.
__host__ __device__ __attribute__((noinline)) fcx fd_sincos_any(double x)
{
    fcx r;
    sincos(x, &r.im, &r.re);
    return r;
}
// pre SPA(x) / sqrt(x) from the two derivatives, as the reference forms it
__host__ __device__ __attribute__((noinline)) fcx fd_amp_any(double fdot, double fddot,
                                                            const FdSpaConst kc)
{
    const double targ = 2. * M_PI * fdot * fdot * fdot / (3. * fddot * fddot);
    const double pre = -1.0 * fdot / fabs(fddot) * 2. / sqrt(3.);
    return fcx_div(fcx_scale(fd_spa(targ, kc), pre), fcx_sqrt(fcx_make(targ, 0.0)));
}

// 1 / sqrt(x) for a normal x: the hardware's estimate and two Newton steps.
__host__ __device__ inline double fd_rsqrt(double x)
{
#if defined(__HIP_DEVICE_COMPILE__)
    double r = __builtin_amdgcn_rsq(x);
#pragma unroll
    for (int i = 0; i < 2; i++) r = fma(0.5 * r, fma(-x * r, r, 1.0), r);
    return r;
#else
    return 1.0 / sqrt(x);
#endif
}

// The stationary-phase factor pre SPA(x) / sqrt(x), x = 2 pi fdot^3 / (3 fddot^2),
// pre = -2 fdot / (sqrt(3) |fddot|).  Beyond |x| = 7 (fd_spa's asymptotic series,
// whose powers of i alternate between real and imaginary terms) fddot cancels
// out of the prefactor: pre / sqrt|x| = -+ 2 / sqrt(2 pi |fdot|), and
// 1 / x = 3 fddot^2 / (2 pi fdot^3) needs no quotient either.
__host__ __device__ inline fcx fd_amp(double fdot, double fddot, const FdSpaConst &kc)
{
    const double rs = fd_rsqrt(fabs(fdot)), rs2 = rs * rs;
    const double v2 = fddot * rs2;
    const double y = copysign((3. / (2. * M_PI)) * (v2 * v2) * rs2, fdot);
    // |y| up to 1/7 within rounding; 0, infinities and NaN: the general form
    if (!(fabs(y) < 0.14285714285714 && fabs(y) > 0.0 && rs < 1e150)) return fd_amp_any(fdot, fddot, kc);
    const double y2 = y * y;
    const double im = fma(y2, fma(y2, fma(y2, fma(y2, 3.0794530301731669934, -0.29159139923075051147), 0.057649190412669721333), -0.037133487654320987654), 1.);
    const double re = y * fma(y2, fma(y2, fma(y2, -0.87766696951001691647, 0.11609906402551541102), -0.037993059127800640146), 0.069444444444444444444);
    const double sq = -copysign(rs * 0.79788456080286535588, fdot);  // 2 / sqrt(2 pi)
    const fcx v = fcx_make((kc.pref_asym.re * re - kc.pref_asym.im * im) * sq,
                           (kc.pref_asym.re * im + kc.pref_asym.im * re) * sq);
    return fdot > 0.0 ? v : fcx_make(v.im, -v.re);  // sqrt of a negative number: i sqrt(|x|)
}

// Constants of the roots: xi, xi^2, cos of the halved argument of a negative
// number, cos and sin of a third of it (as fcx_sqrt and fcx_pow round them).
struct FdRootConst {
    fcx xi, xixi;
    double cos_half, cos_third, sin_third;
};

__host__ __device__ inline FdRootConst fd_root_const()
{
    FdRootConst k;
    k.xi = fd_xi();
    k.xixi = fcx_mul(k.xi, k.xi);
    double sn;
    sincos(M_PI / 2.0, &sn, &k.cos_half);
    sincos((1. / 3.) * M_PI, &k.sin_third, &k.cos_third);
    return k;
}

// C, C xi and C xi^2 of the cubic at d = F0 - f, xi = (-1 + sqrt(-3)) / 2.
__host__ __device__ inline void fd_cube_c(const FdSeg &it, double d, const FdRootConst &k, fcx (&C)[3])
{
    const double D1 = (it.D1c + it.a27 * d);
    const double D = D1 * D1 - it.D03;
    const double rho = sqrt(fabs(D));
    const bool neg = D < 0.0;
    const double zr = (D1 + (neg ? rho * k.cos_half : rho)) / 2., zi = rho / 2.;
    const double e = exp((1. / 3.) * log(neg ? hypot(zr, zi) : fabs(zr)));
    double sn = zr < 0.0 ? k.sin_third : 0.0, cs = zr < 0.0 ? k.cos_third : 1.0;
    if (neg) {
        // a third of an angle in [0, pi]: no reduction, and no library large-argument code
        const double th = (1. / 3.) * atan2(zi, zr);
        sincos_half_turns(th, sn, cs);
    }
    C[0] = fcx_make(e * cs, e * sn);
    C[1] = fcx_make(k.xi.re * C[0].re - k.xi.im * C[0].im, k.xi.re * C[0].im + k.xi.im * C[0].re);
    C[2] = fcx_make(k.xixi.re * C[0].re - k.xixi.im * C[0].im,
                    k.xixi.re * C[0].im + k.xixi.im * C[0].re);
}

// Real part of the root of C: -(b + C + D0 / C) / (3 a).
__host__ __device__ inline double fd_root_of(const FdSeg &it, fcx C)
{
    return ((C.re + it.b) + it.D0 * C.re / (C.re * C.re + C.im * C.im)) * it.a;
}

// Bin of frequency f: emit(x, B) for every root inside the segment, in root
// order, x the time since its start and B the stationary-phase factor times
// exp(i (2 pi f t - phase)), so that the +f term is Y+ A(x) B.
template <class Emit>
__host__ __device__ inline void fd_bin_fast(const FdSeg &it, double f, const FdRootConst &kr,
                                            const FdSpaConst &kc, Emit emit)
{
    fcx C[3];
    fd_cube_c(it, it.F0 - f, kr, C);
    // the three roots to ~1e-14 of their largest term with one quotient (|C| is
    // common to them); a margin of 1e-10 of it decides which are formed exactly
    const double c2 = C[0].re * C[0].re + C[0].im * C[0].im;
    const double q = 1.0 + it.D0 / c2;
    const double span = it.t1 - it.t0;
    const double tol = 1e-10 * (fabs(it.a) * (fabs(it.b) + sqrt(c2) * (1.0 + fabs(q))) + fabs(it.t1));
    unsigned cand = 0;
#pragma unroll
    for (int r = 0; r < 3; r++) {
        const double x = fma(C[r].re, q, it.b) * it.a;
        if (x > -tol && x < span + tol) cand |= 1u << r;
    }
#pragma nounroll
    while (cand) {
        const double cre = (cand & 1u) ? C[0].re : ((cand & 2u) ? C[1].re : C[2].re);
        const double cim = (cand & 1u) ? C[0].im : ((cand & 2u) ? C[1].im : C[2].im);
        cand &= cand - 1u;
        const double root = fd_root_of(it, fcx_make(cre, cim));
        const double t = it.t0 + root;
        if (!((t < it.t1) && (t >= it.t0))) continue;
        // (t - pt0) / pw correctly rounded (one residual step on x * RN(1 / pw))
        const double xs = t - it.pt0;
        const double s0 = xs * it.rpw;
        const double s = fma(fma(-s0, it.pw, xs), it.rpw, s0);
        const double s1 = 1.0 - s;
        const double Pp = fd_phase(it.pp, s, s1), Pr = fd_phase(it.pr, s, s1);
        const double phase = it.theta != 0.0
                                 ? it.mm * Pp + it.kk * fd_phase(it.pt, s, s1) + it.nn * Pr
                                 : it.mm * Pp + it.nn * Pr;
        double fdot = it.f[5], fddot = it.g[4];
#pragma unroll
        for (int c = 4; c >= 0; c--) fdot = fma(fdot, s, it.f[c]);
#pragma unroll
        for (int c = 3; c >= 0; c--) fddot = fma(fddot, s, it.g[c]);
        const fcx amp = fd_amp(fdot, fddot, kc);
        double sn, cs;
        const double arg = 2. * M_PI * f * t - phase;
        if (!sincos_half_turns(arg, sn, cs)) {
            const fcx any = fd_sincos_any(arg);
            sn = any.im;
            cs = any.re;
        }
        emit(root, fcx_make(fma(amp.re, cs, -amp.im * sn), fma(amp.re, sn, amp.im * cs)));
    }
}

// Power p of the combined cubics of one cell: C+ = sum Y+ A, C- = sum Y- conj(A).
__host__ __device__ inline void fd_cell_add(double a_re, double a_im, double2 yp, double2 ym, fcx &cp,
                                            fcx &cm)
{
    cp.re += yp.x * a_re - yp.y * a_im;
    cp.im += yp.x * a_im + yp.y * a_re;
    cm.re += ym.x * a_re + ym.y * a_im;
    cm.im += ym.y * a_re - ym.x * a_im;
}

// In-range bins of item (q, j): [max(start, 0), min(end, Nf - 1)].
__host__ __device__ inline void fd_item_range(const FdArgs &a, long item, int &lo, int &hi)
{
    lo = a.seg_start[item];
    hi = a.seg_end[item];
    if (lo < 0) lo = 0;
    if (hi > a.data_length - 1) hi = a.data_length - 1;
}

#define FD_SCAN_BLOCK 1024

// Block-local exclusive scan of the per-item bin counts.
__global__ __launch_bounds__(FD_SCAN_BLOCK) void fd_scan1_kernel(FdArgs a, long nitems, long *local,
                                                                 long *bsum)
{
    __shared__ long s[FD_SCAN_BLOCK];
    const int tid = threadIdx.x;
    const long q = (long)blockIdx.x * FD_SCAN_BLOCK + tid;
    long c = 0;
    if (q < nitems) {
        int lo, hi;
        fd_item_range(a, q, lo, hi);
        c = hi >= lo ? (long)(hi - lo + 1) : 0;
    }
    s[tid] = c;
    __syncthreads();
    for (int off = 1; off < FD_SCAN_BLOCK; off <<= 1) {
        const long v = tid >= off ? s[tid - off] : 0;
        __syncthreads();
        s[tid] += v;
        __syncthreads();
    }
    if (q < nitems) local[q] = s[tid] - c;
    if (tid == FD_SCAN_BLOCK - 1) bsum[blockIdx.x] = s[tid];
}

// Exclusive scan of the block sums (one workgroup, sequential over chunks).
__global__ __launch_bounds__(FD_SCAN_BLOCK) void fd_scan2_kernel(long *bsum, long nb, long *total)
{
    __shared__ long s[FD_SCAN_BLOCK];
    __shared__ long carry;
    const int tid = threadIdx.x;
    if (tid == 0) carry = 0;
    __syncthreads();
    for (long b0 = 0; b0 < nb; b0 += FD_SCAN_BLOCK) {
        const long b = b0 + tid;
        const long v0 = b < nb ? bsum[b] : 0;
        s[tid] = v0;
        __syncthreads();
        for (int off = 1; off < FD_SCAN_BLOCK; off <<= 1) {
            const long v = tid >= off ? s[tid - off] : 0;
            __syncthreads();
            s[tid] += v;
            __syncthreads();
        }
        if (b < nb) bsum[b] = carry + s[tid] - v0;
        __syncthreads();
        if (tid == FD_SCAN_BLOCK - 1) carry += s[tid];
        __syncthreads();
    }
    if (tid == 0) *total = carry;
}

__global__ __launch_bounds__(FD_SCAN_BLOCK) void fd_scan3_kernel(const long *local, const long *bsum,
                                                                 long nitems, const long *total,
                                                                 long *prefix)
{
    const long q = (long)blockIdx.x * FD_SCAN_BLOCK + threadIdx.x;
    if (q < nitems) prefix[q] = local[q] + bsum[blockIdx.x];
    if (q == 0) prefix[nitems] = *total;
}

#define FD_THREADS 256

// separate_modes: persistent walk over the flattened bins: workgroup b owns a
// contiguous range; each thread strides through it, reloading the item only
// when its next bin belongs to another (mode, segment).  Two waves per SIMD (197
// registers): 60 modes of one year 0.98 ms (one wave 1.56, three with 36 registers
// spilled 1.02, four 1.65).
__global__ __launch_bounds__(FD_THREADS) __attribute__((amdgpu_waves_per_eu(2, 2)))
void fd_sum_kernel(FdArgs a, long nitems)
{
    const long total = a.prefix[nitems];
    const long per = (total + gridDim.x - 1) / gridDim.x;
    const long w0 = (long)blockIdx.x * per;
    const long w1 = min(total, w0 + per);
    if (w0 >= w1) return;
    const FdSpaConst kc = fd_spa_const();
    const FdRootConst kr = fd_root_const();
    const long nb = (2L * a.K + 3) * a.L;
    long item = -1;
    long item_end = 0, item_begin = 0;
    int lo = 0;
    FdSeg it;
    for (long w = w0 + threadIdx.x; w < w1; w += FD_THREADS) {
        if (item < 0 || w >= item_end) {
            // last item with prefix[item] <= w (items without bins have equal prefixes)
            long l = item < 0 ? 0 : item, h = nitems;
            while (h - l > 1) {
                const long mid = (l + h) >> 1;
                if (a.prefix[mid] <= w) l = mid; else h = mid;
            }
            item = l;
            item_begin = a.prefix[item];
            item_end = a.prefix[item + 1];
            int hi;
            fd_item_range(a, item, lo, hi);
            fd_load_seg(a, (int)(item / a.nseg), (int)(item % a.nseg), it);
        }
        const int i = lo + (int)(w - item_begin);
        const double f = a.freqs[i];
        const int q = (int)(item / a.nseg);
        double2 *out = a.wave + (long)q * a.data_length + i;
        // one writer per (mode, bin); the -f terms are not part of this output
        fd_bin_fast(it, f, kr, kc, [&](double x, fcx B) {
            const double *c = a.interp + (long)q * a.L + (int)(item % a.nseg);
            fcx v = fcx_make(0.0, 0.0);
#pragma unroll
            for (int p = 3; p >= 0; p--) {
                v.re = v.re * x + c[p * nb];
                v.im = v.im * x + c[p * nb + (long)a.K * a.L];
            }
            const double2 yp = a.ylm[q];
            const fcx te = fcx_make(v.re * B.re - v.im * B.im, v.re * B.im + v.im * B.re);
            *out = make_double2(yp.x * te.re - yp.y * te.im, yp.x * te.im + yp.y * te.re);
        });
    }
}

// ------------------------------------------------ bin-owned accumulation
// Each output bin b is written by exactly one thread, which adds every
// contribution to it in a fixed order (no atomics, run-to-run identical).
// The +f and -f terms of one (item, bin) evaluation go to bins i and 2z - i
// (z = zero_index), so a thread owns a bin pair: owner o = b <= z with its
// mirror b' = 2z - b ("low" owners), or a bin b > 2z with no mirror partner
// ("high" owners).  The modes are summed by cell (modes sharing (m, k, n) and
// every segment's bin range, cells.hpp: they share roots, phase and
// stationary-phase factor, and their amplitudes add to one pair of cubics).  A
// workgroup takes 64 or 128 owners; for every cell it finds the segments whose
// bin range meets the tile's bins or their mirrors (each cell's segments sorted
// by first bin, with the running maximum of their last bins, so two binary
// searches bound the candidates).  Its four waves hold the same owners and take
// every fourth cell of the list each; their sums are added at the end.
//
// What bounds it: VALU issue, ~600 instructions per (cell, bin) evaluation, half
// of them the log, exp, atan2 and hypot of Cardano's cube root.  One year, 3843
// modes: 7.8 ms (122.6 ms with one evaluation per mode in the reference's
// operations); 0.1 yr, 1000 modes: 0.76 ms.

#define FD_OWN_TILE 256  // threads per workgroup (four waves)
// Owners per lane: two from 2^17 owner pairs on (one year, all modes: 7.7 ms
// with two, 8.0 with one, 8.0 with four), one below, where two would leave the
// chip idle (39,000 pairs, 1000 modes: 0.39 ms with one, 0.60 with two).
#define FD_OWN_LONG (1 << 17)

struct FdOwnIndex {
    int *cnt;   // (cells,) segments with in-range bins
    int *slo;   // (cells, nseg) their first bins, ascending (ties by segment)
    int *sj;    // (cells, nseg) the segment of each sorted position
    int *pmx;   // (cells, nseg) running maximum of the last bins in that order
};

__host__ __device__ inline size_t fd_align256(size_t x) { return (x + 255) & ~(size_t)255; }

#define FD_IDX_CHUNK 1024

// One wave per cell: its non-empty segments sorted by first bin (ties by
// segment) by counting the segments before each, then the running maximum of
// the last bins.  119 segments, 671 cells: 29 us (2.7 ms with one thread per
// mode sorting by insertion in global memory).
__global__ __launch_bounds__(64) void fd_index_kernel(FdArgs a, CellIndex cells, FdOwnIndex ix)
{
    __shared__ int s_lo[FD_IDX_CHUNK];
    const int c = blockIdx.x, lane = threadIdx.x;
    if (c >= (cells.start ? *cells.count : a.K)) return;
    const int q = cells.start ? cells.member[cells.start[c]] : c;
    const long rows = (long)q * a.nseg, base = (long)c * a.nseg;
    const int none = 0x7fffffff;  // an empty range: after every other
    int cnt = 0;
    for (int jb = 0; jb < a.nseg; jb += 64) {
        const int j = jb + lane;
        int lo = none, hi = -1;
        if (j < a.nseg) fd_item_range(a, rows + j, lo, hi);
        const bool has = j < a.nseg && hi >= lo;
        int before = 0;
        for (int b0 = 0; b0 < a.nseg; b0 += FD_IDX_CHUNK) {
            const int n = min(FD_IDX_CHUNK, a.nseg - b0);
            if (jb == 0 || a.nseg > FD_IDX_CHUNK) {
                __syncthreads();
                for (int i = lane; i < n; i += 64) {
                    int l, h;
                    fd_item_range(a, rows + b0 + i, l, h);
                    s_lo[i] = h >= l ? l : none;
                }
                __syncthreads();
            }
            for (int i = 0; i < n; i++) {
                const int l = s_lo[i];
                before += l < lo || (l == lo && l != none && b0 + i < j) ? 1 : 0;
            }
        }
        if (has) {
            ix.slo[base + before] = lo;
            ix.sj[base + before] = j;
        }
        cnt += __popcll(__ballot(has));
    }
    __threadfence_block();
    __syncthreads();
    int carry = -1;
    for (int p0 = 0; p0 < cnt; p0 += 64) {
        const int p = p0 + lane;
        int mx = -1;
        if (p < cnt) {
            int l;
            fd_item_range(a, rows + ix.sj[base + p], l, mx);
        }
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const int v = __shfl_up(mx, off, 64);
            if (lane >= off) mx = max(mx, v);
        }
        mx = max(mx, carry);
        if (p < cnt) ix.pmx[base + p] = mx;
        carry = __shfl(mx, 63, 64);
    }
    if (lane == 0) ix.cnt[c] = cnt;
}

// The item of (cell c, segment j): its first mode's segment and the combined
// cubics of its members.
__device__ inline void fd_form_item(const FdArgs &a, const CellIndex &cells, int c, int j, FdSeg &v)
{
    const int s0 = cells.start ? cells.start[c] : c, s1 = cells.start ? cells.start[c + 1] : c + 1;
    const long nb = (2L * a.K + 3) * a.L;
    fd_load_seg(a, cells.start ? cells.member[s0] : c, j, v);
    fcx cp[4], cm[4];
#pragma unroll
    for (int p = 0; p < 4; p++) cp[p] = cm[p] = fcx_make(0.0, 0.0);
    for (int s = s0; s < s1; s++) {
        const int q = cells.start ? cells.member[s] : s;
        const double2 yp = a.ylm[q], ym = a.ylm[a.K + q];
        const double *re = a.interp + (long)q * a.L + j, *im = re + (long)a.K * a.L;
#pragma unroll
        for (int p = 0; p < 4; p++) fd_cell_add(re[p * nb], im[p * nb], yp, ym, cp[p], cm[p]);
    }
#pragma unroll
    for (int p = 0; p < 4; p++) {
        v.tab[4 * p] = cp[p].re;
        v.tab[4 * p + 1] = cp[p].im;
        v.tab[4 * p + 2] = cm[p].re;
        v.tab[4 * p + 3] = cm[p].im;
    }
    v.pad[0] = v.pad[1] = v.pad2[0] = v.pad2[1] = v.pad2[2] = 0.0;
}

// The items of every segment of the cells [c0, c0 + ncells) (FdSeg's first part)
// and, with cell 0, of every segment (the rest), so that the sum fetches an item
// with two loads per lane.
__global__ __launch_bounds__(256) void fd_table_kernel(FdArgs a, CellIndex cells, int c0, int ncells,
                                                       double *cell_tab, double *seg_tab)
{
    const long at = (long)blockIdx.x * 256 + threadIdx.x;
    const int i = (int)(at / a.nseg), j = (int)(at - (long)i * a.nseg), c = c0 + i;
    if (i >= ncells || c >= (cells.start ? *cells.count : a.K)) return;
    FdSeg v;
    fd_form_item(a, cells, c, j, v);
    const double *d = reinterpret_cast<const double *>(&v);
#pragma unroll
    for (int e = 0; e < FD_CELL_DOUBLES; e++) cell_tab[FD_CELL_DOUBLES * at + e] = d[e];
    if (c == 0) {
#pragma unroll
        for (int e = 0; e < FD_SEG_DOUBLES; e++)
            seg_tab[FD_SEG_DOUBLES * j + e] = d[FD_CELL_DOUBLES + e];
    }
}

// Sorted positions [s, e) of a cell that can meet bins [w0, w1]: first bin
// <= w1 and running maximum of last bins >= w0 (e <= s: none).
__device__ inline void fd_candidates(const FdOwnIndex &ix, long base, int c, int w0, int w1,
                                     int &s, int &e)
{
    s = 0;
    e = 0;
    if (c == 0 || w1 < w0 || ix.slo[base] > w1 || ix.pmx[base + c - 1] < w0) return;
    int l = 0, h = c;  // e: first position with slo > w1
    while (l < h) {
        const int mid = (l + h) >> 1;
        if (ix.slo[base + mid] <= w1) l = mid + 1; else h = mid;
    }
    e = l;
    l = 0;
    h = e;  // s: first position with pmx >= w0
    while (l < h) {
        const int mid = (l + h) >> 1;
        if (ix.pmx[base + mid] >= w0) h = mid; else l = mid + 1;
    }
    s = l;
}

// Cells [c0, c0 + ncells).  TABLE: items from fd_table_kernel's tables of these
// cells; otherwise a wave's first lane forms each (workspaces without tables).
template <int BPT, bool TABLE>
__global__ __launch_bounds__(FD_OWN_TILE) __attribute__((amdgpu_waves_per_eu(4, 4)))
void fd_own_kernel(FdArgs a, CellIndex cells, int c0, int ncells, const double *cell_tab,
                   const double *seg_tab, FdOwnIndex ix, int n_low, int hb0, int tiles_low)
{
    constexpr int SPAN = 64 * BPT;  // owners per tile
    const int ncell = min(cells.start ? *cells.count : a.K, c0 + ncells);
    if (c0 >= ncell) return;  // uniform over the grid: fewer cells than modes
    __shared__ int s_q[2 * FD_OWN_TILE], s_s[2 * FD_OWN_TILE], s_e[2 * FD_OWN_TILE];
    __shared__ int s_scan[FD_OWN_TILE];
    __shared__ FdSeg s_it[FD_OWN_TILE / 64];  // the item each wave evaluates
    // per wave, the lane's accumulators: [0] its bins, [1] their mirrors
    __shared__ double2 s_acc[FD_OWN_TILE / 64][2][BPT][64];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    FdSeg &it = s_it[wv];
    auto &acc = s_acc[wv];
    const int z = a.zero_index, nf = a.data_length;
    // Low tiles in descending order: the frequencies nearest zero, where most
    // modes' bands overlap, carry the most work and start first.
    const bool low = (int)blockIdx.x < tiles_low;
    const int tile = low ? tiles_low - 1 - (int)blockIdx.x : (int)blockIdx.x;
    // this tile's bins [w0, w1] and their mirrors [m0, m1] (empty when m1 < m0)
    int w0, w1, m0 = 0, m1 = -1;
    if (low) {
        w0 = tile * SPAN;
        w1 = min(w0 + SPAN, n_low) - 1;
        m0 = max(2 * z - w1, 0);
        m1 = min(2 * z - w0, nf - 1);
    } else {
        w0 = hb0 + (tile - tiles_low) * SPAN;
        w1 = min(w0 + SPAN, nf) - 1;
    }
    // owner k of this lane: bin w0 + k * 64 + lane and (low tiles) its mirror
#pragma unroll
    for (int k = 0; k < BPT; k++) {
        acc[0][k][lane] = make_double2(0.0, 0.0);
        acc[1][k][lane] = make_double2(0.0, 0.0);
    }
    const FdSpaConst kc = fd_spa_const();
    const FdRootConst kr = fd_root_const();
    const bool minus_on = a.include_minus_m != 0;
    for (int q0 = c0; q0 < ncell; q0 += FD_OWN_TILE) {
        // candidate segment ranges of cell q0 + tid, compacted in cell order
        const int q = q0 + tid;
        int sa = 0, ea = 0, sb = 0, eb = 0;
        if (q < ncell) {
            const long base = (long)q * a.nseg;
            const int c = ix.cnt[q];
            fd_candidates(ix, base, c, w0, w1, sa, ea);
            fd_candidates(ix, base, c, m0, m1, sb, eb);
            if (ea > sa && eb > sb && sb <= ea && sa <= eb) {  // overlapping: one range
                sa = min(sa, sb);
                ea = max(ea, eb);
                eb = sb;
            }
        }
        const int na = (ea > sa ? 1 : 0) + (eb > sb ? 1 : 0);
        s_scan[tid] = na;
        __syncthreads();
        for (int off = 1; off < FD_OWN_TILE; off <<= 1) {
            const int v = tid >= off ? s_scan[tid - off] : 0;
            __syncthreads();
            s_scan[tid] += v;
            __syncthreads();
        }
        int pos = s_scan[tid] - na;
        const int nent = s_scan[FD_OWN_TILE - 1];
        if (ea > sa) {
            s_q[pos] = q;
            s_s[pos] = sa;
            s_e[pos] = ea;
            pos++;
        }
        if (eb > sb) {
            s_q[pos] = q;
            s_s[pos] = sb;
            s_e[pos] = eb;
        }
        __syncthreads();
        // The cells of the list, dealt to the waves in order (each adds into its
        // own accumulators).  A lane evaluates up to 2 BPT bins per item (its
        // bins and their mirrors), so one item load serves several evaluations,
        // all through one body (a second inlined copy of the large evaluation
        // costs instruction-cache misses).
        for (int en = wv; en < nent; en += FD_OWN_TILE / 64) {
            const int qe = __builtin_amdgcn_readfirstlane(s_q[en]);
            const int ps = __builtin_amdgcn_readfirstlane(s_s[en]);
            const int pe = __builtin_amdgcn_readfirstlane(s_e[en]);
            const long base = (long)qe * a.nseg;
            const int lead = cells.start ? cells.member[cells.start[qe]] : qe;
            const bool conj_term = minus_on && a.m[lead] != 0;
            for (int p = ps; p < pe; p++) {
                const int j = __builtin_amdgcn_readfirstlane(ix.sj[base + p]);
                int lo, hi;
                fd_item_range(a, (long)lead * a.nseg + j, lo, hi);
                unsigned mask = 0;  // bit 2k: bin of owner k, bit 2k + 1: its mirror
#pragma unroll
                for (int k = 0; k < BPT; k++) {
                    const int bk = w0 + k * 64 + lane;
                    if (bk <= w1) {
                        if (bk >= lo && bk <= hi) mask |= 1u << (2 * k);
                        const int mk = 2 * z - bk;
                        if (low && mk != bk && mk < nf && mk >= lo && mk <= hi)
                            mask |= 2u << (2 * k);
                    }
                }
                if (!__any(mask != 0)) continue;
                // the item's values, one copy per wave in LDS
                __builtin_amdgcn_wave_barrier();
                if (TABLE) {
                    double *d = reinterpret_cast<double *>(&it);
                    const long at = (long)(qe - c0) * a.nseg + j;
                    if (lane < FD_CELL_DOUBLES) d[lane] = cell_tab[FD_CELL_DOUBLES * at + lane];
                    if (lane < FD_SEG_DOUBLES)
                        d[FD_CELL_DOUBLES + lane] = seg_tab[FD_SEG_DOUBLES * j + lane];
                } else if (lane == 0) {
                    fd_form_item(a, cells, qe, j, it);
                }
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                __builtin_amdgcn_wave_barrier();
#pragma nounroll
                for (int slot = 0; slot < 2 * BPT; slot++) {
                    asm volatile("" ::: "memory");  // read the item again rather than hold it
                    const bool act = (mask >> slot) & 1u;
                    if (!__any(act)) continue;
                    if (act) {
                        const int k = slot >> 1;
                        const bool mirror = slot & 1;
                        const int bk = w0 + k * 64 + lane;
                        const int mk = 2 * z - bk;
                        // mirror == 0: +f to bk, -f to 2z - bk; mirror == 1: +f to the
                        // mirror bin, -f back to bk
                        fd_bin_fast(it, a.freqs[mirror ? mk : bk], kr, kc, [&](double x, fcx B) {
                            auto poly = [&](int e) {
                                return fma(fma(fma(it.tab[12 + e], x, it.tab[8 + e]), x, it.tab[4 + e]),
                                           x, it.tab[e]);
                            };
                            const fcx P = fcx_make(poly(0), poly(1));
                            double2 &tp = acc[mirror ? 1 : 0][k][lane];
                            tp.x += fma(P.re, B.re, -P.im * B.im);
                            tp.y += fma(P.re, B.im, P.im * B.re);
                            if (conj_term) {
                                const fcx M = fcx_make(poly(2), poly(3));
                                const fcx v = fcx_make(fma(M.re, B.re, M.im * B.im),
                                                       fma(M.im, B.re, -M.re * B.im));
                                if (mirror || mk == bk) {
                                    double2 &tm = acc[0][k][lane];
                                    tm.x += v.re;
                                    tm.y += v.im;
                                } else if (low && mk >= 0 && mk < nf) {
                                    double2 &tm = acc[1][k][lane];
                                    tm.x += v.re;
                                    tm.y += v.im;
                                }
                            }
                        });
                    }
                }
            }
        }
        __syncthreads();
    }
    // the loop's last barrier has passed: every wave's sums are in LDS
    for (int o = tid; o < SPAN; o += FD_OWN_TILE) {
        const int bk = w0 + o, k = o >> 6, l = o & 63;
        if (bk > w1) continue;
        const int mk = 2 * z - bk;
        auto add = [&](int m, int bin) {
            const double2 a0 = s_acc[0][m][k][l], a1 = s_acc[1][m][k][l];
            const double2 a2 = s_acc[2][m][k][l], a3 = s_acc[3][m][k][l], w = a.wave[bin];
            a.wave[bin] = make_double2(w.x + ((a0.x + a1.x) + (a2.x + a3.x)),
                                       w.y + ((a0.y + a1.y) + (a2.y + a3.y)));
        };
        add(0, bk);
        if (low && mk != bk && mk < nf) add(1, mk);
    }
}

// Owners and tiles of the bin-owned sum.
inline void fd_owner_split(int z, int nf, int bpt, int &n_low, int &hb0, int &tiles_low, int &tiles)
{
    n_low = z >= 0 ? min(z, nf - 1) + 1 : 0;
    hb0 = (int)std::max(2L * z + 1, 0L);
    const int n_high = hb0 < nf ? nf - hb0 : 0;
    const int span = 64 * bpt;
    tiles_low = (n_low + span - 1) / span;
    tiles = tiles_low + (n_high + span - 1) / span;
}

static size_t fd_scan_ws_bytes(int K, int nseg)
{
    const long nitems = (long)K * nseg;
    const long nb = (nitems + FD_SCAN_BLOCK - 1) / FD_SCAN_BLOCK;
    // local (nitems) + prefix (nitems + 1) + block sums (nb) + total
    return sizeof(long) * (size_t)(2 * nitems + 1 + nb + 1);
}

// What either path takes at least: the scan of the item walk (separate_modes)
// and the index of the bin-owned sum.
static size_t fd_base_bytes(int K, int nseg)
{
    const size_t nitems = (size_t)K * nseg;
    return fd_align256(fd_scan_ws_bytes(K, nseg)) + fd_align256(sizeof(int) * (size_t)K) +
           3 * fd_align256(sizeof(int) * nitems);
}

// Bin-owned sum: its index, the cells and the tables, from the workspace's start
// (the item walk's scan is not used there).  The number of cells is known on the
// device only, so the tables are sized for a slab of cells and the sum runs once
// per slab the modes could fill; past the last cell a launch ends at once.  64 MB
// hold 1762 cells of 119 segments, all 671 of the l <= 10, |n| <= 30 set: 3843
// modes in 0.02 yr take 559 us with the two empty passes and 551 us with tables
// for a cell per mode (146 MB).
#define FD_TABLE_BYTES ((size_t)1 << 26)

struct FdOwnLayout {
    size_t cnt, slo, sj, pmx, cells, seg, tab, total;
    int slab;  // cells per pass
};

static FdOwnLayout fd_own_layout(int K, int nseg)
{
    const size_t nitems = (size_t)K * nseg;
    const size_t per_cell = FD_CELL_DOUBLES * sizeof(double) * (size_t)nseg;
    FdOwnLayout l;
    l.cnt = 0;
    l.slo = fd_align256(sizeof(int) * (size_t)K);
    l.sj = l.slo + fd_align256(sizeof(int) * nitems);
    l.pmx = l.sj + fd_align256(sizeof(int) * nitems);
    l.cells = l.pmx + fd_align256(sizeof(int) * nitems);
    l.seg = l.cells + (K >= CELL_MIN_MODES ? cell_index_bytes(K) : 0);
    l.tab = l.seg + fd_align256(FD_SEG_DOUBLES * sizeof(double) * (size_t)nseg);
    l.slab = (int)std::min((size_t)K, std::max(FD_TABLE_BYTES / std::max(per_cell, (size_t)1), (size_t)1));
    l.total = l.tab + fd_align256(per_cell * (size_t)l.slab);
    return l;
}

size_t fd_workspace_bytes(int K, int nseg)
{
    return std::max(fd_base_bytes(K, nseg), fd_own_layout(K, nseg).total);
}

int launch_fd_sum(FdArgs a, void *workspace, size_t workspace_bytes, hipStream_t stream)
{
    const long nitems = (long)a.K * a.nseg;
    if (nitems <= 0) return FEW_OK;
    if (workspace_bytes < fd_base_bytes(a.K, a.nseg)) {
        set_error("fd_sum: workspace of %zu bytes, need %zu", workspace_bytes,
                  fd_base_bytes(a.K, a.nseg));
        return FEW_ERR_ARG;
    }
    const long nb = (nitems + FD_SCAN_BLOCK - 1) / FD_SCAN_BLOCK;
    if (nb > 0x7fffffffL) {
        set_error("fd_sum: too many (mode, segment) items (%ld)", nitems);
        return FEW_ERR_LIMIT;
    }
    if (!a.separate_modes) {
        // bin-owned: every bin written once per slab, contributions in a fixed order
        const FdOwnLayout l = fd_own_layout(a.K, a.nseg);
        char *w = static_cast<char *>(workspace);
        FdOwnIndex ix;
        ix.cnt = reinterpret_cast<int *>(w + l.cnt);
        ix.slo = reinterpret_cast<int *>(w + l.slo);
        ix.sj = reinterpret_cast<int *>(w + l.sj);
        ix.pmx = reinterpret_cast<int *>(w + l.pmx);
        double *seg_tab = reinterpret_cast<double *>(w + l.seg);
        double *cell_tab = reinterpret_cast<double *>(w + l.tab);
        CellIndex cells;
        if (a.K >= CELL_MIN_MODES && workspace_bytes >= l.seg) {
            int rc = launch_cell_index(a.m, a.k, a.n, a.K, a.seg_start, a.seg_end, a.nseg,
                                       w + l.cells, cells, stream);
            if (rc) return rc;
        }
        hipLaunchKernelGGL(fd_index_kernel, dim3(a.K), dim3(64), 0, stream, a, cells, ix);
        FEW_HIP(hipGetLastError());
        // a workspace between the least and the one asked for holds no tables
        const bool tables = workspace_bytes >= l.total;
        const int slab = tables ? l.slab : a.K;
        int n_low, hb0, tiles_low, tiles;
        const int bpt = tables && std::max(a.zero_index + 1, a.data_length - a.zero_index) >= FD_OWN_LONG
                            ? 2 : 1;
        fd_owner_split(a.zero_index, a.data_length, bpt, n_low, hb0, tiles_low, tiles);
        const dim3 grid(tiles), block(FD_OWN_TILE);
        for (int c0 = 0; c0 < a.K && tiles > 0; c0 += slab) {
            if (!tables) {
                hipLaunchKernelGGL((fd_own_kernel<1, false>), grid, block, 0, stream, a, cells, c0,
                                   slab, cell_tab, seg_tab, ix, n_low, hb0, tiles_low);
                FEW_HIP(hipGetLastError());
                break;
            }
            const long items = (long)std::min(slab, a.K - c0) * a.nseg;
            hipLaunchKernelGGL(fd_table_kernel, dim3((unsigned)((items + 255) / 256)), dim3(256), 0,
                               stream, a, cells, c0, slab, cell_tab, seg_tab);
            FEW_HIP(hipGetLastError());
            if (bpt == 1)
                hipLaunchKernelGGL((fd_own_kernel<1, true>), grid, block, 0, stream, a, cells, c0,
                                   slab, cell_tab, seg_tab, ix, n_low, hb0, tiles_low);
            else
                hipLaunchKernelGGL((fd_own_kernel<2, true>), grid, block, 0, stream, a, cells, c0,
                                   slab, cell_tab, seg_tab, ix, n_low, hb0, tiles_low);
            FEW_HIP(hipGetLastError());
        }
        return FEW_OK;
    }
    long *local = static_cast<long *>(workspace);
    long *prefix = local + nitems;
    long *bsum = prefix + nitems + 1;
    long *total = bsum + nb;
    hipLaunchKernelGGL(fd_scan1_kernel, dim3((unsigned)nb), dim3(FD_SCAN_BLOCK), 0, stream, a,
                       nitems, local, bsum);
    FEW_HIP(hipGetLastError());
    hipLaunchKernelGGL(fd_scan2_kernel, dim3(1), dim3(FD_SCAN_BLOCK), 0, stream, bsum, nb, total);
    FEW_HIP(hipGetLastError());
    hipLaunchKernelGGL(fd_scan3_kernel, dim3((unsigned)nb), dim3(FD_SCAN_BLOCK), 0, stream, local,
                       bsum, nitems, total, prefix);
    FEW_HIP(hipGetLastError());
    a.prefix = prefix;
    int dev = 0, ncu = 256;
    FEW_HIP(hipGetDevice(&dev));
    FEW_HIP(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
    // 8 workgroups per CU, each a contiguous bin range: 300 modes of 0.1 yr 0.72 ms,
    // 6 modes of 0.02 yr 25 us (64 per CU 0.85 ms and 99 us: short ranges form their
    // first item for few bins)
    hipLaunchKernelGGL(fd_sum_kernel, dim3((unsigned)(ncu * 8)), dim3(FD_THREADS), 0, stream, a,
                       nitems);
    FEW_HIP(hipGetLastError());
    return FEW_OK;
}

}  // namespace few
