// The reference's operations one for one, for the host tests (test infrastructure).
//
// The kernels evaluate shorter forms of these (cell_term_fp64, fd_bin_fast,
// aak_sample_fast, the wave-parallel AAK plan, amp2d_basis_kernel); host_twin.hip
// runs both, so the tests can hold these against the oracle bit for bit and the
// kernels' forms against them.  Included after the kernel sources, whose helpers
// (dense output, complex functions, Bessel routines) both share.
#pragma once

namespace few {

// ------------------------------------------------------------- direct mode sum
struct ModeCoef {
    double ry, rc1, rc2, rc3;     // real-part cubic
    double iy, ic1, ic2, ic3;     // imaginary-part cubic
    double yp_re, yp_im, ym_re, ym_im;
    double m, k, n;
};

// One mode's contribution at one sample (interpolate.cu:647-684):
//   P = exp(-i*phase) * A(x);  tr += [m != 0] conj(P) Y- ;  tr += P Y+
inline void mode_term_fp64(const ModeCoef &c, double x, double x2, double x3,
                                               double Pp, double Pt, double Pr, double &tr_re,
                                               double &tr_im)
{
    const double phase = mode_phase(c.m, Pp, c.k, Pt, c.n, Pr);
    double e_im, e_re;
    if (!sincos_cw(-phase, e_im, e_re)) sincos(-phase, &e_im, &e_re);
    const double a_re = c.ry + c.rc1 * x + c.rc2 * x2 + c.rc3 * x3;
    const double a_im = c.iy + c.ic1 * x + c.ic2 * x2 + c.ic3 * x3;
    const double p_re = e_re * a_re - e_im * a_im;
    const double p_im = e_re * a_im + e_im * a_re;
    const double tp_re = p_re * c.yp_re - p_im * c.yp_im;
    const double tp_im = p_re * c.yp_im + p_im * c.yp_re;
    double tm_re = 0.0, tm_im = 0.0;
    if (c.m != 0.0) {
        tm_re = p_re * c.ym_re + p_im * c.ym_im;
        tm_im = p_re * c.ym_im - p_im * c.ym_re;
    }
    tr_re = tr_re + tm_re + tp_re;
    tr_im = tr_im + tm_im + tp_im;
}

// --------------------------------------------------------- frequency domain
#pragma clang fp contract(off)

inline fcx fcx_rdiv(double x, fcx w) { return fcx_div(fcx_make(x, 0.0), w); }

// cube_roots (interpolate.cu:1113-1134): Cardano with the principal complex
// cube root; xi = (-1 + sqrt(-3)) / 2 is passed in (computed once per thread).
inline void fd_cube_roots(double a, double b, double c, double d, fcx xi,
                                              double out[3])
{
#pragma clang fp contract(off)
    const double b2 = b * b;
    const double b3 = b2 * b;
    const double a2 = a * a;
    const double D0 = (b2 - 3 * a * c);
    const double D1 = (2 * b3 - 9 * a * b * c + 27 * a2 * d);
    const fcx sq = fcx_sqrt(fcx_make(D1 * D1 - 4 * (D0 * D0 * D0), 0.0));
    const fcx C = fcx_pow(fcx_divr(fcx_addr(D1, sq), 2.), 1. / 3.);
    const double pre = -(1. / (3 * a));
    const fcx xiC = fcx_mul(xi, C);
    const fcx xixiC = fcx_mul(fcx_mul(xi, xi), C);
    out[0] = fcx_scale(fcx_add(fcx_addr(b, C), fcx_rdiv(D0, C)), pre).re;
    out[1] = fcx_scale(fcx_add(fcx_addr(b, xiC), fcx_rdiv(D0, xiC)), pre).re;
    out[2] = fcx_scale(fcx_add(fcx_addr(b, xixiC), fcx_rdiv(D0, xixiC)), pre).re;
}

// Everything one (mode, segment) item reads (interpolate.cu:1240-1345).
struct FdItem {
    double ar[4], ai[4];          // amplitude cubic, Re and Im
    double pp[8], pt[8], pr[8];   // dense-output phases
    double F0, F1, F2, F3;        // mode-frequency cubic
    double t0, t1, pt0, pw;       // segment bounds, phase segment start and width
    double mm, kk, nn;
    fcx yp, ym;
};

inline void fd_load_item(const FdArgs &a, int q, int j, FdItem &it)
{
#pragma clang fp contract(off)
    const long nb = (2L * a.K + 3) * a.L;
    const long np = (long)(a.L - 1) * 3;
    double fph[4], fth[4], frr[4];
    for (int c = 0; c < 4; c++) {
        it.ar[c] = a.interp[c * nb + (long)q * a.L + j];
        it.ai[c] = a.interp[c * nb + (long)(a.K + q) * a.L + j];
        fph[c] = a.interp[c * nb + (long)(2 * a.K) * a.L + j];
        fth[c] = a.interp[c * nb + (long)(2 * a.K + 1) * a.L + j];
        frr[c] = a.interp[c * nb + (long)(2 * a.K + 2) * a.L + j];
    }
    for (int c = 0; c < 8; c++) {
        it.pp[c] = a.pcoef[c * np + j];
        it.pt[c] = a.pcoef[c * np + (a.L - 1) + j];
        it.pr[c] = a.pcoef[c * np + 2 * (a.L - 1) + j];
    }
    const int m = a.m[q], k = a.k[q], n = a.n[q];
    it.mm = m;
    it.kk = k;
    it.nn = n;
    it.F0 = m * fph[0] + k * fth[0] + n * frr[0];
    it.F1 = m * fph[1] + k * fth[1] + n * frr[1];
    it.F2 = m * fph[2] + k * fth[2] + n * frr[2];
    it.F3 = m * fph[3] + k * fth[3] + n * frr[3];
    it.t0 = a.t_knots[j];
    it.t1 = a.t_knots[j + 1];
    it.pt0 = a.phase_t[j];
    it.pw = a.phase_t[j + 1] - a.phase_t[j];
    it.yp = fcx_make(a.ylm[q].x, a.ylm[q].y);
    it.ym = fcx_make(a.ylm[a.K + q].x, a.ylm[a.K + q].y);
}

inline double fd_fdot(const double *r, double s, double s2, double s3,
                                          double s4, double s5, double w2)
{
#pragma clang fp contract(off)
    return (-2. * r[2] + r[3] * (2. - 6. * s) + r[4] * (2. - 12. * s + 12. * s2) +
            r[5] * (6. * s - 24. * s2 + 20. * s3) + r[6] * (6. * s - 36. * s2 + 60. * s3 - 30. * s4) +
            r[7] * (12. * s2 - 60. * s3 + 90. * s4 - 42. * s5)) /
           (2. * M_PI * w2);
}

inline double fd_fddot(const double *r, double s, double s2, double s3,
                                           double s4, double w3)
{
#pragma clang fp contract(off)
    return (-6. * r[3] + r[4] * (-12. + 24. * s) + r[5] * (6. - 48. * s + 60. * s2) +
            r[6] * (6. - 72. * s + 180. * s2 - 120. * s3) +
            r[7] * (24. * s - 180. * s2 + 360. * s3 - 210. * s4)) /
           (2. * M_PI * w3);
}

// The contributions of bin i of an item: one per root inside the segment
// (up to three), each the +f term and the -f (conjugate) term, handed to
// emit(plus, minus) in root order.
template <class Emit>
inline void fd_bin(const FdItem &it, double f, fcx xi, const FdSpaConst &kc,
                                       Emit emit)
{
#pragma clang fp contract(off)
    double roots[3];
    fd_cube_roots(it.F3, it.F2, it.F1, (it.F0 - f), xi, roots);
    for (int r = 0; r < 3; r++) {
        const double root = roots[r];
        const double t = it.t0 + root;
        if (!((t < it.t1) && (t >= it.t0))) continue;
        const double x = root, x2 = x * x, x3 = x * x2;
        const double Are = it.ar[0] + it.ar[1] * x + it.ar[2] * x2 + it.ar[3] * x3;
        const double Aim = it.ai[0] + it.ai[1] * x + it.ai[2] * x2 + it.ai[3] * x3;
        const double s = (t - it.pt0) / it.pw;
        const double s1 = 1.0 - s;
        const double s2 = s * s, s3 = s * s2, s4 = s * s3, s5 = s * s4;
        const double w2 = it.pw * it.pw;
        const double w3 = it.pw * w2;
        const double phase = it.mm * fd_phase(it.pp, s, s1) + it.kk * fd_phase(it.pt, s, s1) +
                             it.nn * fd_phase(it.pr, s, s1);
        const double fdot = it.mm * fd_fdot(it.pp, s, s2, s3, s4, s5, w2) +
                            it.kk * fd_fdot(it.pt, s, s2, s3, s4, s5, w2) +
                            it.nn * fd_fdot(it.pr, s, s2, s3, s4, s5, w2);
        const double fddot = it.mm * fd_fddot(it.pp, s, s2, s3, s4, w3) +
                             it.kk * fd_fddot(it.pt, s, s2, s3, s4, w3) +
                             it.nn * fd_fddot(it.pr, s, s2, s3, s4, w3);
        const double targ = 2. * M_PI * fdot * fdot * fdot / (3. * fddot * fddot);
        const double pre = -1.0 * fdot / fabs(fddot) * 2. / sqrt(3.);
        const fcx amp2 = fcx_div(fcx_scale(fd_spa(targ, kc), pre), fcx_sqrt(fcx_make(targ, 0.0)));
        const fcx ph = fcx_exp(fcx_scale(fcx_make(0.0, 1.0), 2. * M_PI * f * t - phase));
        const fcx te = fcx_mul(fcx_mul(fcx_make(Are, Aim), amp2), ph);
        emit(fcx_mul(it.yp, te), fcx_mul(it.ym, fcx_make(te.re, -te.im)));
    }
}

inline int fd_minus_index(int zero_index, int i)
{
    const int diff = abs(zero_index - i);
    return (i < zero_index) ? zero_index + diff : zero_index - diff;
}

// ------------------------------------------------------------------------ AAK
// One output sample i of segment j (gpuAAK.cu:270-451); sc[p][c] are the
// segment's dense coefficients.  Returns hI - i hII, by the reference's
// operations one for one (the host tests' form; the kernel's is below).
inline double2 aak_sample(const AakArgs &a, const double (*sc)[8], double start_t,
                                              double segwidth, long i)
{
    const AakGeom G = aak_geom(a);
    const double phiS = a.phiS, phiK = a.phiK;
    const double cosqS = G.cosqS, sinqS = G.sinqS, cosqK = G.cosqK, sinqK = G.sinqK;
    const double cosphiK = G.cosphiK, sinphiK = G.sinphiK, cosphiS = G.cosphiS, sinphiS = G.sinphiS;
    const double cosdphi = G.cosdphi, sindphi = G.sindphi;
    const double halfsqrt3 = sqrt(3.) / 2.;
    const double mu_sec = a.mu * AAK_MTSUN_SI;
    const double zeta = mu_sec / a.dist / AAK_GPCINSEC;
    const double t = a.dt * i;
    const double s = (t - start_t) / segwidth;
    const double s1 = (1.0 - s);
    const double s2 = s * s, s3 = s * s2, s4 = s * s3, s5 = s * s4, s6 = s * s5;
    const double e = aak_dense(sc[1], s, s1);
    const double Y = aak_dense(sc[2], s, s1);
    const double Phi_phi = aak_dense(sc[3], s, s1);
    const double Phi_theta = aak_dense(sc[4], s, s1);
    const double Phi_r = aak_dense(sc[5], s, s1);
    const double OmegaPhi = aak_dense_dot(sc[3], s, s2, s3, s4, s5, s6) / segwidth;
    const double OmegaTheta = aak_dense_dot(sc[4], s, s2, s3, s4, s5, s6) / segwidth;
    const double OmegaR = aak_dense_dot(sc[5], s, s2, s3, s4, s5, s6) / segwidth;
    const double Phi = Phi_r;
    const double gim = Phi_theta - Phi_r;
    const double alp = Phi_phi - Phi_theta;
    const double nu = OmegaR / (2. * M_PI);
    const double gimdot = OmegaTheta - OmegaR;
    const double lam = acos(Y);
    double coslam, sinlam, cosalp, sinalp;
    sincos(lam, &sinlam, &coslam);
    sincos(alp, &sinalp, &cosalp);
    const double cosqL = cosqK * coslam + sinqK * sinlam * cosalp;
    const double sinqL = sqrt(1. - cosqL * cosqL);
    const double phiLup = sinqK * sinphiK * coslam - cosphiK * sinlam * sinalp - cosqK * sinphiK * sinlam * cosalp;
    const double phiLdown = sinqK * cosphiK * coslam + sinphiK * sinlam * sinalp - cosqK * cosphiK * sinlam * cosalp;
    const double phiL = atan2(phiLup, phiLdown);
    const double Ldotn = cosqL * cosqS + sinqL * sinqS * cos(phiL - phiS);
    const double Ldotn2 = Ldotn * Ldotn;
    const double Sdotn = cosqK * cosqS + sinqK * sinqS * cosdphi;
    double beta;
    if (a.S_phys == 0.0 || lam < 1e-10 || lam > (M_PI - 1e-10)) {
        beta = 0.0;
    } else {
        const double betaup = -Sdotn + coslam * Ldotn;
        const double betadown = sinqS * sindphi * sinlam * cosalp + (cosqK * Sdotn - cosqS) / sinqK * sinlam * sinalp;
        beta = atan2(betaup, betadown);
    }
    const double gam = 2. * (gim + beta);
    double cos2gam, sin2gam;
    sincos(gam, &sin2gam, &cos2gam);
    double cosorbphs = 0, FplusI, FcrosI, FplusII, FcrosII;
    if (a.mich) {
        const double orbphs = 2. * M_PI * t / AAK_YRSID_SI;
        double sinorbphs, sinorb, cosorb;
        sincos(orbphs - phiS, &sinorbphs, &cosorbphs);
        sincos(orbphs, &sinorb, &cosorb);
        const double cosq = .5 * cosqS - halfsqrt3 * sinqS * cosorbphs;
        const double phiw = orbphs + atan2(halfsqrt3 * cosqS + .5 * sinqS * cosorbphs, sinqS * sinorbphs);
        const double psiup = .5 * cosqK - halfsqrt3 * sinqK * cos(orbphs - phiK) - cosq * (cosqK * cosqS + sinqK * sinqS * cosdphi);
        const double psidown = .5 * sinqK * sinqS * sindphi - halfsqrt3 * cosorb * (cosqK * sinqS * sinphiS - cosqS * sinqK * sinphiK) - halfsqrt3 * sinorb * (cosqS * sinqK * cosphiK - cosqK * sinqS * cosphiS);
        const double psi = atan2(psiup, psidown);
        const double cosq1 = .5 * (1. + cosq * cosq);
        double cos2phi, sin2phi, cos2psi, sin2psi;
        sincos(2. * phiw, &sin2phi, &cos2phi);
        sincos(2. * psi, &sin2psi, &cos2psi);
        FplusI = cosq1 * cos2phi * cos2psi - cosq * sin2phi * sin2psi;
        FcrosI = cosq1 * cos2phi * sin2psi + cosq * sin2phi * cos2psi;
        FplusII = cosq1 * sin2phi * cos2psi + cosq * cos2phi * sin2psi;
        FcrosII = cosq1 * sin2phi * sin2psi - cosq * cos2phi * cos2psi;
    } else {
        FplusI = 1.0;
        FcrosI = 0.0;
        FplusII = 0.0;
        FcrosII = 1.0;
    }
    const double Amp = pow(fabs(OmegaPhi) * a.M_phys * AAK_MTSUN_SI, 2. / 3.) * zeta;
    double rot[4];
    aak_rot_coeff(rot, sinlam, coslam, sinqS, cosqS, sinphiS, cosphiS, sinqK, cosqK, sinphiK, cosphiK,
                  sinalp, cosalp);
    double hItemp = 0.0, hIItemp = 0.0;
    const double sq1e = sqrt(1 - e * e);
    for (int n = 1; n <= a.nmodes; n++) {
        double nPhi;
        if (a.mich) {
            const double fn = n * nu + gimdot / M_PI;
            const double Doppler = 2. * M_PI * fn * AAK_AUSEC * sinqS * cosorbphs;
            nPhi = n * Phi + Doppler;
        } else {
            nPhi = n * Phi;
        }
        const double ne = n * e;
        double Jv[5];
        nr_jn5(n - 2, ne, Jv);
        const double J0 = (n == 1) ? -1.0 * Jv[2] : Jv[0];
        const double J1 = Jv[1], J2 = Jv[2], J3 = Jv[3], J4 = Jv[4];
        double sn, cn;
        sincos(nPhi, &sn, &cn);
        const double aa = -n * Amp * (J0 - 2. * e * J1 + 2. / n * J2 + 2. * e * J3 - J4) * cn;
        const double bb = -n * Amp * sq1e * (J0 - 2. * J2 + J4) * sn;
        const double cc = 2. * Amp * J2 * cn;
        const double Aplus0 = -(1. + Ldotn2) * (aa * cos2gam - bb * sin2gam) + cc * (1 - Ldotn2);
        const double Acros0 = 2. * Ldotn * (bb * cos2gam + aa * sin2gam);
        const double Aplus = Aplus0 * rot[0] + Acros0 * rot[1];
        const double Acros = Aplus0 * rot[2] + Acros0 * rot[3];
        double hnI, hnII;
        if (a.mich) {
            hnI = halfsqrt3 * (FplusI * Aplus + FcrosI * Acros);
            hnII = halfsqrt3 * (FplusII * Aplus + FcrosII * Acros);
        } else {
            hnI = FplusI * Aplus + FcrosI * Acros;
            hnII = FplusII * Aplus + FcrosII * Acros;
        }
        hItemp += hnI;
        hIItemp += hnII;
    }
    return make_double2(hItemp, -hIItemp);
}

// gpuAAK.cu:458-483: start index of every segment and the number of knots
// used; segments stop at the last knot when none reaches the end (the
// reference then reads past its arrays).
inline int aak_plan(const double *h_t, int L, double dt, int out_len, int *st)
{
    const double T = (out_len - 1) * dt;
    st[0] = 0;
    int i;
    for (i = 1; i < L; i++) {
        const double t = h_t[i];
        if (t < T) {
            st[i] = (int)ceil(t / dt);
        } else {
            st[i] = out_len;
            break;
        }
    }
    return i < L ? i + 1 : L;
}

// ------------------------------------------------------- bicubic amplitudes
// One point's intervals and weights, as amp2d_basis_kernel lays them out.
inline void amp_point_basis(const double *tx, int nx, const double *ty, int ny,
                                                int kx, int ky, double x, double y, double *b)
{
    const int lx = amp_interval(tx, nx, kx, x, b + 2);
    const int ly = amp_interval(ty, ny, ky, y, b + 8);
    b[0] = (double)lx;
    b[1] = (double)ly;
}

}  // namespace few
