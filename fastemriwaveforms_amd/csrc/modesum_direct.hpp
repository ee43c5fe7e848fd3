// Per-sample / per-mode arithmetic of the direct mode sum, shared by the
// kernels and (host-callable) by the CPU test harness.
#pragma once

#include <math.h>

#include "cells.hpp"
#include "few_common.hpp"
#include "few_math.hpp"

namespace few {

struct PlanArgs {
    const double *h_t;   // (L,) amplitude knot times (device)
    const double *pt;    // (L,) phase dense-output segment times (device)
    int L;
    double dt;
    int out_len;
    int tile;            // samples per tile of the consuming kernel
    Segment *segs;       // (L-1,) out
    int *prefix;         // (L,) out: exclusive tile prefix, prefix[L-1] = total
};

struct DirectArgs {
    double2 *wave;            // (out_len,) complex128, accumulated into
    const double *interp;     // (4, L, 2K) knot-major coefficients (reference layout)
    const double *pcoef;      // (8, L-1, 3) dense-output phase coefficients
    const int *m, *k, *n;     // (K,)
    const double2 *ylm;       // (2K,) Y+ then Y- (already times (-1)^l)
    const Segment *segs;      // (L-1,)
    const int *prefix;        // (L,)
    int nseg;                 // L-1
    int L;
    int K;
    double dt;
    CellIndex cells;          // modes sharing (m, k, n); ungrouped: one cell per mode
    int out_len;
    int overwrite;            // write the samples (0 where no interval has any) instead of adding
};

// Output sample index -> start of its interval, find_start_inds rule
// (interpolate.cu:706-717): ceil(t/dt) while the knot is before
// (out_len-1)*dt, out_len afterwards.
__host__ __device__ inline int plan_start(const double *h_t, int j, double T, double dt, int out_len)
{
    if (j == 0) return 0;
    const double t = h_t[j];
    return (t < T) ? (int)ceil(t / dt) : out_len;
}

// Sample range [*st, *en) of interval j, given `used` (the find_start_inds
// stop: the first i >= 1 with h_t[i] >= T gives used = i + 1, else L).  The
// last used interval runs to out_len when the rule stopped early
// (interpolate.cu:711-715).  Intervals at or after used - 1 own no samples
// and are parked at out_len, so the covered samples are [0, en) of the last
// interval in every case.
__host__ __device__ inline void plan_interval(const double *h_t, int j, int used, int L, double T,
                                              double dt, int out_len, int *st, int *en)
{
    int s = out_len, e = out_len;
    if (j < used - 1) {
        s = plan_start(h_t, j, T, dt, out_len);
        e = plan_start(h_t, j + 1, T, dt, out_len);
        if (j + 1 == used - 1 && used < L) e = out_len;
        s = s < 0 ? 0 : (s > out_len ? out_len : s);
        e = e < 0 ? 0 : (e > out_len ? out_len : e);
        if (e < s) e = s;
    }
    *st = s;
    *en = e;
}

struct SampleState {
    double x;             // x = t - h_t[j] (amplitude cubic)
    double Pp, Pt, Pr;    // Phi_phi, Phi_theta, Phi_r at t
};

// Dense-output phase (interpolate.cu:642-644), contraction off.
__host__ __device__ inline double dense_phase(const double *r, double s, double s1)
{
#pragma clang fp contract(off)
    return r[0] + s * (r[1] + s1 * (r[2] + s * (r[3] + s1 * (r[4] + s * (r[5] + s1 * (r[6] + s * r[7]))))));
}

// The same polynomial with fused steps (seven FMAs instead of seven
// multiplications and seven additions), for the FP16-split paths: its
// rounding differs from dense_phase's by a few ulp of the phase (~1e-10 rad
// at 1e6 rad), far below those paths' ~1e-7 relative error.
__host__ __device__ inline double dense_phase_fused(const double *r, double s, double s1)
{
    double v = fma(s, r[7], r[6]);
    v = fma(s1, v, r[5]);
    v = fma(s, v, r[4]);
    v = fma(s1, v, r[3]);
    v = fma(s, v, r[2]);
    v = fma(s1, v, r[1]);
    return fma(s, v, r[0]);
}

// Sample-level quantities of make_waveform (interpolate.cu:626-644).
__host__ __device__ inline void sample_state(double dt, int i, double h_t, double pt, double pw,
                                             const double *rp, const double *rt, const double *rr,
                                             SampleState &st)
{
#pragma clang fp contract(off)
    const double t = dt * (double)i;
    st.x = t - h_t;
    const double s = (t - pt) / pw;
    const double s1 = 1.0 - s;
    st.Pp = dense_phase(rp, s, s1);
    st.Pt = dense_phase(rt, s, s1);
    st.Pr = dense_phase(rr, s, s1);
}

// m*Phi_phi + k*Phi_theta + n*Phi_r rounded exactly as the oracle
// (interpolate.cu:662); contraction off.
__host__ __device__ inline double mode_phase(double m, double Pp, double k, double Pt, double n,
                                             double Pr)
{
#pragma clang fp contract(off)
    return m * Pp + k * Pt + n * Pr;
}

// The contribution of all modes of one cell (one phase) at a sample, the sum of
// Y+ P + [m != 0] Y- conj(P) with P = exp(-i phase) A (interpolate.cu:647-684): with
// the cubics C+ = sum Y+ A and C- = sum Y- conj(A) (m != 0) of its members,
//   C+ exp(-i phase) + C- exp(+i phase)
//     = (P cos + Q sin) + i (R cos + S sin),
//   P = Re C+ + Re C-, Q = Im C+ - Im C-, R = Im C+ + Im C-, S = Re C- - Re C+.
// cell_coef_add adds a member's power p to (P, Q, R, S) of that power.
__host__ __device__ inline void cell_coef_add(double a_re, double a_im, double yp_re, double yp_im,
                                              double ym_re, double ym_im, bool minus, double (&v)[4])
{
    const double p_re = a_re * yp_re - a_im * yp_im, p_im = a_re * yp_im + a_im * yp_re;
    const double m_re = minus ? a_re * ym_re + a_im * ym_im : 0.0;
    const double m_im = minus ? a_re * ym_im - a_im * ym_re : 0.0;
    v[0] += p_re + m_re;
    v[1] += p_im - m_im;
    v[2] += p_im + m_im;
    v[3] += m_re - p_re;
}

// Sample term of one cell; c[p] holds (P, Q, R, S) of power p.  BIG: any phase
// (the library's sincos beyond sincos_cw's range); otherwise sincos_half_turns, and returns whether
// the phase was within that range (the term is meaningless if not).
template <bool BIG>
__host__ __device__ inline bool cell_term_fp64(const double (&c)[4][4], double m, double k, double n,
                                               double x, double Pp, double Pt, double Pr,
                                               double &tr_re, double &tr_im)
{
    const double phase = mode_phase(m, Pp, k, Pt, n, Pr);
    double sn, cs;
    bool ok = true;
    if (BIG) {
        if (!sincos_cw(phase, sn, cs)) sincos(phase, &sn, &cs);
    } else {
        ok = sincos_half_turns(phase, sn, cs);
    }
    double v[4];
#pragma unroll
    for (int e = 0; e < 4; e++) v[e] = fma(fma(fma(c[3][e], x, c[2][e]), x, c[1][e]), x, c[0][e]);
    tr_re = fma(v[0], cs, fma(v[1], sn, tr_re));
    tr_im = fma(v[2], cs, fma(v[3], sn, tr_im));
    return ok;
}

int launch_plan(const PlanArgs &p, hipStream_t stream);
constexpr int DIRECT_SPT = 4;                  // output samples per lane of a tile
constexpr int DIRECT_TILE = 64 * DIRECT_SPT;
// Sets of at most DIRECT_FEW modes: a lane per sample, in tiles of DIRECT_FEW_TILE
// samples (a batch keeps DIRECT_TILE).
constexpr int DIRECT_FEW = 16;
constexpr int DIRECT_FEW_TILE = 512;
// Samples per tile of the FP64 direct sum of K modes for an output of out_len samples.
int direct_tile(long out_len, int K);
// Whether launch_direct_fp64 takes tiles of this many samples (for any set of modes).
constexpr bool direct_tile_ok(int tile)
{
    return tile == 64 || tile == DIRECT_TILE || tile == DIRECT_FEW_TILE;
}
int launch_direct_fp64(const DirectArgs &a, int tile, int max_blocks, hipStream_t stream);

}  // namespace few
