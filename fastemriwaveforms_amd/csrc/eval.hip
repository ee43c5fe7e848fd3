// Spline evaluation (CubicSplineInterpolant.__call__) and the direct mode sum
// over dense per-sample amplitudes and phases (DirectModeSum.sum).
//
// Spline evaluation (summation/interpolatedmodesum.py:139-257): one lane per
// (array, point).  The interval is found by binary search with the
// reference's rule: searchsorted(t, x, side="right") - 1, and x == t[-1]
// belongs to the last interval.  The value or derivative is evaluated with
// the reference's expressions and operation order (contraction off), so the
// result equals numpy's bit for bit.  Order 0 fills points outside the knot
// range with the edge values; the flags report points outside the range
// (flags[0] left, flags[1] right) so the caller can warn, or raise for
// derivatives, as the reference does.
//
// Direct mode sum (summation/directmodesum.py:70-126): one lane per output
// sample; mode data staged through LDS in chunks; per mode
//   h += Y+ A e^{-i phi} + [m > 0] (-1)^l Y- conj(A) e^{+i phi},
// phi = m Phi_phi + k Phi_theta + n Phi_r, FP64 throughout.  The amplitude
// tile of a workgroup (its samples x a chunk of modes) is read with the
// modes contiguous, so the (N, K) amplitude array is read coalesced.
#include <math.h>

#include "eval.hpp"
#include "few_common.hpp"
#include "few_math.hpp"
#include "modesum_direct.hpp"

namespace few {

// The knot interval of point x0 (the reference's rule, clamped), and whether
// the point lies left or right of the knots.
__device__ __forceinline__ int spline_interval(const double *t, long tk, int L, double x0,
                                               bool &left, bool &right)
{
    const double tfirst = t[0], tlast = t[(long)(L - 1) * tk];
    // largest j with t[j] <= x0 (j = -1 when x0 < t[0]); x0 == t[L-1] -> L-2
    int lo = -1, hi = L;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (t[(long)mid * tk] <= x0) lo = mid; else hi = mid;
    }
    int j = lo;
    if (x0 == tlast) j = L - 2;
    left = x0 < tfirst;
    right = x0 > tlast;
    return j < 0 ? 0 : (j > L - 1 ? L - 1 : j);
}

// Value or derivative of a cubic at x past its knot (no edge values).
__device__ __forceinline__ double spline_value(int deriv, double x, double y, double c1, double c2,
                                               double c3)
{
#pragma clang fp contract(off)
    const double x2 = x * x;
    const double x3 = x2 * x;
    if (deriv == 0) return y + c1 * x + c2 * x2 + c3 * x3;
    if (deriv == 1) return c1 + 2 * c2 * x + 3 * c3 * x2;
    if (deriv == 2) return 2 * c2 + 6 * c3 * x;
    return 6 * c3;
}

__global__ __launch_bounds__(256) void spline_eval_kernel(SplineEvalArgs a)
{
    const long gid = (long)blockIdx.x * 256 + threadIdx.x;
    if (gid >= (long)a.ninterps * a.npts) return;
    const int s = (int)(gid / a.npts);
    const int q = (int)(gid - (long)s * a.npts);
    const double *t = a.t + (long)s * a.t_sys;
    const int L = a.length;
    const double x0 = a.tnew[(long)s * a.tn_sys + q];
    bool left, right;
    const int j = spline_interval(t, a.t_knot, L, x0, left, right);
    if (left) a.flags[0] = 1;    // benign race: every writer stores 1
    if (right) a.flags[1] = 1;
    const double *c = a.coef + (long)s * a.c_sys + (long)j * a.c_knot;
    const double y = c[0], c1 = c[a.c_coef], c2 = c[2 * a.c_coef], c3 = c[3 * a.c_coef];
    double v = spline_value(a.deriv, x0 - t[(long)j * a.t_knot], y, c1, c2, c3);
    if (a.deriv == 0) {
        if (left) v = a.coef[(long)s * a.c_sys];
        if (right) v = a.coef[(long)s * a.c_sys + (long)(L - 1) * a.c_knot];
    }
    a.out[(long)s * a.npts + q] = v;
}

#define SE_ARRAYS 64   // arrays of a shared-point tile (lanes of the evaluation)
#define SE_POINTS 64   // points of a tile (lanes of the search and of the stores)
#define SE_UNROLL 4    // points in flight per wave (2 and 8 measure the same)

// Arrays on one set of knots and points, their coefficients array-contiguous
// (what CubicSplineInterpolant holds): a workgroup takes 64 arrays x 64
// points.  One wave finds the intervals of the points, each wave then evaluates
// 16 points with one lane per array, so the four coefficients are read as whole
// 512-byte rows, and the tile is turned in LDS so that the values are stored
// along the points.
//
// What bounds it: the writes.  7686 arrays x 1000 points, 120 knots: 30 us,
// 61 MB written and 30 MB read (105 us with one lane per (array, point), whose
// four reads fall on 64 different lines per wave; 67 us if the points ascend).
// Workgroup i runs on XCD i % 8, whose L2 holds the coefficients of the groups it
// works on: every eighth group goes to an XCD, its tiles one after another.  Fewer
// than 32 groups would leave XCDs with less or no work (64 arrays x 16384 points:
// 28 us); each XCD then takes an equal run of the tiles instead (9.4 us; for 7686
// arrays x 256 points such runs cost 5 %, the XCDs being far apart in memory).
__global__ __launch_bounds__(256) void spline_eval_shared_kernel(SplineEvalArgs a, int chunks,
                                                                 int groups, int per)
{
    __shared__ double s_v[SE_ARRAYS][SE_POINTS + 1];
    __shared__ double s_x[SE_POINTS];
    __shared__ int s_j[SE_POINTS], s_out[SE_POINTS];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int xcd = (int)blockIdx.x & 7, slot = (int)blockIdx.x >> 3;
    const int tile = per ? xcd * per + slot : slot;
    int grp = tile / chunks;
    const int q0 = (tile - grp * chunks) * SE_POINTS;
    if (!per) grp = xcd + 8 * grp;
    if (grp >= groups) return;
    const int s0 = grp * SE_ARRAYS;
    const int nq = min(SE_POINTS, a.npts - q0), ns = min(SE_ARRAYS, a.ninterps - s0);
    const int L = a.length;
    if (wv == 0) {
        const double x0 = a.tnew[q0 + min(lane, nq - 1)];
        bool left, right;
        const int j = spline_interval(a.t, a.t_knot, L, x0, left, right);
        if (left) a.flags[0] = 1;    // benign race: every writer stores 1
        if (right) a.flags[1] = 1;
        s_x[lane] = x0 - a.t[(long)j * a.t_knot];
        s_j[lane] = j;
        s_out[lane] = right ? 2 : left ? 1 : 0;
    }
    __syncthreads();
    const double *cs = a.coef + s0 + min(lane, ns - 1);
    for (int qb = wv * SE_UNROLL; qb < nq; qb += 4 * SE_UNROLL) {
        double c[SE_UNROLL][4];
#pragma unroll
        for (int u = 0; u < SE_UNROLL; u++) {
            const double *p = cs + (long)s_j[min(qb + u, nq - 1)] * a.c_knot;
#pragma unroll
            for (int e = 0; e < 4; e++) c[u][e] = p[e * a.c_coef];
        }
#pragma unroll
        for (int u = 0; u < SE_UNROLL; u++) {
            const int q = min(qb + u, nq - 1);
            double v = spline_value(a.deriv, s_x[q], c[u][0], c[u][1], c[u][2], c[u][3]);
            const int edge = a.deriv == 0 ? __builtin_amdgcn_readfirstlane(s_out[q]) : 0;
            if (edge) v = cs[edge == 2 ? (long)(L - 1) * a.c_knot : 0];
            s_v[lane][q] = v;
        }
    }
    __syncthreads();
    if (lane >= nq) return;
    for (int r = wv; r < ns; r += 4) a.out[(long)(s0 + r) * a.npts + q0 + lane] = s_v[r][lane];
}

// Tiles where they are faster whatever the order of the points (a lane per value
// reads fewer lines where neighbouring points share an interval).  A tile's search,
// loads and stores follow each other, so a call in tiles takes 8.8 us or more:
//                              tiles     lane per value, points ascending / random
//   512 arrays x 1024 points   8.8       6.6 / 10.1
//   64 x 16384, 512 x 2048     9.4       10.4, 10.6 / 17.0, 16.9
//   448 x 2048, 800 x 1024     9.5, 9.1  9.4, 9.2 / 15.0, 14.2
// and with few points per array the lanes of a wave share less:
//   1600 x 512, 2048 x 256     9.2, 8.8  9.5, 14.5
//   1100 x 512                 8.9       7.5
static bool spline_eval_tiled(const SplineEvalArgs &a, long n)
{
    if (a.t_sys != 0 || a.tn_sys != 0 || a.c_sys != 1) return false;
    if (a.ninterps < SE_ARRAYS || a.npts < SE_POINTS) return false;
    return n >= 7L << 17 || (a.ninterps >= 1536 && n >= 1L << 19);
}

int launch_spline_eval(const SplineEvalArgs &a, hipStream_t stream)
{
    const long n = (long)a.ninterps * a.npts;
    if (n <= 0) return FEW_OK;
    if (spline_eval_tiled(a, n)) {
        const int groups = (a.ninterps + SE_ARRAYS - 1) / SE_ARRAYS;
        const int chunks = (int)(((long)a.npts + SE_POINTS - 1) / SE_POINTS);
        // 0: every eighth group to an XCD
        const long per = groups < 32 ? ((long)groups * chunks + 7) / 8 : 0;
        const long blocks = 8 * (per ? per : (long)((groups + 7) / 8) * chunks);
        if (blocks <= 0x7fffffffL) {
            hipLaunchKernelGGL(spline_eval_shared_kernel, dim3((unsigned)blocks), dim3(256), 0,
                               stream, a, chunks, groups, (int)per);
            FEW_HIP(hipGetLastError());
            return FEW_OK;
        }
    }
    if ((n + 255) / 256 > 0x7fffffffL) {
        set_error("spline_eval: too many points (%ld)", n);
        return FEW_ERR_LIMIT;
    }
    hipLaunchKernelGGL(spline_eval_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream,
                       a);
    FEW_HIP(hipGetLastError());
    return FEW_OK;
}

// ------------------------------------------------------------ direct mode sum

#define DS_SAMPLES 64          // samples (lanes) per workgroup
#define DS_MODES 32            // modes staged per step (LDS tile 64 x 33 complex = 33.8 KB)

__global__ __launch_bounds__(DS_SAMPLES) void dense_sum_kernel(DenseSumArgs a)
{
    __shared__ double2 sA[DS_SAMPLES][DS_MODES + 1];
    __shared__ double sY[4][DS_MODES];
    __shared__ double sQ[5][DS_MODES];   // m, k, n, (-1)^l, [m > 0]
    const int tid = threadIdx.x;
    const long i0 = (long)blockIdx.x * DS_SAMPLES;
    const long i = i0 + tid;
    const bool ok = i < a.N;
    double pp = 0.0, pt = 0.0, pr = 0.0;
    if (ok) {
        pp = a.phi_phi[i];
        pt = a.phi_theta[i];
        pr = a.phi_r[i];
    }
    double hr = 0.0, hi = 0.0;
    for (int q0 = 0; q0 < a.K; q0 += DS_MODES) {
        const int cnt = min(DS_MODES, a.K - q0);
        __syncthreads();
        // amplitude tile: row r (sample i0 + r), modes q0 .. q0+cnt-1, read along the modes
        for (int r = 0; r < DS_SAMPLES; r++) {
            const long ii = i0 + r;
            if (ii < a.N && tid < cnt) sA[r][tid] = a.teuk[ii * a.K + q0 + tid];
        }
        if (tid < cnt) {
            const int q = q0 + tid;
            const double2 yp = a.ylm[q], ym = a.ylm[a.K + q];
            sY[0][tid] = yp.x; sY[1][tid] = yp.y; sY[2][tid] = ym.x; sY[3][tid] = ym.y;
            sQ[0][tid] = (double)a.m[q];
            sQ[1][tid] = (double)a.k[q];
            sQ[2][tid] = (double)a.n[q];
            sQ[3][tid] = (a.l[q] & 1) ? -1.0 : 1.0;
            sQ[4][tid] = a.m[q] > 0 ? 1.0 : 0.0;
        }
        __syncthreads();
        if (!ok) continue;
        for (int u = 0; u < cnt; u++) {
            const double phase = mode_phase(sQ[0][u], pp, sQ[1][u], pt, sQ[2][u], pr);
            double sn, cs;
            if (!sincos_cw(phase, sn, cs)) sincos(phase, &sn, &cs);
            const double2 A = sA[tid][u];
            // Y+ A e^{-i phi}
            const double ya_r = sY[0][u] * A.x - sY[1][u] * A.y;
            const double ya_i = sY[0][u] * A.y + sY[1][u] * A.x;
            hr += ya_r * cs + ya_i * sn;
            hi += ya_i * cs - ya_r * sn;
            // [m > 0] (-1)^l Y- conj(A) e^{+i phi}
            const double w = sQ[3][u] * sQ[4][u];
            const double yb_r = w * (sY[2][u] * A.x + sY[3][u] * A.y);
            const double yb_i = w * (sY[3][u] * A.x - sY[2][u] * A.y);
            hr += yb_r * cs - yb_i * sn;
            hi += yb_i * cs + yb_r * sn;
        }
    }
    if (ok) a.out[i] = make_double2(hr, hi);
}

int launch_dense_sum(const DenseSumArgs &a, hipStream_t stream)
{
    if (a.N <= 0) return FEW_OK;
    const long blocks = ((long)a.N + DS_SAMPLES - 1) / DS_SAMPLES;
    if (blocks > 0x7fffffffL) {
        set_error("direct_mode_sum: too many samples (%d)", a.N);
        return FEW_ERR_LIMIT;
    }
    hipLaunchKernelGGL(dense_sum_kernel, dim3((unsigned)blocks), dim3(DS_SAMPLES), 0, stream, a);
    FEW_HIP(hipGetLastError());
    return FEW_OK;
}

}  // namespace few
