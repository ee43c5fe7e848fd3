// Direct (per-mode) interpolated mode summation for gfx950.
//
// Two kernels:
//   * plan_segments_kernel -- the interval -> output-sample map of
//     find_start_inds (src/few/cutils/interpolate.cu:694-723) computed on the
//     device, plus an exclusive prefix of fixed-size sample tiles per
//     interval, so one launch covers every interval (the reference launches
//     once per interval with a device sync after each, interpolate.cu:750-771).
//   * direct_fp64_kernel -- the plain FP64 mode sum of make_waveform
//     (interpolate.cu:444-689), one term per cell (modes sharing (m, k, n),
//     cells.hpp): per output sample and cell the phase m*Phi_phi + k*Phi_theta
//     + n*Phi_r, one FP64 sincos and four real cubics.  The waveform is
//     accumulated into without atomics (every sample belongs to exactly one
//     lane of one block).
//
// Precision policy: the phase pipeline (dense-output evaluation, s, the
// m/k/n combination) is evaluated with contraction off in exactly the
// oracle's operation order, so the argument of sincos is bit-identical to
// the CPU restatement.  Amplitudes, their sums over the modes of a cell and
// the products may use FMA.

#include "batch.hpp"
#include "few_common.hpp"
#include "modesum_direct.hpp"

namespace few {

// One workgroup plans one waveform (256 threads).
__device__ void plan_segments_block(const PlanArgs &a)
{
    __shared__ int s_used;
    __shared__ int s_scan[256];
    __shared__ int s_carry;
    const int tid = threadIdx.x;
    const int L = a.L;
    const double T = (a.out_len - 1) * a.dt;
    if (tid == 0) {
        s_used = L;
        s_carry = 0;
    }
    __syncthreads();
    for (int i = 1 + tid; i < L; i += 256)
        if (!(a.h_t[i] < T)) atomicMin(&s_used, i + 1);
    __syncthreads();
    const int used = s_used;
    const int nseg = L - 1;
    for (int base = 0; base < nseg; base += 256) {
        const int j = base + tid;
        int nt = 0;
        if (j < nseg) {
            Segment sg;
            int st, en;
            plan_interval(a.h_t, j, used, L, T, a.dt, a.out_len, &st, &en);
            sg.start = st;
            sg.end = en;
            sg.h_t = a.h_t[j];
            sg.pt = a.pt[j];
            sg.pw = a.pt[j + 1] - a.pt[j];
            sg.hw = a.h_t[j + 1] - a.h_t[j];
            a.segs[j] = sg;
            nt = (en - st + a.tile - 1) / a.tile;
        }
        s_scan[tid] = nt;
        __syncthreads();
        // Hillis-Steele inclusive scan over 256 entries
        for (int off = 1; off < 256; off <<= 1) {
            int v = (tid >= off) ? s_scan[tid - off] : 0;
            __syncthreads();
            s_scan[tid] += v;
            __syncthreads();
        }
        const int carry = s_carry;
        if (j < nseg) a.prefix[j] = carry + s_scan[tid] - nt;
        __syncthreads();
        if (tid == 255) s_carry = carry + s_scan[255];
        __syncthreads();
    }
    if (tid == 0) a.prefix[nseg] = s_carry;
}

__global__ __launch_bounds__(256) void plan_segments_kernel(PlanArgs a) { plan_segments_block(a); }

// Block -> (interval, tile) by binary search over the tile prefix.
__device__ __forceinline__ int find_segment(const int *prefix, int nseg, int b)
{
    int lo = 0, hi = nseg;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (prefix[mid] <= b) lo = mid; else hi = mid;
    }
    return lo;
}

#define CELL_CH 64       // cells staged per LDS chunk

// One tile (64 SPT samples, tile q of interval j) of the FP64 direct sum: the
// four waves of the workgroup hold the same samples and take every fourth cell
// each, in a fixed order, and their partial sums are added at the end, so the
// result of a sample depends on neither the tile size nor the output length.
// Cells are staged CELL_CH at a time: a thread forms one power of one cell's
// combined cubics (cell_coef_add over its modes), wave w power w, so the loads
// of consecutive cells are consecutive modes.
//
// What bounds it: FP64 VALU issue, 52 instructions per (sample, cell), 30 of them
// the sincos.  One year at 10 s, 3843 modes (671 cells): 3.6 ms, 90 % of the
// VALU issue rate these take (33.7 ms with one term per mode, a sincos with a
// quarter-turn swap and the library's large-argument path inside the loop).
// Four samples per lane amortise the staging and the LDS reads (one: 6.0 ms,
// two: 4.4 ms, the same arithmetic).
struct DirectLds {
    double4 c[4][CELL_CH];  // [power][cell] (P, Q, R, S)
    double mkn[3][CELL_CH];
};

// The cell loop of a tile: this wave's partial sums (re, im) of its samples.
// Returns whether every phase was within sincos_half_turns' range (always, if BIG).
template <int SPT, bool BIG>
__device__ __forceinline__ bool direct_cells(const DirectArgs &a, int j, DirectLds &sh,
                                             const double (&x)[SPT], const double (&Pp)[SPT],
                                             const double (&Pt)[SPT], const double (&Pr)[SPT],
                                             double (&re)[SPT], double (&im)[SPT])
{
    const int tid = threadIdx.x;
    const int part = __builtin_amdgcn_readfirstlane(tid >> 6);  // power staged, cells summed
    const int own = tid & 63;                                   // cell staged
    const int K = a.K;
    const long nb = (long)a.L * 2 * K;
    const double *ip = a.interp + (long)part * nb + (long)j * 2 * K;
    const int ncell = a.cells.start ? *a.cells.count : K;
    bool ok = true;
#pragma unroll
    for (int u = 0; u < SPT; u++) re[u] = im[u] = 0.0;
    for (int c0 = 0; c0 < ncell; c0 += CELL_CH) {
        const int cnt = min(CELL_CH, ncell - c0);
        __syncthreads();
        if (own < cnt) {
            int s0 = c0 + own, s1 = s0 + 1;
            if (a.cells.start) {
                s0 = a.cells.start[c0 + own];
                s1 = a.cells.start[c0 + own + 1];
            }
            const int lead = a.cells.start ? a.cells.member[s0] : s0;
            const int m = a.m[lead];
            double v[4] = {0.0, 0.0, 0.0, 0.0};
            for (int s = s0; s < s1; s++) {
                const int mode = a.cells.start ? a.cells.member[s] : s;
                const double2 yp = a.ylm[mode], ym = a.ylm[K + mode];
                cell_coef_add(ip[mode], ip[K + mode], yp.x, yp.y, ym.x, ym.y, m != 0, v);
            }
            sh.c[part][own] = make_double4(v[0], v[1], v[2], v[3]);
            if (part == 0)
                sh.mkn[0][own] = (double)m;
            else if (part == 1)
                sh.mkn[1][own] = (double)a.k[lead];
            else if (part == 2)
                sh.mkn[2][own] = (double)a.n[lead];
        }
        __syncthreads();
        for (int jj = part; jj < cnt; jj += 4) {
            double c[4][4];
#pragma unroll
            for (int p = 0; p < 4; p++) {
                const double4 t = sh.c[p][jj];
                c[p][0] = t.x;
                c[p][1] = t.y;
                c[p][2] = t.z;
                c[p][3] = t.w;
            }
            const double m = sh.mkn[0][jj], k = sh.mkn[1][jj], n = sh.mkn[2][jj];
#pragma unroll
            for (int u = 0; u < SPT; u++) {
                const bool in = cell_term_fp64<BIG>(c, m, k, n, x[u], Pp[u], Pt[u], Pr[u], re[u],
                                                    im[u]);
                ok = ok && in;
            }
        }
    }
    return ok;
}

template <int SPT>
__device__ __forceinline__ void direct_fp64_tile(const DirectArgs &a, int j, int q)
{
    __shared__ DirectLds sh;
    __shared__ double2 s_sum[3][64 * SPT];
    const int tid = threadIdx.x, lane = tid & 63;
    const int part = __builtin_amdgcn_readfirstlane(tid >> 6);
    const Segment sg = a.segs[j];
    const int base = sg.start + q * (64 * SPT) + lane;
    double x[SPT], Pp[SPT], Pt[SPT], Pr[SPT], re[SPT], im[SPT];
    {
        const long np = (long)a.nseg * 3;
        double rp[8], rt[8], rr[8];
#pragma unroll
        for (int c = 0; c < 8; c++) {
            rp[c] = a.pcoef[c * np + (long)j * 3 + 0];
            rt[c] = a.pcoef[c * np + (long)j * 3 + 1];
            rr[c] = a.pcoef[c * np + (long)j * 3 + 2];
        }
#pragma unroll
        for (int u = 0; u < SPT; u++) {
            SampleState st;
            // samples past the interval repeat its last one (their sums are dropped)
            sample_state(a.dt, min(base + u * 64, sg.end - 1), sg.h_t, sg.pt, sg.pw, rp, rt, rr, st);
            x[u] = st.x;
            Pp[u] = st.Pp;
            Pt[u] = st.Pt;
            Pr[u] = st.Pr;
        }
    }
    const bool ok = direct_cells<SPT, false>(a, j, sh, x, Pp, Pt, Pr, re, im);
    // phases beyond 1e8 rad (or NaN): the tile again with the library's sincos
    if (__syncthreads_or(!ok)) direct_cells<SPT, true>(a, j, sh, x, Pp, Pt, Pr, re, im);
    if (part > 0) {
#pragma unroll
        for (int u = 0; u < SPT; u++) s_sum[part - 1][u * 64 + lane] = make_double2(re[u], im[u]);
    }
    __syncthreads();
    if (part == 0) {
#pragma unroll
        for (int u = 0; u < SPT; u++) {
            const int idx = base + u * 64;
            if (idx >= sg.end) continue;
            const double2 s1 = s_sum[0][u * 64 + lane], s2 = s_sum[1][u * 64 + lane];
            const double2 s3 = s_sum[2][u * 64 + lane];
            double2 w = make_double2((re[u] + s1.x) + (s2.x + s3.x), (im[u] + s1.y) + (s2.y + s3.y));
            if (!a.overwrite) {
                const double2 o = a.wave[idx];
                w.x += o.x;
                w.y += o.y;
            }
            a.wave[idx] = w;
        }
    }
}

// Overwriting sum: samples past the last interval's are zero.
__device__ __forceinline__ void direct_zero_tail(const DirectArgs &a, long block, long blocks)
{
    const long end = a.nseg > 0 ? a.segs[a.nseg - 1].end : 0;
    for (long i = end + block * blockDim.x + threadIdx.x; i < a.out_len; i += blocks * blockDim.x)
        a.wave[i] = make_double2(0.0, 0.0);
}

// Four waves per SIMD (at most 128 registers)
template <int SPT>
__global__ __launch_bounds__(256, 4) void direct_fp64_kernel(DirectArgs a)
{
    const int b = blockIdx.x;
    if (a.overwrite) direct_zero_tail(a, b, gridDim.x);
    const int total = a.prefix[a.nseg];
    if (b >= total) return;
    const int j = find_segment(a.prefix, a.nseg, b);
    direct_fp64_tile<SPT>(a, j, b - a.prefix[j]);
}

// ------------------------------------------------------------------ batch
__global__ __launch_bounds__(256) void batch_plan_kernel(BatchDev B, BatchRunDev r, BatchPtrs p,
                                                         int tile)
{
    const WaveDesc d = B.desc[blockIdx.x];
    const double *t = p.t + d.t_off;
    PlanArgs a{t, t, d.L, d.dt, d.N, tile, r.segs + d.seg_off, r.tpref + d.tpref_off};
    plan_segments_block(a);
}

// tiles before each waveform (one workgroup)
__global__ __launch_bounds__(256) void batch_tile_scan_kernel(BatchDev B, BatchRunDev r)
{
    __shared__ int s_scan[256];
    __shared__ int s_carry;
    const int tid = threadIdx.x;
    if (tid == 0) s_carry = 0;
    __syncthreads();
    for (int base = 0; base < B.B; base += 256) {
        const int b = base + tid;
        int nt = 0;
        if (b < B.B) {
            const WaveDesc d = B.desc[b];
            nt = r.tpref[d.tpref_off + d.L - 1];
        }
        s_scan[tid] = nt;
        __syncthreads();
        for (int off = 1; off < 256; off <<= 1) {
            const int v = (tid >= off) ? s_scan[tid - off] : 0;
            __syncthreads();
            s_scan[tid] += v;
            __syncthreads();
        }
        const int carry = s_carry;
        if (b < B.B) r.wt_prefix[b] = carry + s_scan[tid] - nt;
        __syncthreads();
        if (tid == 255) s_carry = carry + s_scan[255];
        __syncthreads();
    }
    if (tid == 0) r.wt_prefix[B.B] = s_carry;
}

int launch_batch_plan(const BatchDev &B, const BatchRunDev &r, const BatchPtrs &p, int tile,
                      hipStream_t stream)
{
    if (B.B <= 0) return FEW_OK;
    hipLaunchKernelGGL(batch_plan_kernel, dim3(B.B), dim3(256), 0, stream, B, r, p, tile);
    FEW_HIP(hipGetLastError());
    hipLaunchKernelGGL(batch_tile_scan_kernel, dim3(1), dim3(256), 0, stream, B, r);
    FEW_HIP(hipGetLastError());
    return FEW_OK;
}

// FP64 control run over the batch: block -> (waveform, interval, tile).
template <int SPT>
__global__ __launch_bounds__(256, 4) void batch_direct_fp64_kernel(BatchDev B, BatchRunDev r,
                                                                BatchPtrs p)
{
    const int g = blockIdx.x;
    if (g >= r.wt_prefix[B.B]) return;
    const int b = upper_index(r.wt_prefix, B.B, g);
    const WaveDesc d = B.desc[b];
    const int *pref = r.tpref + d.tpref_off;
    const int lt = g - r.wt_prefix[b];
    const int j = upper_index(pref, d.L - 1, lt);
    DirectArgs a;
    a.wave = p.wave + d.wave_off / 2;
    a.interp = p.interp + d.interp_off;
    a.pcoef = p.pcoef + d.pc_off;
    a.m = B.m + d.mode_off;
    a.k = B.k + d.mode_off;
    a.n = B.n + d.mode_off;
    a.ylm = reinterpret_cast<const double2 *>(p.ylm + d.ylm_off);
    a.segs = r.segs + d.seg_off;
    a.prefix = pref;
    a.nseg = d.L - 1;
    a.L = d.L;
    a.K = d.K;
    a.dt = d.dt;
    if (d.K >= CELL_MIN_MODES) {
        a.cells.count = B.dcell_start + d.dcell_off;
        a.cells.start = a.cells.count + 1;
        a.cells.member = B.dcell_member + d.mode_off;
    }
    a.out_len = d.N;
    a.overwrite = 0;
    direct_fp64_tile<SPT>(a, j, lt - pref[j]);
}

int launch_batch_direct_fp64(const BatchDev &B, const BatchRunDev &r, const BatchPtrs &p,
                             int max_blocks, hipStream_t stream)
{
    if (max_blocks <= 0) return FEW_OK;
    hipLaunchKernelGGL(batch_direct_fp64_kernel<DIRECT_SPT>, dim3(max_blocks),
                       dim3(256), 0, stream, B, r, p);
    FEW_HIP(hipGetLastError());
    return FEW_OK;
}

int launch_plan(const PlanArgs &p, hipStream_t stream)
{
    if (p.L < 2) {
        set_error("plan: need at least 2 knots (got %d)", p.L);
        return FEW_ERR_ARG;
    }
    hipLaunchKernelGGL(plan_segments_kernel, dim3(1), dim3(256), 0, stream, p);
    FEW_HIP(hipGetLastError());
    return FEW_OK;
}

// Below 2^17 samples the four-sample tiles are too few to fill the chip: 63,116
// samples of the full set take 128 us with one sample per lane and 183 us with
// four, 315,582 samples of 500 modes 193 us with four and 217 us with one.
int direct_tile(long out_len)
{
    return out_len < (1L << 17) ? 64 : DIRECT_TILE;
}

int launch_direct_fp64(const DirectArgs &a, int tile, int max_blocks, hipStream_t stream)
{
    if (max_blocks <= 0) return FEW_OK;
    const dim3 grid(max_blocks);
    if (tile == DIRECT_TILE)
        hipLaunchKernelGGL(direct_fp64_kernel<DIRECT_SPT>, grid, dim3(256), 0, stream, a);
    else
        hipLaunchKernelGGL(direct_fp64_kernel<1>, grid, dim3(256), 0, stream, a);
    FEW_HIP(hipGetLastError());
    return FEW_OK;
}

}  // namespace few
