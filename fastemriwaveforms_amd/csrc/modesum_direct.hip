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

// Stages cells [c0, c0 + cnt) of interval j (all four waves; the caller syncs).
__device__ __forceinline__ void direct_stage(const DirectArgs &a, int j, int c0, int cnt, DirectLds &sh)
{
    const int part = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // power staged
    const int own = threadIdx.x & 63;                                   // cell staged
    const int K = a.K;
    const double *ip = a.interp + (long)part * ((long)a.L * 2 * K) + (long)j * 2 * K;
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
}

// Adds the staged cells first, first + STEP, ... below cnt to the samples' sums.
// Returns whether every phase was within sincos_half_turns' range (always, if BIG).
template <int SPT, bool BIG, int STEP>
__device__ __forceinline__ bool direct_add(const DirectLds &sh, int first, int cnt,
                                           const double (&x)[SPT], const double (&Pp)[SPT],
                                           const double (&Pt)[SPT], const double (&Pr)[SPT],
                                           double (&re)[SPT], double (&im)[SPT])
{
    bool ok = true;
    for (int jj = first; jj < cnt; jj += STEP) {
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
            const bool in = cell_term_fp64<BIG>(c, m, k, n, x[u], Pp[u], Pt[u], Pr[u], re[u], im[u]);
            ok = ok && in;
        }
    }
    return ok;
}

// The cell loop of a tile: this wave's partial sums (re, im) of its samples, over
// every fourth cell.
template <int SPT, bool BIG>
__device__ __forceinline__ bool direct_cells(const DirectArgs &a, int j, DirectLds &sh,
                                             const double (&x)[SPT], const double (&Pp)[SPT],
                                             const double (&Pt)[SPT], const double (&Pr)[SPT],
                                             double (&re)[SPT], double (&im)[SPT])
{
    const int part = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int ncell = a.cells.start ? *a.cells.count : a.K;
    bool ok = true;
#pragma unroll
    for (int u = 0; u < SPT; u++) re[u] = im[u] = 0.0;
    for (int c0 = 0; c0 < ncell; c0 += CELL_CH) {
        const int cnt = min(CELL_CH, ncell - c0);
        __syncthreads();
        direct_stage(a, j, c0, cnt, sh);
        __syncthreads();
        const bool in = direct_add<SPT, BIG, 4>(sh, part, cnt, x, Pp, Pt, Pr, re, im);
        ok = ok && in;
    }
    return ok;
}

// Sample state of this lane's samples base + u STEP (those past the interval
// repeat its last one; their sums are dropped).
template <int SPT, int STEP>
__device__ __forceinline__ void direct_samples(const DirectArgs &a, int j, const Segment &sg, int base,
                                               double (&x)[SPT], double (&Pp)[SPT],
                                               double (&Pt)[SPT], double (&Pr)[SPT])
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
        sample_state(a.dt, min(base + u * STEP, sg.end - 1), sg.h_t, sg.pt, sg.pw, rp, rt, rr, st);
        x[u] = st.x;
        Pp[u] = st.Pp;
        Pt[u] = st.Pt;
        Pr[u] = st.Pr;
    }
}

template <int SPT>
__device__ __forceinline__ void direct_fp64_tile(const DirectArgs &a, int j, int q, DirectLds &sh)
{
    __shared__ double2 s_sum[3][64 * SPT];
    const int tid = threadIdx.x, lane = tid & 63;
    const int part = __builtin_amdgcn_readfirstlane(tid >> 6);
    const Segment sg = a.segs[j];
    const int base = sg.start + q * (64 * SPT) + lane;
    double x[SPT], Pp[SPT], Pt[SPT], Pr[SPT], re[SPT], im[SPT];
    direct_samples<SPT, 64>(a, j, sg, base, x, Pp, Pt, Pr);
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

// All staged cells for the lane's own samples, summed as the four waves of
// direct_fp64_tile sum them: every fourth cell, then the four sums in pairs.
template <int SPT, bool BIG>
__device__ __forceinline__ bool direct_few_cells(const DirectLds &sh, int cnt, const double (&x)[SPT],
                                                 const double (&Pp)[SPT], const double (&Pt)[SPT],
                                                 const double (&Pr)[SPT], double (&re)[SPT],
                                                 double (&im)[SPT])
{
    bool ok = true;
    double r[SPT], i[SPT], pr[SPT], pi[SPT];  // this part's sum, the even part before it
#pragma unroll
    for (int u = 0; u < SPT; u++) re[u] = im[u] = 0.0;
#pragma nounroll
    for (int part = 0; part < 4; part++) {
#pragma unroll
        for (int u = 0; u < SPT; u++) r[u] = i[u] = 0.0;
        const bool in = direct_add<SPT, BIG, 4>(sh, part, cnt, x, Pp, Pt, Pr, r, i);
        ok = ok && in;
#pragma unroll
        for (int u = 0; u < SPT; u++) {
            re[u] = part & 1 ? re[u] + (pr[u] + r[u]) : re[u];
            im[u] = part & 1 ? im[u] + (pi[u] + i[u]) : im[u];
            pr[u] = r[u];
            pi[u] = i[u];
        }
    }
    return ok;
}

// One tile (256 SPT samples) of a set of few modes: every lane has samples of its
// own and sums all cells, what the output holds being read ahead of them.  Four
// waves on the same samples would form each sample's state four times, which is
// most of the work here: one mode, 3.2 million samples added to: 34 us (66 us with
// direct_fp64_tile), 12 modes 82 us (102 us).  The same bits either way.
//
// What bounds it: with one mode the latency of a workgroup's chain (search, loads,
// staging, one sincos), 3.0 TB/s of the output read and written; from about ten
// modes FP64 VALU issue.
template <int SPT>
__device__ __forceinline__ void direct_few_tile(const DirectArgs &a, int j, int q, DirectLds &sh)
{
    static_assert(DIRECT_FEW <= CELL_CH && DIRECT_FEW < CELL_MIN_MODES,
                  "one staging holds every cell, a cell per mode");
    const Segment sg = a.segs[j];
    const int base = sg.start + q * (256 * SPT) + threadIdx.x;
    double x[SPT], Pp[SPT], Pt[SPT], Pr[SPT], re[SPT], im[SPT];
    double2 o[SPT];
#pragma unroll
    for (int u = 0; u < SPT; u++) {
        const int idx = base + u * 256;
        o[u] = !a.overwrite && idx < sg.end ? a.wave[idx] : make_double2(0.0, 0.0);
    }
    direct_stage(a, j, 0, a.K, sh);
    direct_samples<SPT, 256>(a, j, sg, base, x, Pp, Pt, Pr);
    __syncthreads();
    if (!__all(direct_few_cells<SPT, false>(sh, a.K, x, Pp, Pt, Pr, re, im)))
        direct_few_cells<SPT, true>(sh, a.K, x, Pp, Pt, Pr, re, im);
#pragma unroll
    for (int u = 0; u < SPT; u++) {
        const int idx = base + u * 256;
        if (idx >= sg.end) continue;
        a.wave[idx] = a.overwrite ? make_double2(re[u], im[u])
                                  : make_double2(re[u] + o[u].x, im[u] + o[u].y);
    }
}

// Overwriting sum: samples past the last interval's are zero.  Called after the
// tile: with a store to the output ahead of it, the compiler would take the tile's
// uniform values (interval, phase coefficients) through vector loads, lane by lane
// (one mode, 3.2 million samples: 43 us instead of 32).
__device__ __forceinline__ void direct_zero_tail(const DirectArgs &a, long block, long blocks)
{
    const long end = a.nseg > 0 ? a.segs[a.nseg - 1].end : 0;
    for (long i = end + block * blockDim.x + threadIdx.x; i < a.out_len; i += blocks * blockDim.x)
        a.wave[i] = make_double2(0.0, 0.0);
}

// PER: workgroups per tile of the interval plan, a part of it each.
// Four waves per SIMD: 128 registers, of which the four-sample form spills 51 (208 B
// of scratch), most of them around the repetition with the library sincos.
template <int SPT, int PER>
__global__ __launch_bounds__(256, 4) void direct_fp64_kernel(DirectArgs a)
{
    __shared__ DirectLds sh;
    const int b = blockIdx.x / PER;
    const int total = a.prefix[a.nseg];
    if (b < total) {
        const int j = find_segment(a.prefix, a.nseg, b);
        direct_fp64_tile<SPT>(a, j, PER * (b - a.prefix[j]) + blockIdx.x % PER, sh);
    }
    if (a.overwrite) direct_zero_tail(a, blockIdx.x, gridDim.x);
}

template <int SPT>
__global__ __launch_bounds__(256, 4) void direct_few_kernel(DirectArgs a)
{
    __shared__ DirectLds sh;
    const int b = blockIdx.x;
    const int total = a.prefix[a.nseg];
    if (b < total) {
        const int j = find_segment(a.prefix, a.nseg, b);
        direct_few_tile<SPT>(a, j, b - a.prefix[j], sh);
    }
    if (a.overwrite) direct_zero_tail(a, b, gridDim.x);
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
    __shared__ DirectLds sh;
    if (d.K <= DIRECT_FEW) direct_few_tile<SPT / 4>(a, j, lt - pref[j], sh);
    else direct_fp64_tile<SPT>(a, j, lt - pref[j], sh);
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

// A lane per sample where a set is small and there are samples for the lanes, 4096
// of them per mode.  Added to an output of 94,675 samples 1 / 8 / 12 / 20 modes take
// 8.1 / 10.0 / 10.9 / 13.0 us (11.1 / 12.1 / 12.7 / 13.9 with four waves on the same
// samples), 9468 samples 7.9 / 9.5 / 10.5 / 12.6 us (7.7 / 8.0 / 8.0 / 8.6).
static bool direct_few(long out_len, int K) { return K <= DIRECT_FEW && out_len >= 4096L * K; }

// Otherwise, below 2^17 samples the four-sample tiles are too few to fill the chip.
// One against four samples per lane, us (plan and cell index included):
//                     16,000     64,000     100,000    131,072    300,000 samples
//   20 modes          10 / 12    13 / 14    16 / 14    18 / 17    28 / 23
//   500 modes         46 / 64    72 / 94    97 / 93    118 / 124  225 / 194
//   3843 modes        117 / 143  170 / 202  224 / 204  278 / 261  508 / 401
// (the means of 30 and 120 knots, which change little).
int direct_tile(long out_len, int K)
{
    if (direct_few(out_len, K)) return DIRECT_FEW_TILE;
    return out_len < (1L << 17) ? 64 : DIRECT_TILE;
}

int launch_direct_fp64(const DirectArgs &a, int tile, int max_blocks, hipStream_t stream)
{
    if (max_blocks <= 0) return FEW_OK;
    const dim3 grid(max_blocks), block(256);
    if (tile == DIRECT_FEW_TILE && a.K <= DIRECT_FEW)
        hipLaunchKernelGGL(direct_few_kernel<DIRECT_FEW_TILE / 256>, grid, block, 0, stream, a);
    else if (tile == DIRECT_FEW_TILE)  // laid out for few modes, summed for many
        hipLaunchKernelGGL((direct_fp64_kernel<DIRECT_SPT, DIRECT_FEW_TILE / DIRECT_TILE>),
                           dim3(max_blocks * (DIRECT_FEW_TILE / DIRECT_TILE)), block, 0, stream, a);
    else if (tile == DIRECT_TILE)
        hipLaunchKernelGGL((direct_fp64_kernel<DIRECT_SPT, 1>), grid, block, 0, stream, a);
    else
        hipLaunchKernelGGL((direct_fp64_kernel<1, 1>), grid, block, 0, stream, a);
    FEW_HIP(hipGetLastError());
    return FEW_OK;
}

}  // namespace few
