// Grouping of a mode set into cells (cells.hpp) on the device, from the mode
// arrays alone: the drop-in entry points have no host copy of them.
#include "cells.hpp"

namespace few {

static inline size_t cal256(size_t x) { return (x + 255) & ~(size_t)255; }

// Workspace: counters | start (K + 1) | member (K) | first (K) | rank (K) |
// size (K) | row hash (K)
struct CellWs {
    int *count, *bad, *start, *member, *first, *rank, *size;
    int *hash;
};

static CellWs cell_ws(void *ws, int K)
{
    char *w = static_cast<char *>(ws);
    CellWs c;
    c.count = reinterpret_cast<int *>(w);
    c.bad = c.count + 1;
    w += 256;
    auto take = [&](size_t n) {
        int *p = reinterpret_cast<int *>(w);
        w += cal256(sizeof(int) * n);
        return p;
    };
    c.start = take((size_t)K + 1);
    c.member = take(K);
    c.first = take(K);
    c.rank = take(K);
    c.size = take(K);
    c.hash = take(K);
    return c;
}

size_t cell_index_bytes(int K)
{
    const size_t k = K > 0 ? K : 1;
    return 256 + cal256(sizeof(int) * (k + 1)) + 5 * cal256(sizeof(int) * k);
}

// One wave per mode: a hash of its row values (the match below compares
// hashes; cell_verify_kernel compares the values).
__global__ __launch_bounds__(256) void cell_hash_kernel(const int *ra, const int *rb, int width,
                                                        int K, CellWs c)
{
    const int q = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (blockIdx.x == 0 && threadIdx.x == 0) *c.bad = 0;
    if (q >= K) return;
    unsigned long long h = 0;
    for (int j = lane; j < width; j += 64) {
        unsigned long long v = ((unsigned long long)(unsigned)ra[(long)q * width + j] << 32) |
                               (unsigned)rb[(long)q * width + j];
        v += 0x9e3779b97f4a7c15ull * (unsigned long long)(j + 1);  // splitmix64 of (value, place)
        v = (v ^ (v >> 30)) * 0xbf58476d1ce4e5b9ull;
        v = (v ^ (v >> 27)) * 0x94d049bb133111ebull;
        h += v ^ (v >> 31);
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) h += __shfl_xor(h, off, 64);
    if (lane == 0) c.hash[q] = (int)(h ^ (h >> 32));
}

#define CELL_WAVES 16
#define CELL_CHUNK 2048

// 64 modes per workgroup (one per lane); its 16 waves each compare them with a
// sixteenth of all modes: first mode with the same key, modes with it before
// this one, and their number.  The compared modes are staged in LDS: a 32-bit
// mix of (m, k, n, row hash), four read by a whole wave at once, and the values
// themselves for the few whose mix matches a lane.  K = 3843: 16 us (500: 4 us)
// (40 us comparing the four values of every mode: the 61 workgroups of this
// set run on 61 CUs, so instructions per compare are what counts).
__global__ __launch_bounds__(64 * CELL_WAVES) void cell_match_kernel(const int *m, const int *k,
                                                                     const int *n, int K, CellWs c,
                                                                     int hashed)
{
    __shared__ __attribute__((aligned(16))) unsigned s_mix[CELL_CHUNK];
    __shared__ int4 s_key[CELL_CHUNK];
    __shared__ int s_first[64], s_rank[64], s_size[64];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int q = blockIdx.x * 64 + lane, qc = min(q, K - 1);
    if (wv == 0) {
        s_first[lane] = q;
        s_rank[lane] = 0;
        s_size[lane] = 0;
    }
    auto mix = [](int4 v) {
        return (unsigned)v.x * 0x9e3779b1u + (unsigned)v.y * 0x85ebca77u +
               (unsigned)v.z * 0xc2b2ae3du + (unsigned)v.w;
    };
    const int4 key = make_int4(m[qc], k[qc], n[qc], hashed ? c.hash[qc] : 0);
    const unsigned my = mix(key);
    int first = q, rank = 0, size = 0;
    for (int base = 0; base < K; base += CELL_CHUNK) {
        const int cnt = min(CELL_CHUNK, K - base);
        __syncthreads();
        for (int i = tid; i < cnt; i += 64 * CELL_WAVES) {
            const int j = base + i;
            const int4 v = make_int4(m[j], k[j], n[j], hashed ? c.hash[j] : 0);
            s_key[i] = v;
            s_mix[i] = mix(v);
        }
        __syncthreads();
        auto compare = [&](int i) {
            const int4 o = s_key[i];
            const int j = base + i;
            const bool same =
                ((o.x ^ key.x) | (o.y ^ key.y) | (o.z ^ key.z) | (o.w ^ key.w)) == 0;
            first = same ? min(first, j) : first;
            size += same ? 1 : 0;
            rank += same && j < q ? 1 : 0;
        };
        const int full = cnt & ~3;
        for (int i = 4 * wv; i < full; i += 4 * CELL_WAVES) {
            const uint4 o = *reinterpret_cast<const uint4 *>(&s_mix[i]);
            if (__any(o.x == my)) compare(i);
            if (__any(o.y == my)) compare(i + 1);
            if (__any(o.z == my)) compare(i + 2);
            if (__any(o.w == my)) compare(i + 3);
        }
        if (wv == 0)
            for (int i = full; i < cnt; i++) compare(i);
    }
    if (q < K && size) {
        atomicMin(&s_first[lane], first);
        atomicAdd(&s_rank[lane], rank);
        atomicAdd(&s_size[lane], size);
    }
    __syncthreads();
    if (wv == 0 && q < K) {
        c.first[q] = s_first[lane];
        c.rank[q] = s_rank[lane];
        c.size[q] = s_size[lane];
    }
}

// One wave per mode: its rows against its cell's first mode's.  A difference
// (two rows with one hash) marks the index bad: it then groups nothing.
__global__ __launch_bounds__(256) void cell_verify_kernel(const int *ra, const int *rb, int width,
                                                          int K, CellWs c)
{
    const int q = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (q >= K) return;
    const int f = c.first[q];
    if (f == q) return;
    bool same = true;
    for (int j = lane; j < width; j += 64)
        same = same && ra[(long)q * width + j] == ra[(long)f * width + j] &&
               rb[(long)q * width + j] == rb[(long)f * width + j];
    if (!__all(same) && lane == 0) atomicOr(c.bad, 1);
}

// One workgroup: cells numbered in the order of their first modes, member
// lists.  Thread i takes a contiguous run of modes (its loads in flight
// together), one scan over the threads places the runs.
__global__ __launch_bounds__(1024) void cell_layout_kernel(int K, CellWs c, int verified)
{
    __shared__ int s_cell[16], s_mode[16];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const bool bad = verified && *c.bad != 0;
    const int per = (K + 1023) / 1024;
    const int q0 = min(K, tid * per), q1 = min(K, q0 + per);
    int cells = 0, modes = 0;  // led by this thread's modes
#pragma unroll 4
    for (int q = q0; q < q1; q++) {
        const bool lead = bad || c.first[q] == q;
        const int size = bad ? 1 : c.size[q];
        cells += lead ? 1 : 0;
        modes += lead ? size : 0;
    }
    int a = cells, b = modes;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int x = __shfl_up(a, off, 64), y = __shfl_up(b, off, 64);
        if (lane >= off) {
            a += x;
            b += y;
        }
    }
    if (lane == 63) {
        s_cell[wv] = a;
        s_mode[wv] = b;
    }
    __syncthreads();
    a -= cells;
    b -= modes;
    for (int w = 0; w < wv; w++) {
        a += s_cell[w];
        b += s_mode[w];
    }
    // a cells and b modes before this thread's
    for (int q = q0; q < q1; q++) {
        if (!bad && c.first[q] != q) continue;
        c.start[a++] = b;
        const int size = bad ? 1 : c.size[q];
        c.size[q] = b;  // now the cell's place, read by its members below
        b += size;
    }
    if (tid == 1023) {
        c.start[a] = K;
        *c.count = a;
    }
    __threadfence_block();
    __syncthreads();
    for (int q = tid; q < K; q += 1024) c.member[bad ? q : c.size[c.first[q]] + c.rank[q]] = q;
}

int launch_cell_index(const int *m, const int *k, const int *n, int K, const int *row_a,
                      const int *row_b, int width, void *ws, CellIndex &out, hipStream_t stream)
{
    const CellWs c = cell_ws(ws, K);
    const dim3 per4((K + 3) / 4);
    const bool rows = row_a && row_b;
    if (rows) {
        hipLaunchKernelGGL(cell_hash_kernel, per4, dim3(256), 0, stream, row_a, row_b, width, K, c);
        FEW_HIP(hipGetLastError());
    }
    hipLaunchKernelGGL(cell_match_kernel, dim3((K + 63) / 64), dim3(64 * CELL_WAVES), 0, stream, m,
                       k, n, K, c, rows ? 1 : 0);
    FEW_HIP(hipGetLastError());
    if (rows) {
        hipLaunchKernelGGL(cell_verify_kernel, per4, dim3(256), 0, stream, row_a, row_b, width, K,
                           c);
        FEW_HIP(hipGetLastError());
    }
    hipLaunchKernelGGL(cell_layout_kernel, dim3(1), dim3(1024), 0, stream, K, c, rows ? 1 : 0);
    FEW_HIP(hipGetLastError());
    out.count = c.count;
    out.start = c.start;
    out.member = c.member;
    return FEW_OK;
}

}  // namespace few
