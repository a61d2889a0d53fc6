// egx_build.hip -- COO/CSR -> pull CSC on the device.
//
// Reproduces build_inbound_from_csr (Easy-Graph/gpu_easygraph/functions/
// centrality/pagerank.cu:286-347) bit for bit, without its single-threaded
// host passes:
//   * the stable counting pass over u ascending (:328-346) becomes a stable
//     LSD radix sort of (dst, slot) pairs; the input is in out-CSR order
//     (source ascending), so sources stay ascending inside each dst row and
//     duplicate arcs keep their CSR order;
//   * in_row (:318-319) is the lower bound of every row id in the sorted
//     keys, i.e. the exclusive scan of the in-degree;
//   * endpoints outside [0, n) sort into a sentinel bucket past row n-1 and
//     are dropped (:282-284, :310); non-finite or negative weights count as 0
//     (:311-312);
//   * out-weights are summed per row, sequentially in CSR order, in FP64, so
//     fl32(alpha * (w / outW)) (:344) rounds exactly as the reference does.
#include <algorithm>
#include <cstdlib>
#include <chrono>
#include <cmath>
#include <vector>

#include "egx_graph.h"

namespace egx {

namespace {

// Row of every arc of a run.  One binary search per arc over the whole
// offset array was 80-100 us of every pass over 7-9M arcs (20 dependent
// loads each).  A workgroup now finds the rows of its first and last arc by
// a 64-way search (four loads deep at a million rows), marks the first arc
// of each row in between and spreads the marks by a running maximum.
constexpr int kRunThreads = 512;
constexpr int kRunItems = 8;
constexpr int kRunArcs = kRunThreads * kRunItems;  // arcs per workgroup
// A run that spans more rows than this (most of them without arcs) has each
// arc search between the first and the last instead: marking walks every row.
// 1M arcs, us of k_arc_keys and k_layout_slots with marks | searches at 16K
// rows a run 17 and 41 | 38 and 59, at 32K 27 and 58 | 43 and 71, at 64K 62 and 93 |
// 60 and 91, at 128K 141 and 172 | 86 and 130, at 256K 283 and 304 | 110 and 155.
constexpr int32_t kRunStretch = 65536;
struct RunRows {
    int4 mark[kRunArcs / 4];
    int32_t wave_max[kRunThreads / kWave];
    int32_t ends[2];
};

// The last u in [0, n] with V[u] <= p, for V[0] <= p < V[n]; all 64 lanes take part.
__device__ __forceinline__ int32_t wave_row_of(const int32_t* __restrict__ V, int32_t n, int64_t p) {
    int32_t lo = 0;
    int64_t hi = (int64_t)n + 1;
    while (hi - lo > 1) {
        const int64_t w = (hi - lo + kWave - 1) / kWave;
        const int64_t at = lo + (lane_id() + 1) * w;
        const bool below = at < hi && (int64_t)V[at] <= p;
        const int32_t c = __popcll(__ballot(below));
        lo = (int32_t)(lo + c * w);
        hi = min(hi, lo + w);
    }
    return lo;
}

// rows: rows[i] = row of arc q0 + i, i in [0, cnt), cnt <= kRunArcs, q0 + cnt <= V[n].
// Every thread of a kRunThreads workgroup takes part; the result is valid
// after the call.
__device__ __forceinline__ const int32_t* run_rows(const int32_t* __restrict__ V, int32_t n, int64_t q0, int32_t cnt,
                                                   RunRows& sh) {
    const int t = threadIdx.x;
    int32_t* mark = reinterpret_cast<int32_t*>(sh.mark);
    if (wave_id() < 2) {
        const int32_t r = wave_row_of(V, n, wave_id() == 0 ? q0 : q0 + cnt - 1);
        if (lane_id() == 0) sh.ends[wave_id()] = r;
    }
    for (int i = t; i < kRunArcs / 4; i += kRunThreads) sh.mark[i] = int4{0, 0, 0, 0};
    __syncthreads();
    const int32_t first = sh.ends[0], last = sh.ends[1];
    if (last - first > kRunStretch) {  // (uniform)
        for (int32_t i = t; i < cnt; i += kRunThreads) {
            int32_t lo = first, hi = last + 1;  // V[lo] <= q0 + i, and it is below V[hi] or hi is past the last
            while (hi - lo > 1) {
                const int32_t mid = lo + (hi - lo) / 2;
                if (V[mid] <= q0 + i) lo = mid;
                else hi = mid;
            }
            mark[i] = lo;
        }
        __syncthreads();
        return mark;
    }
    // a row's first arc gets the row; of the rows that share it (all but the last have no arcs) the last wins
    for (int32_t r = first + 1 + t; r <= last; r += kRunThreads) atomicMax(&mark[V[r] - q0], r);
    if (t == 0) atomicMax(&mark[0], first);
    __syncthreads();
    int4 a = sh.mark[2 * t], b = sh.mark[2 * t + 1];
    a.y = max(a.y, a.x); a.z = max(a.z, a.y); a.w = max(a.w, a.z);
    b.x = max(b.x, a.w); b.y = max(b.y, b.x); b.z = max(b.z, b.y); b.w = max(b.w, b.z);
    int32_t inc = b.w;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
        const int32_t o = __shfl_up(inc, off, kWave);
        if (lane_id() >= off) inc = max(inc, o);
    }
    int32_t prev = __shfl_up(inc, 1, kWave);
    if (lane_id() == 0) prev = 0;
    if (lane_id() == kWave - 1) sh.wave_max[wave_id()] = inc;
    __syncthreads();
    for (int w = 0; w < wave_id(); ++w) prev = max(prev, sh.wave_max[w]);
    sh.mark[2 * t] = int4{max(a.x, prev), max(a.y, prev), max(a.z, prev), max(a.w, prev)};
    sh.mark[2 * t + 1] = int4{max(b.x, prev), max(b.y, prev), max(b.z, prev), max(b.w, prev)};
    __syncthreads();
    return mark;
}
static_assert(kRunItems == 8, "a thread spreads two int4 of marks");

// What a weighted arc carries to its place in the pull CSC: gathered as one
// 16-byte record instead of its weight, source and the source's out-weight
// one by one (k_fill_csc over 9.3M arcs: 310 us).
struct __align__(16) ArcRec {
    double w;     // sanitised weight
    int32_t src;
    float val;    // fl32(alpha * (w / outW[src])), pagerank.cu:344
};

// Sort keys (head, or n past the valid ones) and payloads of every arc: the
// source, or for weighted arcs the arc's slot, with its record.
template <bool HasW>
__global__ __launch_bounds__(kRunThreads) void k_arc_keys(const int32_t* __restrict__ V, const int32_t* __restrict__ E,
                                                          const double* __restrict__ W,
                                                          const double* __restrict__ out_w, int32_t n, int64_t m,
                                                          double alpha, uint32_t* __restrict__ keys,
                                                          uint32_t* __restrict__ vals, ArcRec* __restrict__ rec,
                                                          uint32_t* __restrict__ invalid_count) {
    __shared__ RunRows sh;
    __shared__ uint32_t bad;
    if (threadIdx.x == 0) bad = 0;  // run_rows has barriers before it is used
    const int64_t q0 = (int64_t)blockIdx.x * kRunArcs;
    const int32_t cnt = (int32_t)min((int64_t)kRunArcs, m - q0);
    const int32_t* rows = run_rows(V, n, q0, cnt, sh);
    for (int32_t i = threadIdx.x; i < cnt; i += kRunThreads) {
        const int64_t p = q0 + i;
        const int32_t v = E[p];
        const int32_t u = rows[i];
        const bool valid = (0 <= v) && (v < n);
        keys[p] = valid ? (uint32_t)v : (uint32_t)n;
        vals[p] = HasW ? (uint32_t)p : (uint32_t)u;
        if (!valid) atomicAdd(&bad, 1u);
        if (HasW) {
            double w = W[p];
            if (!isfinite(w) || w < 0.0) w = 0.0;
            const double denom = out_w[u];
            rec[p] = ArcRec{w, u, (denom > 0.0) ? (float)(alpha * (w / denom)) : 0.0f};
        }
    }
    __syncthreads();
    if (threadIdx.x == 0 && bad) atomicAdd(invalid_count, bad);
}

// Counters of a build.
enum : int {
    kCtrInvalid,   // arcs with an endpoint outside [0, n)
    kCtrDangling,  // nodes without out-weight
    kCtrMaxOut,    // largest out-degree
    kCtrMaxIn,     // largest in-degree
    kCtrLong,      // rows longer than kOutLong
    kCtrHubs,      // rows above the hub threshold,
    kCtrHubArcs,   // their arcs,
    kCtrHubSegs,   // their segments,
    kCtrHubSplit,  // those of more than one segment
    kCtrHubMany,   // and of kHubMany or more
    kCtrWords = 16  // 64 bytes: a clear is one launch
};

// The weight of arc p as the build counts it (pagerank.cu:308-315): 0 when
// its endpoint is outside [0, n) or the weight is not finite or negative.
template <bool HasW>
__device__ __forceinline__ double arc_weight(const int32_t* __restrict__ E, const double* __restrict__ W, int64_t p,
                                             int32_t n, int32_t& cnt) {
    const int32_t v = E[p];
    if (v < 0 || v >= n) return 0.0;
    ++cnt;
    if (!HasW) return 1.0;
    const double w = W[p];
    return (!isfinite(w) || w < 0.0) ? 0.0 : w;
}

// Out-weight and valid out-arc count of every row.  The sum is the one of
// adding the row's weights one after the other in CSR order (pagerank.cu:308-315),
// bit for bit.  A workgroup takes the rows whose merge-path diagonal (the arcs
// and the rows before them) begins in its kOutTile, so that rows without arcs
// are shared out too (by arcs alone, one workgroup took all that follow each
// other: a build of 16 weighted arcs and 16M nodes 37 ms, now 0.8):
// their arcs come in whole lines into LDS, where each row has a thread that
// adds them (8 lanes per row that loaded their own arcs and passed them on
// by shuffles: 190 us for 9.3M arcs; one thread walking a row in memory paid a
// latency per arc, 95 ns).  Rows longer than kOutLong, listed beforehand,
// are the first workgroups' of the same launch: one of them each (they ran
// 114 us by themselves).  9.3M weighted arcs: 304 us -> 113, the longest row's
// chain of additions, and 18 for the list.
constexpr int kOutThreads = 256;
constexpr int32_t kOutLong = 256;
constexpr int32_t kOutTile = 4096;
constexpr int kLongStage = 1024;
constexpr int kLongBlocks = 1024;
struct OutTile {
    double w[kOutTile + kOutLong];
    int32_t rows[2];
    uint32_t bad;
};
struct OutLong {
    double stage[2][kLongStage];
    double s[4];
    int32_t c[4], low[4];
};

// First row whose diagonal V[r] + r is at least q, n if none is, by one wavefront.
__device__ __forceinline__ int32_t wave_first_row(const int32_t* __restrict__ V, int32_t n, int64_t q) {
    int32_t lo = 0, hi = n;
    while (lo < hi) {
        const int64_t step = ((int64_t)hi - lo + kWave - 1) / kWave;
        const int64_t at = (int64_t)lo + (lane_id() + 1) * step - 1;
        const bool below = at < hi && V[at] + at < q;
        const int k = __popcll(__ballot(below));  // diagonals ascend: a prefix of the lanes
        const int64_t nlo = (int64_t)lo + k * step, nhi = nlo + step - 1;
        lo = (int32_t)min(nlo, (int64_t)hi);
        hi = (int32_t)min(nhi, (int64_t)hi);
    }
    return __builtin_amdgcn_readfirstlane(lo);
}

template <bool HasW>
__device__ __forceinline__ void row_out_tile(const int32_t* __restrict__ V, const int32_t* __restrict__ E,
                                             const double* __restrict__ W, int32_t n, int64_t tile,
                                             double* __restrict__ out_w, int32_t* __restrict__ outcnt, OutTile& sh) {
    const int t = threadIdx.x;
    if (t == 0) sh.bad = 0;
    if (wave_id() < 2) {
        const int32_t r = wave_first_row(V, n, (tile + wave_id()) * kOutTile);
        if (lane_id() == 0) sh.rows[wave_id()] = r;
    }
    __syncthreads();
    const int32_t r0 = sh.rows[0], r1 = sh.rows[1];
    if (r0 >= r1) return;  // (uniform)
    // the arcs of these rows, but no further than a short row that begins here
    // could reach: every row begins less than kOutTile arcs after the first
    const int64_t a0 = V[r0], a1 = min((int64_t)V[r1], a0 + kOutTile + kOutLong);
    for (int64_t p = a0 + t; p < a1; p += kOutThreads) {
        int32_t ok = 0;
        const double w = arc_weight<HasW>(E, W, p, n, ok);
        sh.w[p - a0] = w;
        if (!ok) sh.bad = 1;
    }
    __syncthreads();
    const bool bad = sh.bad != 0;
    for (int32_t r = r0 + t; r < r1; r += kOutThreads) {
        const int32_t beg = V[r], len = V[r + 1] - beg;
        if (len > kOutLong) continue;
        int32_t c = len;
        if (bad) {
            c = 0;
            for (int32_t k = 0; k < len; ++k) {
                const int32_t v = E[beg + k];
                c += (v >= 0 && v < n) ? 1 : 0;
            }
        }
        double s = 0.0;
        if (HasW) {
            const double* w = sh.w + (beg - a0);
            for (int32_t k = 0; k < len; ++k) s += w[k];
        }
        out_w[r] = HasW ? s : (double)c;
        outcnt[r] = c;
    }
}

// Exponent of the lowest set bit of w > 0 (finite).
__device__ __forceinline__ int32_t lowest_bit(double w) {
    const uint64_t b = (uint64_t)__double_as_longlong(w);
    const int32_t e = (int32_t)((b >> 52) & 0x7ffu);
    const uint64_t f = b & 0xfffffffffffffull;
    return e == 0 ? -1074 + (__ffsll((unsigned long long)f) - 1)
                  : e - 1075 + (__ffsll((unsigned long long)(f | 0x10000000000000ull)) - 1);
}

// Rows above kOutLong arcs, one workgroup each.  When every partial sum is
// exact the order does not matter: all weights are multiples of 2^low, so
// with a total below 2^(low + 53) nothing was rounded (a rounded partial
// sum is at least that, and sums of non-negative terms never shrink), and
// the parallel sum is the sequential one.  That holds for unit weights and
// for weights that came from 32-bit floats.  Other rows are staged through
// LDS and added in CSR order by one wavefront.
template <bool HasW>
__device__ __forceinline__ void row_out_long(const int32_t* __restrict__ V, const int32_t* __restrict__ E,
                                             const double* __restrict__ W, int32_t n, uint32_t first, uint32_t step,
                                             double* __restrict__ out_w, int32_t* __restrict__ outcnt,
                                             const int32_t* __restrict__ long_rows, uint32_t rows, OutLong& sh) {
    const int t = threadIdx.x;
    for (uint32_t i = first; i < rows; i += step) {
        const int32_t u = long_rows[i];
        const int32_t beg = V[u], end = V[u + 1];
        double s = 0.0;
        int32_t c = 0, low = 4096;
        for (int64_t p = (int64_t)beg + t; p < end; p += 256) {
            const double w = arc_weight<HasW>(E, W, p, n, c);
            s += w;
            if (HasW && w > 0.0) low = min(low, lowest_bit(w));
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            s += __shfl_xor(s, off, kWave);
            c += __shfl_xor(c, off, kWave);
            low = min(low, __shfl_xor(low, off, kWave));
        }
        if (lane_id() == 0) {
            sh.s[wave_id()] = s;
            sh.c[wave_id()] = c;
            sh.low[wave_id()] = low;
        }
        __syncthreads();
        s = (sh.s[0] + sh.s[1]) + (sh.s[2] + sh.s[3]);
        c = sh.c[0] + sh.c[1] + sh.c[2] + sh.c[3];
        low = min(min(sh.low[0], sh.low[1]), min(sh.low[2], sh.low[3]));
        const bool exact = !HasW || low == 4096 || s < ldexp(1.0, low + 53);  // uniform over the workgroup
        if (!exact) {
            int32_t dummy = 0;
            double run = 0.0;
            for (int32_t q = t; q < kLongStage; q += 256)
                sh.stage[0][q] = (int64_t)beg + q < end ? arc_weight<HasW>(E, W, (int64_t)beg + q, n, dummy) : 0.0;
            __syncthreads();
            int cur = 0;
            for (int64_t p = beg; p < end; p += kLongStage, cur ^= 1) {
                if (wave_id() == 0) {  // every lane reads the same entries
                    const double* st = sh.stage[cur];
#pragma unroll 16
                    for (int q = 0; q < kLongStage; ++q) run += st[q];
                } else {
                    const int64_t nb = p + kLongStage;
                    for (int32_t q = t - kWave; q < kLongStage; q += 256 - kWave)
                        sh.stage[cur ^ 1][q] = nb + q < end ? arc_weight<HasW>(E, W, nb + q, n, dummy) : 0.0;
                }
                __syncthreads();
            }
            s = run;
        }
        if (t == 0) {
            out_w[u] = s;
            outcnt[u] = c;
        }
        __syncthreads();  // sh is reused by the next row
    }
}

// Workgroups [0, long_blocks) take the listed rows, the others a tile each.
template <bool HasW>
__global__ __launch_bounds__(kOutThreads) void k_row_out(const int32_t* __restrict__ V, const int32_t* __restrict__ E,
                                                         const double* __restrict__ W, int32_t n,
                                                         double* __restrict__ out_w, int32_t* __restrict__ outcnt,
                                                         const int32_t* __restrict__ long_rows,
                                                         const uint32_t* __restrict__ n_long, uint32_t long_blocks) {
    __shared__ union {
        OutTile tile;
        OutLong row;
    } sh;
    if (blockIdx.x < long_blocks) {
        row_out_long<HasW>(V, E, W, n, blockIdx.x, long_blocks, out_w, outcnt, long_rows, *n_long, sh.row);
    } else {
        row_out_tile<HasW>(V, E, W, n, blockIdx.x - long_blocks, out_w, outcnt, sh.tile);
    }
}

// The rows longer than kOutLong.
__global__ void k_long_rows(const int32_t* __restrict__ V, int32_t n, int32_t* __restrict__ long_rows,
                            uint32_t* __restrict__ n_long) {
    const int32_t u = blockIdx.x * blockDim.x + threadIdx.x;
    const bool is_long = u < n && V[u + 1] - V[u] > kOutLong;
    const uint64_t mask = __ballot(is_long);
    if (mask == 0) return;
    uint32_t at = 0;
    if (lane_id() == 0) at = atomicAdd(n_long, (uint32_t)__popcll(mask));
    at = __builtin_amdgcn_readfirstlane(at);
    if (is_long) long_rows[at + __popcll(mask & ((1ull << lane_id()) - 1ull))] = u;
}

// Sum / maximum over a 256-thread workgroup, valid in thread 0.
__device__ __forceinline__ uint32_t block_sum_u32(uint32_t v, uint32_t* sh) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, kWave);
    __syncthreads();
    if (lane_id() == 0) sh[wave_id()] = v;
    __syncthreads();
    return sh[0] + sh[1] + sh[2] + sh[3];
}
__device__ __forceinline__ uint32_t block_max_u32(uint32_t v, uint32_t* sh) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = max(v, __shfl_xor(v, off, kWave));
    __syncthreads();
    if (lane_id() == 0) sh[wave_id()] = v;
    __syncthreads();
    return max(max(sh[0], sh[1]), max(sh[2], sh[3]));
}

// Node passes with counters run at most this many workgroups: each adds to a
// counter once, and device-wide atomics on one address cost some 25 ns each
// (one per 256 nodes took 67 us at 700K nodes).
constexpr int kNodeBlocks = 512;

// deg (0 == dangling), dangling count, max out-degree.  Count: the out-arcs
// are the offsets' differences, written here with the out-weights (1 each
// with unit_out, else the counts).
template <bool Count>
__global__ __launch_bounds__(256) void k_node_arrays(const int32_t* __restrict__ V, double* __restrict__ out_w,
                                                     int32_t* __restrict__ outcnt, int32_t n, int unit_out,
                                                     int weighted, float* __restrict__ deg,
                                                     uint32_t* __restrict__ ctr) {
    __shared__ uint32_t sh[4];
    uint32_t nd = 0, most = 0;
    for (int64_t u = (int64_t)blockIdx.x * 256 + threadIdx.x; u < n; u += (int64_t)gridDim.x * 256) {
        const int32_t c = Count ? V[u + 1] - V[u] : outcnt[u];
        const double w = Count ? (unit_out ? 1.0 : (double)c) : out_w[u];
        if (Count) {
            outcnt[u] = c;
            out_w[u] = w;
        }
        const bool dang = !(w > 0.0);  // pagerank.cu:323-326: outW <= 0
        deg[u] = weighted ? (dang ? 0.0f : 1.0f) : (dang ? 0.0f : (float)c);
        nd += dang ? 1u : 0u;
        most = max(most, (uint32_t)c);
    }
    nd = block_sum_u32(nd, sh);
    most = block_max_u32(most, sh);
    if (threadIdx.x == 0) {
        if (nd) atomicAdd(&ctr[kCtrDangling], nd);
        if (most) atomicMax(&ctr[kCtrMaxOut], most);
    }
}

__global__ void k_fill_csc(const uint32_t* __restrict__ vals, const ArcRec* __restrict__ rec, int64_t m_valid,
                           int32_t* __restrict__ in_col, float* __restrict__ in_val, double* __restrict__ w_csc) {
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= m_valid) return;
    const ArcRec r = rec[vals[q]];
    in_col[q] = r.src;
    w_csc[q] = r.w;
    in_val[q] = r.val;
}

__global__ void k_refresh_vals(const int32_t* __restrict__ in_col, const double* __restrict__ w_csc,
                               const double* __restrict__ out_w, int64_t m, double alpha,
                               float* __restrict__ in_val) {
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= m) return;
    const double denom = out_w[in_col[q]];
    in_val[q] = (denom > 0.0) ? (float)(alpha * (w_csc[q] / denom)) : 0.0f;
}

// Unit-weight in_val of the reference (W = ones): fl32(alpha * (1.0 / outW)).
__global__ void k_unit_vals(const int32_t* __restrict__ in_col, const double* __restrict__ out_w, int64_t m,
                            double alpha, float* __restrict__ in_val) {
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= m) return;
    const double denom = out_w[in_col[q]];
    in_val[q] = (denom > 0.0) ? (float)(alpha * (1.0 / denom)) : 0.0f;
}

// Largest in-degree, and the rows above the hub threshold.
__global__ __launch_bounds__(256) void k_in_degrees(const int32_t* __restrict__ in_row, int32_t n, int32_t hub,
                                                    int32_t seg, uint32_t* __restrict__ ctr) {
    __shared__ uint32_t sh[4];
    uint32_t most = 0, hubs = 0, arcs = 0, segs = 0, split = 0, many = 0;
    for (int64_t v = (int64_t)blockIdx.x * 256 + threadIdx.x; v < n; v += (int64_t)gridDim.x * 256) {
        const int32_t d = in_row[v + 1] - in_row[v];
        most = max(most, (uint32_t)d);
        if (d > hub) {
            const uint32_t k = ((uint32_t)d + (uint32_t)seg - 1u) / (uint32_t)seg;
            hubs += 1u;
            arcs += (uint32_t)d;
            segs += k;
            split += k > 1u ? 1u : 0u;
            many += k >= (uint32_t)kHubMany ? 1u : 0u;
        }
    }
    most = block_max_u32(most, sh);
    hubs = block_sum_u32(hubs, sh);
    if (threadIdx.x == 0 && most) atomicMax(&ctr[kCtrMaxIn], most);
    __shared__ uint32_t any;
    if (threadIdx.x == 0) any = hubs;
    __syncthreads();
    if (any == 0) return;
    arcs = block_sum_u32(arcs, sh);
    segs = block_sum_u32(segs, sh);
    split = block_sum_u32(split, sh);
    many = block_sum_u32(many, sh);
    if (threadIdx.x == 0) {
        atomicAdd(&ctr[kCtrHubs], hubs);
        atomicAdd(&ctr[kCtrHubArcs], arcs);
        atomicAdd(&ctr[kCtrHubSegs], segs);
        if (split) atomicAdd(&ctr[kCtrHubSplit], split);
        if (many) atomicAdd(&ctr[kCtrHubMany], many);
    }
}

// First segment of every hub row (rows [0, n_hub); one past them at n_hub),
// and the rows of several segments: those of kHubMany or more first, each
// part in row order.  One workgroup; with the counts known from the degrees
// the host waits for none of it (it read the offsets back and copied both
// lists up: a build and solve of 16,384 nodes 381 us, 374 so).
constexpr int kHubThreads = 1024;
__global__ __launch_bounds__(kHubThreads) void k_hub_rows(const int32_t* __restrict__ row, int32_t n_hub, int32_t seg,
                                                          int32_t n_many, int32_t* __restrict__ first,
                                                          HubRow* __restrict__ rows) {
    __shared__ int32_t sums[3][kHubThreads / kWave];
    int32_t base[3] = {0, 0, n_many};  // segments, rows of many, other rows of several
    const int l = lane_id();
    const uint64_t below = (1ull << l) - 1ull;
    for (int32_t v0 = 0; v0 < n_hub; v0 += kHubThreads) {
        const int32_t v = v0 + (int32_t)threadIdx.x;
        const int32_t len = v < n_hub ? row[v + 1] - row[v] : 0;
        const int32_t k = (int32_t)(((int64_t)len + seg - 1) / seg);
        const bool is_many = k >= kHubMany, is_split = k > 1 && !is_many;
        int32_t inc = k;
#pragma unroll
        for (int off = 1; off < kWave; off <<= 1) {
            const int32_t o = __shfl_up(inc, off, kWave);
            if (l >= off) inc += o;
        }
        const uint64_t bm = __ballot(is_many), bs = __ballot(is_split);
        if (l == kWave - 1) {
            sums[0][wave_id()] = inc;
            sums[1][wave_id()] = __popcll(bm);
            sums[2][wave_id()] = __popcll(bs);
        }
        __syncthreads();
        int32_t at[3] = {base[0] + inc - k, base[1] + (int32_t)__popcll(bm & below),
                         base[2] + (int32_t)__popcll(bs & below)};
        for (int q = 0; q < 3; ++q)
            for (int w = 0; w < kHubThreads / kWave; ++w) {
                base[q] += sums[q][w];
                if (w < wave_id()) at[q] += sums[q][w];
            }
        if (v < n_hub) first[v] = at[0];
        if (is_many) rows[at[1]] = HubRow{v, at[0], k, 0};
        if (is_split) rows[at[2]] = HubRow{v, at[0], k, 0};
        __syncthreads();  // sums is reused
    }
    if (threadIdx.x == 0) first[n_hub] = base[0];
}

__global__ void k_hub_segs(const int32_t* __restrict__ row, const int32_t* __restrict__ first, int32_t n_hub,
                           int32_t seg, int32_t n_segs, HubSeg* __restrict__ out) {
    const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n_segs) return;
    int32_t lo = 0, hi = n_hub;  // first[lo] <= i < first[hi]
    while (hi - lo > 1) {
        const int32_t mid = lo + ((hi - lo) >> 1);
        if (first[mid] <= i) lo = mid;
        else hi = mid;
    }
    HubSeg sg;
    sg.row = lo;
    sg.beg = row[lo] + (i - first[lo]) * seg;
    sg.end = (int32_t)min((int64_t)sg.beg + seg, (int64_t)row[lo + 1]);
    sg.slot = lo;
    sg.nseg = first[lo + 1] - first[lo];
    sg.first = first[lo];
    out[i] = sg;
}

// Relabelling key: hub rows (in-degree > hub) first, then descending
// out-degree when reorder is on; the stable sort keeps ids ascending among
// equal keys.  perm[r] = original id of row r, rank = its inverse.
__global__ void k_layout_keys(const int32_t* __restrict__ in_row, const int32_t* __restrict__ out_cnt, int32_t n,
                              int32_t hub, int32_t bits, uint32_t maxdeg, int reorder, uint32_t* __restrict__ keys,
                              uint32_t* __restrict__ vals, int32_t* __restrict__ pad) {
    const int32_t v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v < kArcPad) pad[v] = 0;  // the zeroed slots past in_col's arcs
    if (v >= n) return;
    const bool is_hub = (in_row[v + 1] - in_row[v]) > hub;
    const uint32_t sec = reorder ? (maxdeg - (uint32_t)out_cnt[v]) : 0u;
    keys[v] = ((is_hub ? 0u : 1u) << bits) | sec;
    vals[v] = (uint32_t)v;
}

// tiles[k] = first row v in [n_hub, n] whose merge-path diagonal
// (it_row[v] - it_row[n_hub]) + (v - n_hub) reaches k * tile_items.
__global__ void k_tile_starts(const int32_t* __restrict__ row, int32_t n_hub, int32_t n, int32_t tile_items,
                              int64_t n_tiles, int32_t* __restrict__ tiles, uint32_t* __restrict__ wave_rows) {
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k == 0) *wave_rows = 0;
    if (k > n_tiles) return;
    if (k == n_tiles) {
        tiles[k] = n;
        return;
    }
    const int64_t target = k * (int64_t)tile_items;
    const int64_t base = row[n_hub];
    int32_t lo = n_hub, hi = n;
    while (lo < hi) {
        const int32_t mid = lo + ((hi - lo) >> 1);
        const int64_t diag = ((int64_t)row[mid] - base) + (int64_t)(mid - n_hub);
        if (diag < target) lo = mid + 1;
        else hi = mid;
    }
    tiles[k] = lo;
}

// Sort keys of the tile arcs: (tile << 32 | source), payload = arc index.
__global__ void k_tile_sort_keys(const int32_t* __restrict__ row, const int32_t* __restrict__ col,
                                 const int32_t* __restrict__ tiles, uint64_t* __restrict__ keys,
                                 uint32_t* __restrict__ vals, int64_t base) {
    const int32_t k = blockIdx.x;
    const int32_t a0 = row[tiles[k]], a1 = row[tiles[k + 1]];
    for (int32_t p = a0 + (int32_t)threadIdx.x; p < a1; p += blockDim.x) {
        keys[p - base] = ((uint64_t)(uint32_t)k << 32) | (uint64_t)(uint32_t)col[p];
        vals[p - base] = (uint32_t)(p - base);
    }
}

// t_col / t_pos (and t_val) of tile k from its sorted (key, arc) pairs.
__global__ void k_tile_sorted_arrays(const int32_t* __restrict__ row, const int32_t* __restrict__ tiles,
                                     const uint64_t* __restrict__ keys, const uint32_t* __restrict__ vals,
                                     const float* __restrict__ val, int64_t base, int32_t* __restrict__ t_col,
                                     uint16_t* __restrict__ t_pos, float* __restrict__ t_val) {
    const int32_t k = blockIdx.x;
    const int32_t a0 = row[tiles[k]], a1 = row[tiles[k + 1]];
    for (int32_t p = a0 + (int32_t)threadIdx.x; p < a1; p += blockDim.x) {
        const int64_t arc = base + (int64_t)vals[p - base];
        t_col[p] = (int32_t)(uint32_t)keys[p - base];
        t_pos[p] = (uint16_t)(arc - a0);
        if (t_val) t_val[p] = val[arc];
    }
}

// t_val of every tile from t_pos (after an alpha change).
__global__ void k_tile_vals(const int32_t* __restrict__ row, const int32_t* __restrict__ tiles,
                            const uint16_t* __restrict__ t_pos, const float* __restrict__ val,
                            float* __restrict__ t_val) {
    const int32_t k = blockIdx.x;
    const int32_t a0 = row[tiles[k]], a1 = row[tiles[k + 1]];
    for (int32_t p = a0 + (int32_t)threadIdx.x; p < a1; p += blockDim.x) t_val[p] = val[a0 + t_pos[p]];
}

__global__ void k_layout_nodes(const uint32_t* __restrict__ perm, const int32_t* __restrict__ in_row,
                               const float* __restrict__ deg, const double* __restrict__ out_w, int32_t n,
                               int32_t* __restrict__ rank, uint32_t* __restrict__ cnt, float* __restrict__ p_deg,
                               double* __restrict__ p_outw, int32_t* __restrict__ pad) {
    const int32_t r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r < kArcPad) pad[r] = 0;  // the zeroed slots past p_col's arcs
    if (r == 0) cnt[n] = 0;
    if (r >= n) return;
    const int32_t v = (int32_t)perm[r];
    rank[v] = r;
    cnt[r] = (uint32_t)(in_row[v + 1] - in_row[v]);
    p_deg[r] = deg[v];
    p_outw[r] = out_w[v];
}

// Every relabelled CSC slot: its row, and the arc with its source relabelled.
__global__ __launch_bounds__(kRunThreads) void k_layout_slots(
    const int32_t* __restrict__ p_row, const int32_t* __restrict__ perm, const int32_t* __restrict__ rank,
    const int32_t* __restrict__ in_row, const int32_t* __restrict__ in_col, const float* __restrict__ in_val,
    const double* __restrict__ w_csc, int32_t n, int64_t m, int weighted, int32_t* __restrict__ p_col,
    float* __restrict__ p_val, double* __restrict__ p_w) {
    __shared__ RunRows sh;
    const int64_t q0 = (int64_t)blockIdx.x * kRunArcs;
    const int32_t cnt = (int32_t)min((int64_t)kRunArcs, m - q0);
    const int32_t* rows = run_rows(p_row, n, q0, cnt, sh);
#pragma unroll 4
    for (int32_t i = threadIdx.x; i < cnt; i += kRunThreads) {
        const int64_t q = q0 + i;
        const int32_t r = rows[i];
        const int64_t src_slot = (int64_t)in_row[perm[r]] + (q - p_row[r]);
        p_col[q] = rank[in_col[src_slot]];
        if (weighted) {
            p_val[q] = in_val[src_slot];
            p_w[q] = w_csc[src_slot];
        }
    }
}

// Non-hub rows with more than row_lane_max arcs (egx_graph_info).
__global__ __launch_bounds__(256) void k_row_stats(const int32_t* __restrict__ row, int32_t n_hub, int32_t n,
                                                   int32_t lane_max, uint32_t* __restrict__ wave_rows) {
    __shared__ uint32_t sh[4];
    uint32_t rows = 0;
    for (int64_t v = n_hub + (int64_t)blockIdx.x * 256 + threadIdx.x; v < n; v += (int64_t)gridDim.x * 256)
        rows += row[v + 1] - row[v] > lane_max ? 1u : 0u;
    rows = block_sum_u32(rows, sh);
    if (threadIdx.x == 0 && rows) atomicAdd(wave_rows, rows);
}

__global__ void k_check_arcs(const int32_t* __restrict__ E, const double* __restrict__ W, int32_t n, int64_t m,
                             uint32_t* __restrict__ flags) {
    uint32_t f = 0;
    for (int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; p < m; p += (int64_t)gridDim.x * blockDim.x) {
        const int32_t v = E[p];
        if (v < 0 || v >= n) f |= kArcBadEndpoint;
        if (W) {
            const double w = W[p];
            if (!isfinite(w) || w < 0.0) f |= kArcBadWeight;
        }
    }
    if (f) atomicOr(flags, f);
}

// Rows of many partials first (in their order); returns how many those are.
int64_t many_first(std::vector<HubRow>& rows) {
    return std::stable_partition(rows.begin(), rows.end(), [](const HubRow& h) { return h.nseg >= kHubMany; }) -
           rows.begin();
}

// The in-degree above which a row is a hub row.
inline int32_t hub_threshold(const BinCfg& cfg) { return std::min(std::max(cfg.wave_row_max, 1), kTileLds - 256); }

// Arcs per hub segment.
inline int32_t hub_segment(const BinCfg& cfg) { return std::max(cfg.hub_segment, 256); }

inline unsigned nblocks(int64_t n, int threads) { return (unsigned)((n + threads - 1) / threads); }

}  // namespace

// Source-ordered copies of the tile arcs (or none when cfg.tile_sort is 0).
// A tile holds at most kTileLds arcs, so an arc's slot fits 16 bits.
int build_tile_sort(Graph& g, const BinCfg& cfg) {
    g.tsorted = false;
    g.t_col.release();
    g.t_pos.release();
    g.t_val.release();
    if (!cfg.tile_sort || g.n_tiles == 0) return EGX_SUCC;
    hipStream_t s = g.stream;
    int32_t base32 = 0;
    EGX_HIP_TRY(hipMemcpyWithStream(&base32, g.it_row + g.n_hub, 4, hipMemcpyDeviceToHost, s), EGX_DEVICE_ERR);
    const int64_t base = base32;
    const int64_t mt = g.m - base;
    if (mt <= 0) return EGX_SUCC;
    const size_t mm = (size_t)std::max<int64_t>(g.m, 1);
    EGX_TRY(g.t_col.alloc(mm * 4));
    EGX_TRY(g.t_pos.alloc(mm * 2));
    if (g.has_values()) EGX_TRY(g.t_val.alloc(mm * 4));
    {
        DevBuf keys, keys_alt, vals, vals_alt;
        EGX_TRY(keys.alloc((size_t)mt * 8));
        EGX_TRY(keys_alt.alloc((size_t)mt * 8));
        EGX_TRY(vals.alloc((size_t)mt * 4));
        EGX_TRY(vals_alt.alloc((size_t)mt * 4));
        const unsigned nt = (unsigned)g.n_tiles;
        k_tile_sort_keys<<<nt, 256, 0, s>>>(g.it_row, g.it_col, g.tiles.as<int32_t>(), keys.as<uint64_t>(),
                                            vals.as<uint32_t>(), base);
        EGX_CHECK_LAUNCH(EGX_DEVICE_ERR);
        EGX_TRY(radix_sort_u64(keys, keys_alt, &vals, &vals_alt, mt, 32 + bits_for((uint64_t)g.n_tiles), s));
        k_tile_sorted_arrays<<<nt, 256, 0, s>>>(g.it_row, g.tiles.as<int32_t>(), keys.as<uint64_t>(),
                                                vals.as<uint32_t>(), g.it_val, base, g.t_col.as<int32_t>(),
                                                g.t_pos.as<uint16_t>(), g.has_values() ? g.t_val.as<float>() : nullptr);
        EGX_CHECK_LAUNCH(EGX_DEVICE_ERR);
        EGX_HIP_TRY(hipStreamSynchronize(s), EGX_DEVICE_ERR);
    }
    g.tsorted = true;
    return EGX_SUCC;
}

namespace {

// Run key of every arc, (chunk of its source) * B + (sub-bin of its row),
// with the arc's CSC position as the value: a stable sort by key keeps CSC
// order (row, then position) inside every run.
__global__ __launch_bounds__(kRunThreads) void k_pb_keys(const int32_t* __restrict__ row,
                                                         const int32_t* __restrict__ col, int32_t n, int64_t m,
                                                         int64_t B, uint32_t* __restrict__ keys,
                                                         uint32_t* __restrict__ vals, int32_t* __restrict__ rowof) {
    __shared__ RunRows sh;
    const int64_t q0 = (int64_t)blockIdx.x * kRunArcs;
    const int32_t cnt = (int32_t)min((int64_t)kRunArcs, m - q0);
    const int32_t* rows = run_rows(row, n, q0, cnt, sh);
    for (int32_t i = threadIdx.x; i < cnt; i += kRunThreads) {
        const int64_t e = q0 + i;
        const int32_t r = rows[i];
        keys[e] = (uint32_t)((int64_t)(col[e] / kPbChunk) * B + r / kPbRows);
        vals[e] = (uint32_t)e;
        rowof[e] = r;
    }
}

// Source slots of every run (its arcs rounded up to kPbVec) from the lower
// bounds of the sorted keys; entry `runs` is 0, so the exclusive scan ends
// with the total.
__global__ void k_pb_run_slots(const int32_t* __restrict__ lb, int64_t runs, uint32_t* __restrict__ out) {
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k > runs) return;
    out[k] = k < runs ? (uint32_t)((lb[k + 1] - lb[k] + kPbVec - 1) / kPbVec * kPbVec) : 0u;
}

__global__ void k_fill_u16(uint16_t* __restrict__ p, int64_t n, uint16_t v) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// Sorted arc i of run k to source slot soff[k] + (i - lb[k]): its source
// label inside the chunk and its row.  Anything out of range raises *bad.
__global__ void k_pb_place(const uint32_t* __restrict__ keys, const uint32_t* __restrict__ vals,
                           const int32_t* __restrict__ lb, const uint32_t* __restrict__ soff,
                           const int32_t* __restrict__ col, const int32_t* __restrict__ rowof, int64_t m,
                           int64_t runs, int64_t B, uint16_t* __restrict__ src16, int32_t* __restrict__ srow,
                           int32_t* __restrict__ arc, int32_t* __restrict__ bad) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= m) return;
    const uint32_t k = keys[i];
    const uint32_t e = vals[i];
    if ((int64_t)k >= runs || (int64_t)e >= m || i < lb[k]) {
        *bad = 1;
        return;
    }
    const int64_t p = (int64_t)soff[k] + (i - lb[k]);
    const int64_t u = (int64_t)col[e] - (int64_t)(k / B) * kPbChunk;
    if (p >= (int64_t)soff[k + 1] || u < 0 || u >= kPbChunk) {
        *bad = 1;
        return;
    }
    src16[p] = (uint16_t)u;
    srow[p] = rowof[e];
    if (arc) arc[p] = (int32_t)e;
}

// FP32 arc value of every source slot of a weighted graph (padding: 0).
__global__ void k_pb_gather_w(const int32_t* __restrict__ arc, const float* __restrict__ val, int64_t slots,
                              int64_t m, float* __restrict__ w) {
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= slots) return;
    const int32_t e = arc[p];
    w[p] = (e >= 0 && (int64_t)e < m) ? val[e] : 0.0f;
}

// Stretch mask of every kPbVec-slot group and its term count; entry
// `groups` of pc is 0 for the scan total.  Bit j >= 1: slot j starts a
// stretch of equal rows (padding slots, row -1, join the stretch before
// them).  Bit 0: the group's last stretch is a term of its own; with
// `merge` (weighted graphs) it is clear when the next group of the same
// kPbWindow-group window of the chunk starts with the same row, and the
// stretch's sum then goes into the next group's first term.
static_assert(kPbVec == 8, "a group is two int4 loads of rows");
__global__ void k_pb_masks(const int32_t* __restrict__ srow, int64_t groups, const uint32_t* __restrict__ soff,
                           int64_t S, int64_t B, bool merge, uint8_t* __restrict__ mask,
                           uint32_t* __restrict__ pc) {
    const int64_t gi = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (gi > groups) return;
    if (gi == groups) {
        pc[gi] = 0;
        return;
    }
    const int4 lo = reinterpret_cast<const int4*>(srow)[2 * gi];
    const int4 hi = reinterpret_cast<const int4*>(srow)[2 * gi + 1];
    const int32_t r[kPbVec] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
    uint32_t mk = 0;
    int32_t last = r[0];  // the group's last real row
#pragma unroll
    for (int j = 1; j < kPbVec; ++j) {
        if (r[j] >= 0 && r[j] != r[j - 1]) mk |= 1u << j;
        if (r[j] >= 0) last = r[j];
    }
    bool cont = false;
    const int64_t nx = gi + 1;
    if (merge && nx < groups && last >= 0) {
        // the chunk of the group: the last c with soff[c * B] <= its first slot
        const int64_t s0 = gi * kPbVec;
        int64_t lo_c = 0, hi_c = S;
        while (lo_c + 1 < hi_c) {
            const int64_t mid = (lo_c + hi_c) >> 1;
            if ((int64_t)soff[mid * B] <= s0) lo_c = mid;
            else hi_c = mid;
        }
        const int64_t c0 = (int64_t)soff[lo_c * B] / kPbVec;
        const int64_t c1 = (int64_t)soff[(lo_c + 1) * B] / kPbVec;
        if (nx < c1 && (nx - c0) % kPbWindow != 0) cont = srow[nx * kPbVec] == last;
    }
    if (!cont) mk |= 1u;
    mask[gi] = (uint8_t)mk;
    pc[gi] = (uint32_t)__popc(mk);
}

// Value slots of every run, rounded up to kPbVec, stored bin-major at
// b * S + c; entry `runs` is 0 for the scan total.  gs is the exclusive scan
// of the groups' value-slot counts.
__global__ void k_pb_run_values(const uint32_t* __restrict__ soff, const uint32_t* __restrict__ gs, int64_t runs,
                                int64_t S, int64_t B, uint32_t* __restrict__ pout) {
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k > runs) return;
    if (k == runs) {
        pout[runs] = 0;
        return;
    }
    const uint32_t o = gs[soff[k + 1] / kPbVec] - gs[soff[k] / kPbVec];
    pout[(k % B) * S + k / B] = (o + kPbVec - 1) / kPbVec * kPbVec;
}

// First value slot of every group and the sub-bin row of each of its value
// slots.  The group's run is the last run whose first slot is at or before
// the group's (empty runs share the next run's first slot).
__global__ void k_pb_groups(const uint32_t* __restrict__ soff, const uint32_t* __restrict__ gs,
                            const uint32_t* __restrict__ voff, const uint8_t* __restrict__ mask,
                            const int32_t* __restrict__ srow, int64_t groups, int64_t runs, int64_t S, int64_t B,
                            int32_t* __restrict__ vgrp, uint16_t* __restrict__ dst16, int32_t* __restrict__ bad) {
    const int64_t gi = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (gi >= groups) return;
    const int64_t s0 = gi * kPbVec;
    // first k in [0, runs] with soff[k] > s0; soff[runs] is the slot total
    int64_t lo = 0, hi = runs;
    while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if ((int64_t)soff[mid] <= s0) lo = mid + 1;
        else hi = mid;
    }
    const int64_t k = lo - 1;
    if (k < 0) {
        *bad = 1;
        return;
    }
    const int64_t v = (k % B) * S + k / B;
    const int64_t o = (int64_t)voff[v] + gs[gi] - gs[soff[k] / kPbVec];
    const uint32_t mk = mask[gi];
    if (o + __popc(mk) > (int64_t)voff[v + 1]) {
        *bad = 1;
        return;
    }
    vgrp[gi] = (int32_t)o;
    const int64_t r0 = (k % B) * kPbRows;
    // the rows of the group's terms: its stretches (slot 0 and every mask
    // bit j >= 1) in order, the first popcount(mk) of them (the last stretch
    // has none when bit 0 is clear)
    int64_t q = o;
    const int64_t end = o + __popc(mk);
    for (int j = 0; j < kPbVec && q < end; ++j)
        if (j == 0 || (mk & (1u << j))) {
            const int64_t d = (int64_t)srow[s0 + j] - r0;
            if (d < 0 || d >= kPbRows) {
                *bad = 1;
                return;
            }
            dst16[q++] = (uint16_t)d;
        }
}

// Work-item sizes of the blocked iteration, in slots (multiples of kPbVec).
// A scatter block holds a whole CU's LDS and stages its chunk's 128 KB of
// sources, so an item is at least 32K slots, and kPbCus items run at a time.
// Where such items of at most 64K slots fit one such round, the smallest that
// do are taken.  Larger graphs take total / items, down to 64K slots, which
// is one batch of 8 groups a lane (weighted: 32K, batches hold 2 groups).
// us per iteration with items of 32K -> 64K slots: 1,048,576 nodes and 16
// arcs each 50 -> 47, 2,097,152 89 -> 86, 4,194,304 151 -> 145; weighted, one
// round: 700,001 nodes 50 -> 41; weighted above that, 32K and 64K: 3,000,017
// nodes 124 and 127, R-MAT 24 with 64K to 256K 633 to 664.
constexpr int64_t kPbCus = 256;
constexpr int64_t kPbScatterItems = 1024;
constexpr int64_t kPbScatterItemsW = 4096;
constexpr int64_t kPbScatterMin = 32768;
constexpr int64_t kPbScatterMax1 = 65536;  // one round; unweighted graphs of several take no less
// A sum item is a workgroup; sub-bins larger than total / items value slots
// are cut into pieces, so that mid-size graphs (few sub-bins, long ones) fill
// the CUs and the heavy sub-bins of skewed graphs do not trail; each piece
// hands its row sums to the reduce launch.  From kPbSumBins sub-bins on fewer
// pieces are the better choice: us per iteration with total / 512 of 16K or
// more against total / 256 of 32K or more: 1,048,576 nodes 46.6 and 48.0,
// 2,097,152 85.0 and 77.7, 4,194,304 142.6 and 134.4, weighted 3,000,017 124
// and 119, R-MAT 24 494 and 494.
constexpr int64_t kPbSumBins = 1024;
constexpr int64_t kPbSumItems = 512, kPbSumMin = 16384;
constexpr int64_t kPbSumItemsMany = 256, kPbSumMinMany = 32768;
// Graphs laid out for shared launches: one size for all.  Scatter items of a
// chunk are joined by the launch when the set is large (kJoinSlots); sum
// items are not, so theirs is the one that costs large sets nothing.  us per
// iteration at 256K and 128K slots, 192K and 64K, 96K and 32K: 48 graphs of
// 1,000 to 300,000 nodes 130, 106, 104; 96 of them 189, 159, 179; 200 337,
// 342, 391; 512 of 1,000 to 1,000,000 2,399, 2,424, 2,791.
constexpr int64_t kPbScatterShared = 98304;
constexpr int64_t kPbSumShared = 65536;

int64_t pb_item_slots(int64_t total, int64_t items, int64_t lo, int64_t hi) {
    const int64_t want = (total / items) / kPbVec * kPbVec;
    return std::max<int64_t>(lo, std::min<int64_t>(hi, want));
}

}  // namespace

// Propagation-blocked layout of the iteration CSC (it_row, it_col), built on
// the device.  Arcs are bucketed by (chunk c, sub-bin b) into runs, in CSC
// order (row, then source) inside each run, each run padded to a multiple
// of kPbVec source slots.  Each kPbVec-slot group of a run is cut into
// stretches of equal rows (bit j of its mask marks a stretch starting at
// slot j); every stretch has one value slot.  Value slots follow
// (sub-bin, chunk) order, each run's stretches in group order, padded to a
// multiple of kPbVec (padding rows 0, values 0: never written).
//
// The runs come from a stable radix sort of the arcs by run key, the slot
// offsets from scans of rounded run sizes; only the run offsets (two arrays
// of S*B + 1 entries) come back to the host, which cuts them into scatter
// and sum work items.
int build_blocked(Graph& g, const BinCfg& cfg, bool layout_changed) {
    // the blocked layout depends only on the iteration CSC
    if (cfg.blocked && g.pb_ready && !layout_changed && g.pb_shared == cfg.blocked_shared) return EGX_SUCC;
    g.pb_ready = false;
    for (DevBuf* d : {&g.pb_src, &g.pb_dst, &g.pb_vals, &g.pb_vgrp, &g.pb_mask, &g.pb_scatter, &g.pb_sum,
                      &g.pb_hrows, &g.pb_hub_part, &g.pb_w, &g.pb_arc})
        d->release();
    g.n_pb_scatter = g.n_pb_sum = g.n_pb_hrows = g.n_pb_hrows_many = 0;
    g.pb_scatter_size.clear();
    g.pb_scatter_chunk.clear();
    g.pb_sum_size.clear();
    if (!cfg.blocked || g.n <= 0 || g.m <= 0) return EGX_SUCC;
    // test hook: a real device allocation failure at the start of the layout
    // build, for the fallback and error-state tests
    if (const char* e = std::getenv("EGGPU_AMD_TEST_FAIL_BLOCKED_ALLOC")) {
        if (e[0] == '1') {
            DevBuf huge;
            EGX_TRY(huge.alloc((size_t)1 << 52));
        }
    }
    const int32_t n = g.n;
    const int64_t m = g.m;
    const int64_t S = (n + kPbChunk - 1) / kPbChunk;
    const int64_t B = (n + kPbRows - 1) / kPbRows;
    const int64_t runs = S * B;
    if (runs > ((int64_t)1 << 28) || m > INT32_MAX) {
        set_last_error("graph too large for the propagation-blocked layout");
        return EGX_UNSUPPORTED_GRAPH;
    }
    hipStream_t s = g.stream;
    const unsigned tb = 256;

    // arcs sorted by run; lower bounds of every run key; source-slot offsets
    DevBuf rowof, keys, vals, lb, soff, bad;
    {
        DevBuf keys_alt, vals_alt;
        EGX_TRY(rowof.alloc((size_t)m * 4));
        EGX_TRY(keys.alloc((size_t)m * 4));
        EGX_TRY(vals.alloc((size_t)m * 4));
        EGX_TRY(keys_alt.alloc((size_t)m * 4));
        EGX_TRY(vals_alt.alloc((size_t)m * 4));
        k_pb_keys<<<nblocks(m, kRunArcs), kRunThreads, 0, s>>>(g.it_row, g.it_col, n, m, B, keys.as<uint32_t>(),
                                                               vals.as<uint32_t>(), rowof.as<int32_t>());
        EGX_CHECK_LAUNCH(EGX_DEVICE_ERR);
        EGX_TRY(radix_sort_u32(keys, keys_alt, &vals, &vals_alt, m, bits_for((uint64_t)(runs - 1)), s));
    }
    EGX_TRY(lb.alloc((size_t)(runs + 1) * 4));
    EGX_TRY(lower_bound_iota_u32(keys.as<uint32_t>(), m, lb.as<int32_t>(), runs + 1, s));
    EGX_TRY(soff.alloc((size_t)(runs + 1) * 4));
    k_pb_run_slots<<<nblocks(runs + 1, tb), tb, 0, s>>>(lb.as<int32_t>(), runs, soff.as<uint32_t>());
    EGX_CHECK_LAUNCH(EGX_DEVICE_ERR);
    EGX_TRY(exclusive_scan_u32(soff.as<uint32_t>(), soff.as<uint32_t>(), runs + 1, s));
    std::vector<uint32_t> soff_h((size_t)runs + 1);
    EGX_HIP_TRY(hipStreamSynchronize(s), EGX_DEVICE_ERR);
    EGX_HIP_TRY(hipMemcpyWithStream(soff_h.data(), soff.p, soff_h.size() * 4, hipMemcpyDeviceToHost, s), EGX_DEVICE_ERR);
    const int64_t slots = soff_h[(size_t)runs];
    if (slots > INT32_MAX) {
        set_last_error("propagation-blocked layout: too many slots");
        return EGX_UNSUPPORTED_GRAPH;
    }
    const int64_t groups = slots / kPbVec;

    // source slots (padding: the zero LDS entry kPbChunk) and their rows
    // (padding: -1)
    DevBuf srow;
    EGX_TRY(bad.alloc(4));
    EGX_TRY(g.pb_src.alloc((size_t)slots * 2));
    EGX_TRY(srow.alloc((size_t)slots * 4));
    EGX_HIP_TRY(hipMemsetAsync(bad.p, 0, 4, s), EGX_DEVICE_ERR);
    EGX_HIP_TRY(hipMemsetAsync(srow.p, 0xFF, (size_t)slots * 4, s), EGX_DEVICE_ERR);
    if (g.has_values()) {
        EGX_TRY(g.pb_arc.alloc((size_t)slots * 4));
        EGX_HIP_TRY(hipMemsetAsync(g.pb_arc.p, 0xFF, (size_t)slots * 4, s), EGX_DEVICE_ERR);
    }
    k_fill_u16<<<nblocks(slots, tb), tb, 0, s>>>(g.pb_src.as<uint16_t>(), slots, (uint16_t)kPbChunk);
    EGX_CHECK_LAUNCH(EGX_DEVICE_ERR);
    k_pb_place<<<nblocks(m, tb), tb, 0, s>>>(keys.as<uint32_t>(), vals.as<uint32_t>(), lb.as<int32_t>(),
                                             soff.as<uint32_t>(), g.it_col, rowof.as<int32_t>(), m, runs, B,
                                             g.pb_src.as<uint16_t>(), srow.as<int32_t>(),
                                             g.has_values() ? g.pb_arc.as<int32_t>() : nullptr, bad.as<int32_t>());
    EGX_CHECK_LAUNCH(EGX_DEVICE_ERR);
    if (g.has_values()) {
        EGX_TRY(g.pb_w.alloc((size_t)slots * 4));
        k_pb_gather_w<<<nblocks(slots, tb), tb, 0, s>>>(g.pb_arc.as<int32_t>(), g.it_val, slots, m,
                                                        g.pb_w.as<float>());
        EGX_CHECK_LAUNCH(EGX_DEVICE_ERR);
    }
    EGX_HIP_TRY(hipStreamSynchronize(s), EGX_DEVICE_ERR);
    keys.release();
    vals.release();
    rowof.release();
    lb.release();

    // stretch masks; value slots per group, per run (bin-major), per group
    DevBuf gs, voff;
    EGX_TRY(g.pb_mask.alloc((size_t)groups));
    EGX_TRY(gs.alloc((size_t)(groups + 1) * 4));
    // merged stretches for the weighted kernels (the solve's weight choice)
    const bool merge = g.has_values();
    k_pb_masks<<<nblocks(groups + 1, tb), tb, 0, s>>>(srow.as<int32_t>(), groups, soff.as<uint32_t>(), S, B, merge,
                                                      g.pb_mask.as<uint8_t>(), gs.as<uint32_t>());
    EGX_CHECK_LAUNCH(EGX_DEVICE_ERR);
    EGX_TRY(exclusive_scan_u32(gs.as<uint32_t>(), gs.as<uint32_t>(), groups + 1, s));
    EGX_TRY(voff.alloc((size_t)(runs + 1) * 4));
    k_pb_run_values<<<nblocks(runs + 1, tb), tb, 0, s>>>(soff.as<uint32_t>(), gs.as<uint32_t>(), runs, S, B,
                                                         voff.as<uint32_t>());
    EGX_CHECK_LAUNCH(EGX_DEVICE_ERR);
    EGX_TRY(exclusive_scan_u32(voff.as<uint32_t>(), voff.as<uint32_t>(), runs + 1, s));
    std::vector<uint32_t> voff_h((size_t)runs + 1);  // bin-major: sub-bin b, chunk c at b*S + c
    EGX_HIP_TRY(hipStreamSynchronize(s), EGX_DEVICE_ERR);
    EGX_HIP_TRY(hipMemcpyWithStream(voff_h.data(), voff.p, voff_h.size() * 4, hipMemcpyDeviceToHost, s), EGX_DEVICE_ERR);
    const int64_t nvals = voff_h[(size_t)runs];
    if (nvals > INT32_MAX) {
        set_last_error("propagation-blocked layout: too many value slots");
        return EGX_UNSUPPORTED_GRAPH;
    }
    EGX_TRY(g.pb_vgrp.alloc((size_t)groups * 4));
    EGX_TRY(g.pb_dst.alloc((size_t)nvals * 2));
    EGX_TRY(g.pb_vals.alloc((size_t)nvals * 4));
    // padding value slots are never written: rows 0, values 0
    EGX_HIP_TRY(hipMemsetAsync(g.pb_dst.p, 0, (size_t)nvals * 2, s), EGX_DEVICE_ERR);
    EGX_HIP_TRY(hipMemsetAsync(g.pb_vals.p, 0, (size_t)nvals * 4, s), EGX_DEVICE_ERR);
    k_pb_groups<<<nblocks(groups, tb), tb, 0, s>>>(soff.as<uint32_t>(), gs.as<uint32_t>(), voff.as<uint32_t>(),
                                                   g.pb_mask.as<uint8_t>(), srow.as<int32_t>(), groups, runs, S, B,
                                                   g.pb_vgrp.as<int32_t>(), g.pb_dst.as<uint16_t>(),
                                                   bad.as<int32_t>());
    EGX_CHECK_LAUNCH(EGX_DEVICE_ERR);
    int32_t bad_h = 0;
    EGX_HIP_TRY(hipStreamSynchronize(s), EGX_DEVICE_ERR);
    EGX_HIP_TRY(hipMemcpyWithStream(&bad_h, bad.p, 4, hipMemcpyDeviceToHost, s), EGX_DEVICE_ERR);

    // scatter work: contiguous group ranges of at most scat_groups groups per
    // chunk, whole windows: an item starts on its chunk's window grid
    auto chunk_groups = [&](int64_t c, int32_t& c0, int32_t& c1) {
        c0 = (int32_t)(soff_h[(size_t)(c * B)] / kPbVec);
        c1 = (int32_t)(soff_h[(size_t)((c + 1) * B)] / kPbVec);
    };
    auto scatter_slots = [&]() -> int64_t {
        if (cfg.blocked_shared) return kPbScatterShared;
        constexpr int64_t kStep = 4 * kPbWindow * kPbVec;
        const int64_t first = std::max<int64_t>(kPbScatterMin, (slots / kPbCus) / kStep * kStep);
        for (int64_t z = first; z <= kPbScatterMax1; z += kStep) {
            int64_t items = 0;
            for (int64_t c = 0; c < S; ++c) {
                int32_t c0, c1;
                chunk_groups(c, c0, c1);
                items += (c1 - c0 + z / kPbVec - 1) / (z / kPbVec);
            }
            if (items <= kPbCus) return z;
        }
        return g.weighted ? pb_item_slots(slots, kPbScatterItemsW, kPbScatterMin, kPbScatterItem)
                          : pb_item_slots(slots, kPbScatterItems, kPbScatterMax1, kPbScatterItem);
    };
    const int32_t scat_groups =
        std::max<int32_t>(kPbWindow, (int32_t)(scatter_slots() / kPbVec / kPbWindow * kPbWindow));
    const bool many_bins = B >= kPbSumBins;
    const int32_t sum_slots =
        (int32_t)(cfg.blocked_shared ? kPbSumShared
                                     : pb_item_slots(nvals, many_bins ? kPbSumItemsMany : kPbSumItems,
                                                     many_bins ? kPbSumMinMany : kPbSumMin, kPbItem));
    std::vector<PbScatter> scat;
    for (int64_t c = 0; c < S; ++c) {
        int32_t c0, c1;
        chunk_groups(c, c0, c1);
        for (int32_t q0 = c0; q0 < c1; q0 += scat_groups)
            scat.push_back(PbScatter{(int32_t)c, q0, (int32_t)std::min<int64_t>(c1, (int64_t)q0 + scat_groups), 0});
    }
    // sum work: a sub-bin per item, or pieces of at most sum_slots value slots
    // whose row sums go through hub_part (rows `pieces` apart) to the reduce
    std::vector<PbSum> sums;
    std::vector<HubRow> hrows;
    int64_t parts = 0;
    for (int64_t b = 0; b < B; ++b) {
        const int32_t e0 = (int32_t)voff_h[(size_t)(b * S)];  // chunk 0 of sub-bin b
        const int32_t e1 = (int32_t)voff_h[(size_t)((b + 1) * S)];
        const int32_t r0 = (int32_t)(b * kPbRows);
        const int32_t nr = std::min<int32_t>(kPbRows, n - r0);
        if (e1 - e0 <= sum_slots) {
            sums.push_back(PbSum{(int32_t)b, e0, e1, -1, 1, 0, 0, 0});
            continue;
        }
        const int32_t np = (e1 - e0 + sum_slots - 1) / sum_slots;
        if (parts + (int64_t)nr * np > INT32_MAX) {
            set_last_error("propagation-blocked layout: too many split rows");
            return EGX_UNSUPPORTED_GRAPH;
        }
        const int64_t vecs = (e1 - e0) / kPbVec;
        for (int32_t q = 0; q < np; ++q) {
            const int32_t a0 = e0 + (int32_t)((vecs * q) / np) * kPbVec;
            const int32_t a1 = e0 + (int32_t)((vecs * (q + 1)) / np) * kPbVec;
            sums.push_back(PbSum{(int32_t)b, a0, a1, q, np, (int32_t)parts, 0, 0});
        }
        for (int32_t i = 0; i < nr; ++i) hrows.push_back(HubRow{r0 + i, (int32_t)(parts + (int64_t)i * np), np, 0});
        parts += (int64_t)nr * np;
    }
    const int64_t many = many_first(hrows);
    // every range the kernels will touch, checked before any item upload
    // (the groups' value slots and rows were checked on the device)
    bool ok = bad_h == 0;
    for (const PbScatter& it : scat)
        ok = ok && it.chunk >= 0 && (int64_t)it.chunk * kPbChunk < n && it.g0 >= 0 && it.g0 < it.g1 &&
             it.g1 <= groups;
    for (const PbSum& it : sums) {
        ok = ok && it.sub_bin >= 0 && (int64_t)it.sub_bin * kPbRows < n && 0 <= it.e0 && it.e0 <= it.e1 &&
             (int64_t)it.e1 <= nvals && it.e0 % kPbVec == 0 && it.e1 % kPbVec == 0;
        if (ok && it.piece >= 0) {
            // the last row's slot of this piece: part0 + (nr - 1) * pieces + piece
            const int64_t nr = std::min<int64_t>(kPbRows, (int64_t)n - (int64_t)it.sub_bin * kPbRows);
            ok = it.piece < it.pieces && it.part0 >= 0 && (int64_t)it.part0 + (nr - 1) * it.pieces + it.piece < parts;
        }
    }
    for (const HubRow& h : hrows) ok = ok && h.row >= 0 && h.row < n && h.first >= 0 && (int64_t)h.first + h.nseg <= parts;
    if (!ok) {
        set_last_error("propagation-blocked layout failed its range check");
        return EGX_UNKNOW_ERROR;
    }
    EGX_TRY(g.pb_scatter.alloc(std::max<size_t>(scat.size(), 1) * sizeof(PbScatter)));
    EGX_TRY(g.pb_sum.alloc(std::max<size_t>(sums.size(), 1) * sizeof(PbSum)));
    EGX_TRY(g.pb_hrows.alloc(std::max<size_t>(hrows.size(), 1) * sizeof(HubRow)));
    EGX_TRY(g.pb_hub_part.alloc((size_t)std::max<int64_t>(parts, 1) * 8));
    if (!scat.empty())
        EGX_HIP_TRY(hipMemcpyWithStream(g.pb_scatter.p, scat.data(), scat.size() * sizeof(PbScatter), hipMemcpyHostToDevice, s),
                    EGX_DEVICE_ERR);
    EGX_HIP_TRY(hipMemcpyWithStream(g.pb_sum.p, sums.data(), sums.size() * sizeof(PbSum), hipMemcpyHostToDevice, s),
                EGX_DEVICE_ERR);
    if (!hrows.empty())
        EGX_HIP_TRY(hipMemcpyWithStream(g.pb_hrows.p, hrows.data(), hrows.size() * sizeof(HubRow), hipMemcpyHostToDevice, s),
                    EGX_DEVICE_ERR);
    g.n_pb_scatter = (int64_t)scat.size();
    g.n_pb_sum = (int64_t)sums.size();
    g.n_pb_hrows = (int64_t)hrows.size();
    g.n_pb_hrows_many = many;
    g.pb_scatter_size.resize(scat.size());
    g.pb_scatter_chunk.resize(scat.size());
    for (size_t i = 0; i < scat.size(); ++i) {
        g.pb_scatter_size[i] = scat[i].g1 - scat[i].g0;
        g.pb_scatter_chunk[i] = scat[i].chunk;
    }
    g.pb_sum_size.resize(sums.size());
    for (size_t i = 0; i < sums.size(); ++i) g.pb_sum_size[i] = sums[i].e1 - sums[i].e0;
    g.pb_shared = cfg.blocked_shared;
    g.pb_merged = merge;
    g.pb_ready = true;
    return EGX_SUCC;
}

// Items per tile: what the caller set, or (EGX_TILE_ITEMS_AUTO) a size for the
// graph.  Large tiles leave a small graph's device idle, small ones pay more
// for their barriers than for their arcs.  Measured (us per SpMV launch at
// tiles of 512 / 1024 / 2048 / 4096 / 5888 items, FP32): 244K items 10.4 /
// 10.8 / 13.6 / 17.6 / 18.9; 1M items 14.1 / 11.0 / 12.2 / 17.0 / 20.0; 4.5M 45.6 / 32.9
// / 28.5 / 35.7 / 37.1; 8M 82.9 / 55.7 / 42.5 / 38.2 / 43.5; 34M 345 / 243 / 184 / 160 / 172;
// FP64 alike (34M: 206 / 192 / 220 at 2048 / 4096 / 5888).  A graph of a few thousand
// items is cut into up to 64 tiles of at least 256 (7.5K items: 8.1 us at 256, 11.7 at 5888).
int32_t tile_size(const BinCfg& cfg, int64_t items) {
    if (cfg.tile_items != EGX_TILE_ITEMS_AUTO) return cfg.tile_items;
    const int64_t most = std::min(4096, kTileLds - cfg.wave_row_max);
    const int64_t fill = std::min(most, std::max<int64_t>(1024, items / 2048));
    return (int32_t)std::min(fill, std::max<int64_t>(256, items / 64));
}

int rebuild_bins(Graph& g, const BinCfg& cfg_in, const uint32_t* counters) {
    BinCfg cfg = cfg_in;
    if (cfg.thread_row_max < 0) cfg.thread_row_max = 0;
    cfg.wave_row_max = hub_threshold(cfg);
    if (cfg.tile_items != EGX_TILE_ITEMS_AUTO)
        cfg.tile_items = std::min(std::max(cfg.tile_items, 256), kTileLds - cfg.wave_row_max);
    cfg.hub_segment = hub_segment(cfg);
    if (cfg.reorder != 0) cfg.reorder = 1;
    if (cfg.tile_sort != 0) cfg.tile_sort = 1;
    if (cfg.blocked != 0) cfg.blocked = 1;
    const bool layout_changed =
        !g.layout_built || g.layout_hub != cfg.wave_row_max || g.layout_reorder != cfg.reorder;
    hipStream_t s = g.stream;
    const int32_t n = g.n;
    uint32_t hctr[kCtrWords] = {};
    if (counters) {
        std::copy(counters, counters + kCtrWords, hctr);
    } else if (n > 0) {
        DevBuf ctr;
        EGX_TRY(ctr.alloc(sizeof(hctr)));
        EGX_HIP_TRY(hipMemsetAsync(ctr.p, 0, sizeof(hctr), s), EGX_DEVICE_ERR);
        k_in_degrees<<<std::min<unsigned>(nblocks(n, 256), kNodeBlocks), 256, 0, s>>>(
            g.in_row.as<int32_t>(), n, cfg.wave_row_max, cfg.hub_segment, ctr.as<uint32_t>());
        EGX_CHECK_LAUNCH(EGX_DEVICE_ERR);
        EGX_HIP_TRY(hipMemcpyWithStream(hctr, ctr.p, sizeof(hctr), hipMemcpyDeviceToHost, s), EGX_DEVICE_ERR);
    }
    if (layout_changed) EGX_TRY(build_layout(g, cfg, (int32_t)hctr[kCtrHubs]));
    g.bins = cfg;
    g.n_hseg = g.n_hrows = g.n_hrows_split = g.n_hrows_many = g.n_tiles = 0;
    g.rows_thread = g.rows_wave = 0;
    if (n <= 0) return EGX_SUCC;

    // hub rows [0, n_hub): fixed-size segments; a row of one segment is
    // finished by its workgroup
    g.n_hrows = g.n_hub;
    g.n_hrows_split = hctr[kCtrHubSplit];
    g.n_hrows_many = hctr[kCtrHubMany];
    g.n_hseg = hctr[kCtrHubSegs];
    EGX_TRY(g.hsegs.alloc(std::max<size_t>((size_t)g.n_hseg, 1) * sizeof(HubSeg)));
    EGX_TRY(g.hrows.alloc(std::max<size_t>((size_t)g.n_hrows_split, 1) * sizeof(HubRow)));
    EGX_TRY(g.hub_part.alloc(std::max<size_t>((size_t)g.n_hseg, 1) * 8));
    DevBuf first_seg;
    if (g.n_hub > 0) {
        EGX_TRY(first_seg.alloc(((size_t)g.n_hub + 1) * 4));
        k_hub_rows<<<1, kHubThreads, 0, s>>>(g.it_row, g.n_hub, cfg.hub_segment, (int32_t)g.n_hrows_many,
                                             first_seg.as<int32_t>(), g.hrows.as<HubRow>());
        EGX_CHECK_LAUNCH(EGX_DEVICE_ERR);
        k_hub_segs<<<nblocks(g.n_hseg, 256), 256, 0, s>>>(g.it_row, first_seg.as<int32_t>(), g.n_hub, cfg.hub_segment,
                                                          (int32_t)g.n_hseg, g.hsegs.as<HubSeg>());
        EGX_CHECK_LAUNCH(EGX_DEVICE_ERR);
    }

    // merge-path tiles over rows [n_hub, n)
    const int64_t items = (g.m - (int64_t)hctr[kCtrHubArcs]) + (int64_t)(n - g.n_hub);
    const int32_t per_tile = tile_size(cfg, items);
    g.tile_items = per_tile;
    g.n_tiles = (items + per_tile - 1) / per_tile;
    g.tile_lds = per_tile + cfg.wave_row_max;
    DevBuf wave_rows;
    EGX_TRY(wave_rows.alloc(sizeof(uint32_t)));
    EGX_TRY(g.tiles.alloc(((size_t)g.n_tiles + 1) * 4));
    k_tile_starts<<<nblocks(g.n_tiles + 1, 256), 256, 0, s>>>(g.it_row, g.n_hub, n, per_tile, g.n_tiles,
                                                               g.tiles.as<int32_t>(), wave_rows.as<uint32_t>());
    EGX_CHECK_LAUNCH(EGX_DEVICE_ERR);
    k_row_stats<<<std::min<unsigned>(nblocks(n, 256), kNodeBlocks), 256, 0, s>>>(
        g.it_row, g.n_hub, n, row_lane_max(cfg), wave_rows.as<uint32_t>());
    EGX_CHECK_LAUNCH(EGX_DEVICE_ERR);
    int rc = build_tile_sort(g, cfg);
    if (rc == EGX_SUCC) {
        rc = build_blocked(g, cfg, layout_changed);
        if (rc != EGX_SUCC) g.bins.blocked = 0;  // the pull layout stays usable
    }
    // the one wait, after all that can be queued without it
    uint32_t rows_wave = 0;
    EGX_HIP_TRY(hipMemcpyWithStream(&rows_wave, wave_rows.p, 4, hipMemcpyDeviceToHost, s), EGX_DEVICE_ERR);
    g.rows_wave = rows_wave;
    g.rows_thread = (int64_t)(n - g.n_hub) - g.rows_wave;
    if (layout_changed) {
        float ms = 0.0f;
        EGX_HIP_TRY(hipEventElapsedTime(&ms, g.ev0, g.ev1), EGX_DEVICE_ERR);
        g.layout_seconds = (double)ms * 1e-3;
    }
    return rc;
}

int check_arcs(const int32_t* dE, const double* dW, int32_t n, int64_t m, uint32_t* flags, hipStream_t s) {
    EGX_HIP_TRY(hipMemsetAsync(flags, 0, sizeof(uint32_t), s), EGX_DEVICE_ERR);
    if (m <= 0) return EGX_SUCC;
    const unsigned blocks = (unsigned)std::min<int64_t>((m + 255) / 256, 4096);
    k_check_arcs<<<blocks, 256, 0, s>>>(dE, dW, n, m, flags);
    EGX_CHECK_LAUNCH(EGX_DEVICE_ERR);
    return EGX_SUCC;
}

// out_w[u] = 1: adjacency values keep alpha * w undivided.
__global__ void k_unit_out_w(double* __restrict__ out_w, int32_t n) {
    const int32_t u = blockIdx.x * blockDim.x + threadIdx.x;
    if (u < n) out_w[u] = 1.0;
}

int build_from_device_csr(Graph& g, const int32_t* dV, const int32_t* dE, const double* dW, int32_t n, int64_t m,
                          double alpha) {
    hipStream_t s = g.stream;
    g.n = n;
    g.weighted = dW != nullptr || g.adjacency;
    g.adjacency_weights = g.adjacency && dW != nullptr;
    g.alpha_vals = alpha;
    g.alpha_orig = alpha;
    const auto t_start = std::chrono::steady_clock::now();
    const bool values = g.has_values();
    const size_t mm = (size_t)std::max<int64_t>(m, 1);
    const size_t nn = (size_t)std::max(n, 1);

    // The sizes that the host needs (valid arcs, hub rows, the largest
    // out-degree) come back in one copy, after everything that does not
    // depend on them has been queued.
    DevBuf ctr_buf, long_rows, keys, keys_alt, vals, vals_alt, rec;
    EGX_TRY(ctr_buf.alloc(kCtrWords * sizeof(uint32_t)));
    uint32_t* ctr = ctr_buf.as<uint32_t>();
    EGX_HIP_TRY(hipMemsetAsync(ctr, 0, kCtrWords * sizeof(uint32_t), s), EGX_DEVICE_ERR);
    EGX_TRY(g.out_w.alloc(nn * 8));
    EGX_TRY(g.deg.alloc(nn * 4));
    EGX_TRY(g.out_cnt.alloc(nn * 4));
    EGX_TRY(g.in_row.alloc(((size_t)n + 1) * 4));
    int32_t* outcnt_p = g.out_cnt.as<int32_t>();
    double* out_w = g.out_w.as<double>();
    EGX_TRY(keys.alloc(mm * 4));
    EGX_TRY(keys_alt.alloc(mm * 4));
    EGX_TRY(vals.alloc((mm + kArcPad) * 4));
    EGX_TRY(vals_alt.alloc((mm + kArcPad) * 4));
    if (values) EGX_TRY(rec.alloc(mm * sizeof(ArcRec)));

    // Out-weights, counts and what follows from them: by the arcs themselves
    // (weights that count, or endpoints to skip), or by the offsets.
    const bool sum_weights = dW && !g.adjacency;  // out-weights of adjacency graphs are 1
    const unsigned node_blocks = std::min<unsigned>(nblocks(n, 256), kNodeBlocks);
    auto out_by_arcs = [&]() -> int {
        // at most m / kOutLong rows are longer than kOutLong
        const int64_t max_long = m / kOutLong;
        EGX_TRY(long_rows.alloc((size_t)std::max<int64_t>(max_long, 1) * 4));
        int32_t* lr = long_rows.as<int32_t>();
        uint32_t* nl = ctr + kCtrLong;
        const unsigned lb = (unsigned)std::min<int64_t>(max_long, kLongBlocks);
        if (lb > 0) {
            k_long_rows<<<nblocks(n, 256), 256, 0, s>>>(dV, n, lr, nl);
            EGX_CHECK_LAUNCH(EGX_DEVICE_ERR);
        }
        const unsigned tiles = nblocks(m + n, kOutTile);
        if (sum_weights)
            k_row_out<true><<<lb + tiles, kOutThreads, 0, s>>>(dV, dE, dW, n, out_w, outcnt_p, lr, nl, lb);
        else
            k_row_out<false><<<lb + tiles, kOutThreads, 0, s>>>(dV, dE, nullptr, n, out_w, outcnt_p, lr, nl, lb);
        EGX_CHECK_LAUNCH(EGX_DEVICE_ERR);
        if (g.adjacency) {
            k_unit_out_w<<<nblocks(n, 256), 256, 0, s>>>(out_w, n);
            EGX_CHECK_LAUNCH(EGX_DEVICE_ERR);
        }
        k_node_arrays<false><<<node_blocks, 256, 0, s>>>(dV, out_w, outcnt_p, n, 0, g.weighted ? 1 : 0,
                                                         g.deg.as<float>(), ctr);
        EGX_CHECK_LAUNCH(EGX_DEVICE_ERR);
        return EGX_SUCC;
    };
    if (n > 0) {
        if (sum_weights) {
            EGX_TRY(out_by_arcs());
        } else {
            k_node_arrays<true><<<node_blocks, 256, 0, s>>>(dV, out_w, outcnt_p, n, g.adjacency ? 1 : 0,
                                                            g.weighted ? 1 : 0, g.deg.as<float>(), ctr);
            EGX_CHECK_LAUNCH(EGX_DEVICE_ERR);
        }
    }
    if (m > 0) {
        const unsigned rb = nblocks(m, kRunArcs);
        if (values)
            k_arc_keys<true><<<rb, kRunThreads, 0, s>>>(dV, dE, dW, out_w, n, m, alpha, keys.as<uint32_t>(),
                                                        vals.as<uint32_t>(), rec.as<ArcRec>(), ctr + kCtrInvalid);
        else
            k_arc_keys<false><<<rb, kRunThreads, 0, s>>>(dV, dE, nullptr, nullptr, n, m, alpha, keys.as<uint32_t>(),
                                                         vals.as<uint32_t>(), nullptr, ctr + kCtrInvalid);
        EGX_CHECK_LAUNCH(EGX_DEVICE_ERR);
    }
    // stable sort of (dst-or-sentinel, slot-or-src) on the bits that can hold n
    EGX_TRY(radix_sort_u32(keys, keys_alt, &vals, &vals_alt, m, bits_for((uint64_t)n), s));
    EGX_TRY(lower_bound_iota_u32(keys.as<uint32_t>(), m, g.in_row.as<int32_t>(), (int64_t)n + 1, s));
    if (n > 0) {
        k_in_degrees<<<node_blocks, 256, 0, s>>>(g.in_row.as<int32_t>(), n, hub_threshold(g.bins),
                                             hub_segment(g.bins), ctr);
        EGX_CHECK_LAUNCH(EGX_DEVICE_ERR);
    }
    uint32_t hctr[kCtrWords];
    EGX_HIP_TRY(hipMemcpyWithStream(hctr, ctr, sizeof(hctr), hipMemcpyDeviceToHost, s), EGX_DEVICE_ERR);
    if (hctr[kCtrInvalid] > 0 && !sum_weights && n > 0) {
        // skipped endpoints: the offsets counted them
        EGX_HIP_TRY(hipMemsetAsync(ctr, 0, kCtrWords * sizeof(uint32_t), s), EGX_DEVICE_ERR);
        EGX_TRY(out_by_arcs());
        uint32_t again[kCtrWords];
        EGX_HIP_TRY(hipMemcpyWithStream(again, ctr, sizeof(again), hipMemcpyDeviceToHost, s), EGX_DEVICE_ERR);
        hctr[kCtrDangling] = again[kCtrDangling];
        hctr[kCtrMaxOut] = again[kCtrMaxOut];
    }
    const int64_t m_valid = m - (int64_t)hctr[kCtrInvalid];
    g.m = m_valid;
    g.n_dangling = hctr[kCtrDangling];
    g.max_out_degree = (int32_t)hctr[kCtrMaxOut];
    g.max_in_degree = (int32_t)hctr[kCtrMaxIn];
    keys.release();
    keys_alt.release();
    vals_alt.release();

    if (values) {
        const size_t mv = (size_t)std::max<int64_t>(m_valid, 1);
        EGX_TRY(g.in_col.alloc((mv + kArcPad) * 4));
        EGX_TRY(g.in_val.alloc(mv * 4));
        EGX_TRY(g.w_csc.alloc(mv * 8));
        if (m_valid > 0) {
            k_fill_csc<<<nblocks(m_valid, 256), 256, 0, s>>>(vals.as<uint32_t>(), rec.as<ArcRec>(), m_valid,
                                                              g.in_col.as<int32_t>(), g.in_val.as<float>(),
                                                              g.w_csc.as<double>());
            EGX_CHECK_LAUNCH(EGX_DEVICE_ERR);
        }
        vals.release();
        rec.release();
    } else {
        g.in_col = std::move(vals);  // the sorted sources
        g.in_val.release();
        g.w_csc.release();
    }
    if (n <= 0) EGX_HIP_TRY(hipMemsetAsync(g.in_col.p, 0, kArcPad * 4, s), EGX_DEVICE_ERR);  // else the layout's
    g.layout_built = false;
    EGX_TRY(rebuild_bins(g, g.bins, hctr));
    // large PageRank graphs iterate propagation-blocked; one the layout
    // cannot hold keeps the pull layout alone
    if (!g.adjacency && m >= kPbDefaultArcs && !g.bins.blocked) {
        BinCfg cfg = g.bins;
        cfg.blocked = 1;
        if (build_blocked(g, cfg, true) == EGX_SUCC) {
            g.bins.blocked = 1;
        } else {
            cfg.blocked = 0;
            EGX_TRY(build_blocked(g, cfg, true));  // releases what the attempt allocated
        }
    }
    EGX_HIP_TRY(hipStreamSynchronize(s), EGX_DEVICE_ERR);
    pool_stream_idle(s);
    g.build_seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t_start).count();
    return EGX_SUCC;
}

int build_from_device_rows(Graph& g, DevBuf&& V, DevBuf&& E, int32_t n, int64_t m, double alpha, bool* bad_endpoint) {
    hipStream_t s = g.stream;
    g.n = n;
    g.m = m;
    g.weighted = true;
    g.adjacency_weights = false;
    g.alpha_vals = alpha;
    g.alpha_orig = alpha;
    const auto t_start = std::chrono::steady_clock::now();
    g.in_row = std::move(V);
    g.in_col = std::move(E);
    g.in_val.release();
    g.w_csc.release();
    DevBuf ctr_buf, keys, keys_alt, offsets;
    EGX_TRY(ctr_buf.alloc(kCtrWords * sizeof(uint32_t)));
    uint32_t* ctr = ctr_buf.as<uint32_t>();
    EGX_HIP_TRY(hipMemsetAsync(ctr, 0, kCtrWords * sizeof(uint32_t), s), EGX_DEVICE_ERR);
    EGX_TRY(g.out_w.alloc((size_t)n * 8));
    EGX_TRY(g.deg.alloc((size_t)n * 4));
    EGX_TRY(g.out_cnt.alloc((size_t)n * 4));
    EGX_TRY(keys.alloc((size_t)m * 4));
    EGX_TRY(keys_alt.alloc((size_t)m * 4));
    EGX_TRY(offsets.alloc(((size_t)n + 1) * 4));
    k_check_arcs<<<(unsigned)std::min<int64_t>((m + 255) / 256, 4096), 256, 0, s>>>(g.in_col.as<int32_t>(), nullptr, n,
                                                                                  m, ctr + kCtrInvalid);
    EGX_CHECK_LAUNCH(EGX_DEVICE_ERR);
    // how often each node is a source: by a sort of the sources alone (one
    // counter per node would take a device-wide atomic per arc)
    EGX_HIP_TRY(hipMemcpyAsync(keys.p, g.in_col.p, (size_t)m * 4, hipMemcpyDeviceToDevice, s), EGX_DEVICE_ERR);
    EGX_TRY(radix_sort_u32(keys, keys_alt, nullptr, nullptr, m, bits_for((uint64_t)(n - 1)), s));
    EGX_TRY(lower_bound_iota_u32(keys.as<uint32_t>(), m, offsets.as<int32_t>(), (int64_t)n + 1, s));
    const unsigned node_blocks = std::min<unsigned>(nblocks(n, 256), kNodeBlocks);
    k_node_arrays<true><<<node_blocks, 256, 0, s>>>(offsets.as<int32_t>(), g.out_w.as<double>(),
                                                    g.out_cnt.as<int32_t>(), n, 1, 1, g.deg.as<float>(), ctr);
    EGX_CHECK_LAUNCH(EGX_DEVICE_ERR);
    k_in_degrees<<<node_blocks, 256, 0, s>>>(g.in_row.as<int32_t>(), n, hub_threshold(g.bins),
                                             hub_segment(g.bins), ctr);
    EGX_CHECK_LAUNCH(EGX_DEVICE_ERR);
    uint32_t hctr[kCtrWords];
    EGX_HIP_TRY(hipMemcpyWithStream(hctr, ctr, sizeof(hctr), hipMemcpyDeviceToHost, s), EGX_DEVICE_ERR);
    *bad_endpoint = hctr[kCtrInvalid] != 0;
    if (*bad_endpoint) return EGX_SUCC;  // the caller's to report; nothing else was built
    g.n_dangling = hctr[kCtrDangling];
    g.max_out_degree = (int32_t)hctr[kCtrMaxOut];
    g.max_in_degree = (int32_t)hctr[kCtrMaxIn];
    keys.release();
    keys_alt.release();
    offsets.release();
    g.layout_built = false;
    EGX_TRY(rebuild_bins(g, g.bins, hctr));
    EGX_HIP_TRY(hipStreamSynchronize(s), EGX_DEVICE_ERR);
    pool_stream_idle(s);
    g.build_seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t_start).count();
    return EGX_SUCC;
}

int build_layout(Graph& g, const BinCfg& cfg, int32_t hubs) {
    hipStream_t s = g.stream;
    const int32_t n = g.n;
    const int64_t m = g.m;
    g.p_row.release();
    g.p_col.release();
    g.p_val.release();
    g.p_w.release();
    g.p_outw.release();
    g.p_deg.release();
    g.p_nval.release();
    g.perm.release();
    g.rank.release();
    g.reordered = false;
    g.layout_built = false;
    g.n_hub = 0;
    g.it_row = g.in_row.as<int32_t>();
    g.it_col = g.in_col.as<int32_t>();
    g.it_val = g.in_val.as<float>();
    g.it_w = g.w_csc.as<double>();
    g.it_outw = g.out_w.as<double>();
    g.it_deg = g.deg.as<float>();
    g.alpha_vals = g.alpha_orig;
    g.layout_seconds = 0.0;
    if (n <= 0) {
        g.layout_built = true;
        g.layout_hub = cfg.wave_row_max;
        g.layout_reorder = cfg.reorder;
        return EGX_SUCC;
    }

    EGX_HIP_TRY(hipEventRecord(g.ev0, s), EGX_DEVICE_ERR);
    const uint32_t maxdeg = (uint32_t)g.max_out_degree;
    const int bits = cfg.reorder ? bits_for(maxdeg) : 0;
    DevBuf keys, keys_alt, vals_alt, cnt;
    EGX_TRY(keys.alloc((size_t)n * 4));
    EGX_TRY(keys_alt.alloc((size_t)n * 4));
    EGX_TRY(g.perm.alloc((size_t)n * 4));
    EGX_TRY(vals_alt.alloc((size_t)n * 4));
    k_layout_keys<<<nblocks(n, 256), 256, 0, s>>>(g.in_row.as<int32_t>(), g.out_cnt.as<int32_t>(), n,
                                                   cfg.wave_row_max, bits, maxdeg, cfg.reorder,
                                                   keys.as<uint32_t>(), g.perm.as<uint32_t>(),
                                                   g.in_col.as<int32_t>() + m);
    EGX_CHECK_LAUNCH(EGX_DEVICE_ERR);
    EGX_TRY(radix_sort_u32(keys, keys_alt, &g.perm, &vals_alt, n, bits + 1, s));
    keys.release();
    keys_alt.release();
    vals_alt.release();

    EGX_TRY(g.rank.alloc((size_t)n * 4));
    EGX_TRY(cnt.alloc(((size_t)n + 1) * 4));
    EGX_TRY(g.p_col.alloc(((size_t)std::max<int64_t>(m, 1) + kArcPad) * 4));
    EGX_TRY(g.p_deg.alloc((size_t)n * 4));
    EGX_TRY(g.p_outw.alloc((size_t)n * 8));
    EGX_TRY(g.p_row.alloc(((size_t)n + 1) * 4));
    k_layout_nodes<<<nblocks(n, 256), 256, 0, s>>>(g.perm.as<uint32_t>(), g.in_row.as<int32_t>(), g.deg.as<float>(),
                                                    g.out_w.as<double>(), n, g.rank.as<int32_t>(),
                                                    cnt.as<uint32_t>(), g.p_deg.as<float>(), g.p_outw.as<double>(),
                                                    g.p_col.as<int32_t>() + m);
    EGX_CHECK_LAUNCH(EGX_DEVICE_ERR);
    EGX_TRY(exclusive_scan_u32(cnt.as<uint32_t>(), g.p_row.as<uint32_t>(), (int64_t)n + 1, s));
    cnt.release();
    if (g.has_values()) {
        EGX_TRY(g.p_val.alloc((size_t)std::max<int64_t>(m, 1) * 4));
        EGX_TRY(g.p_w.alloc((size_t)std::max<int64_t>(m, 1) * 8));
    }
    if (m > 0) {
        k_layout_slots<<<nblocks(m, kRunArcs), kRunThreads, 0, s>>>(g.p_row.as<int32_t>(), g.perm.as<int32_t>(),
                                                        g.rank.as<int32_t>(), g.in_row.as<int32_t>(),
                                                        g.in_col.as<int32_t>(), g.in_val.as<float>(),
                                                        g.w_csc.as<double>(), n, m, g.has_values() ? 1 : 0,
                                                        g.p_col.as<int32_t>(), g.p_val.as<float>(),
                                                        g.p_w.as<double>());
        EGX_CHECK_LAUNCH(EGX_DEVICE_ERR);
    }
    g.reordered = true;
    g.n_hub = hubs;
    g.it_row = g.p_row.as<int32_t>();
    g.it_col = g.p_col.as<int32_t>();
    g.it_val = g.p_val.as<float>();
    g.it_w = g.p_w.as<double>();
    g.it_outw = g.p_outw.as<double>();
    g.it_deg = g.p_deg.as<float>();
    EGX_HIP_TRY(hipEventRecord(g.ev1, s), EGX_DEVICE_ERR);
    g.layout_built = true;
    g.layout_hub = cfg.wave_row_max;
    g.layout_reorder = cfg.reorder;
    return EGX_SUCC;
}

int refresh_alpha(Graph& g, double alpha) {
    if (!g.has_values() || alpha == g.alpha_vals) {
        if (!g.has_values()) g.alpha_vals = alpha;
        return EGX_SUCC;
    }
    if (g.m > 0) {
        k_refresh_vals<<<nblocks(g.m, 256), 256, 0, g.stream>>>(g.it_col, g.it_w, g.it_outw, g.m, alpha, g.it_val);
        EGX_CHECK_LAUNCH(EGX_DEVICE_ERR);
        if (g.tsorted && g.n_tiles > 0) {
            k_tile_vals<<<(unsigned)g.n_tiles, 256, 0, g.stream>>>(g.it_row, g.tiles.as<int32_t>(),
                                                                   g.t_pos.as<uint16_t>(), g.it_val,
                                                                   g.t_val.as<float>());
            EGX_CHECK_LAUNCH(EGX_DEVICE_ERR);
        }
        if (g.pb_ready && g.pb_w.p) {
            const int64_t slots = (int64_t)(g.pb_w.bytes / 4);
            k_pb_gather_w<<<nblocks(slots, 256), 256, 0, g.stream>>>(g.pb_arc.as<int32_t>(), g.it_val, slots, g.m,
                                                                     g.pb_w.as<float>());
            EGX_CHECK_LAUNCH(EGX_DEVICE_ERR);
        }
    }
    g.alpha_vals = alpha;
    if (!g.reordered) g.alpha_orig = alpha;  // in_val is the iteration array
    return EGX_SUCC;
}

int download_csc(Graph& g, int32_t* in_row, int32_t* in_col, float* in_val, int32_t* dangling01) {
    hipStream_t s = g.stream;
    EGX_HIP_TRY(hipStreamSynchronize(s), EGX_DEVICE_ERR);
    if (in_row)
        EGX_HIP_TRY(hipMemcpyWithStream(in_row, g.in_row.p, ((size_t)g.n + 1) * 4, hipMemcpyDeviceToHost, s), EGX_DEVICE_ERR);
    if (in_col && g.m > 0)
        EGX_HIP_TRY(hipMemcpyWithStream(in_col, g.in_col.p, (size_t)g.m * 4, hipMemcpyDeviceToHost, s), EGX_DEVICE_ERR);
    if (in_val && g.m > 0) {
        // values for the alpha of the last build or solve
        if (g.weighted && g.alpha_orig == g.alpha_vals) {
            EGX_HIP_TRY(hipMemcpyWithStream(in_val, g.in_val.p, (size_t)g.m * 4, hipMemcpyDeviceToHost, s), EGX_DEVICE_ERR);
        } else {
            DevBuf tmp;
            EGX_TRY(tmp.alloc((size_t)g.m * 4));
            if (g.weighted)
                k_refresh_vals<<<nblocks(g.m, 256), 256, 0, s>>>(g.in_col.as<int32_t>(), g.w_csc.as<double>(),
                                                                  g.out_w.as<double>(), g.m, g.alpha_vals,
                                                                  tmp.as<float>());
            else
                k_unit_vals<<<nblocks(g.m, 256), 256, 0, s>>>(g.in_col.as<int32_t>(), g.out_w.as<double>(), g.m,
                                                               g.alpha_vals, tmp.as<float>());
            EGX_CHECK_LAUNCH(EGX_DEVICE_ERR);
            EGX_HIP_TRY(hipStreamSynchronize(s), EGX_DEVICE_ERR);
            EGX_HIP_TRY(hipMemcpyWithStream(in_val, tmp.p, (size_t)g.m * 4, hipMemcpyDeviceToHost, s), EGX_DEVICE_ERR);
        }
    }
    if (dangling01 && g.n > 0) {
        std::vector<float> d((size_t)g.n);
        EGX_HIP_TRY(hipMemcpyWithStream(d.data(), g.deg.p, (size_t)g.n * 4, hipMemcpyDeviceToHost, s), EGX_DEVICE_ERR);
        for (int32_t i = 0; i < g.n; ++i) dangling01[i] = (d[(size_t)i] == 0.0f) ? 1 : 0;
    }
    return EGX_SUCC;
}

}  // namespace egx
