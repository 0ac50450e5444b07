// knn_rows.hip -- the kNN scans that run on the vector ALUs, a base row a lane: the metrics that are no
// matrix product, squared L2 in direct form (the fallback of the certified GEMM-form search), and
// popcount Hamming of small batches.
//
// Replaces the metric switch of knn_compute_distance_matrix (vector-cuda/src/kernels/knn.cu:84-141,
// 175-195): L1, Minkowski p = 3, L-inf, thresholded Hamming, Mahalanobis (sqrt of direct L2), weighted
// Jaccard and Hellinger (direct L2 of sqrt|x|, then sqrt(0.5 * sum)), fused with the threshold filter
// of the round/merge top-k (topk.hip).
//
// Bound: the vector ALUs, or for few queries the stream of base rows.  A lane owns a base row and the
// queries are wave-uniform: their values come through the scalar cache into SGPRs, which a VALU
// instruction takes as an operand, so an element costs its two operations per query and no LDS read
// (the earlier kernel held 256 queries in a workgroup's registers and broadcast base rows from LDS: a
// batch of a few queries paid for 256, and the LDS return path set the rate of Jaccard's two sums).
// A row is read once per tile of 16 queries.
//
// Whole searches, microseconds, k = 10, queries and results on the device (earlier kernel -> this one):
//   queries                   1           16           128           256            700           4096
//   L1        500k x 128   973 -> 88    990 -> 119   1035 -> 371   1083 -> 746   2486 -> 1869   10863 -> 10268
//   L-inf     500k x 128   961 -> 87    991 -> 116   1028 -> 373   1086 -> 745   2421 -> 1896   10981 -> 10430
//   Minkowski 500k x 128  1402 -> 88   1427 -> 131   1461 -> 526   1522 -> 1044  3571 -> 2661   16580 -> 14827
//   Jaccard   500k x 128  6288 -> 95   6323 -> 171   6348 -> 824   6421 -> 1666 17199 -> 4446   83997 -> 25175
// The marginal cost of 16 queries at 500k x 128 is 42 us under L1: 2.05e9 two-operation elements at 49 T
// operations a second, of 57.5 that independent non-packed adds reach on this card.
#include <algorithm>

#include "valu_metrics.h"
#include "vh_common.h"

namespace vh {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(4))) const float cfloat;        // read through the scalar cache
typedef __attribute__((address_space(4))) const floatx16 cfloatx16;
typedef __attribute__((address_space(4))) const uint32_t cuint32;

constexpr int kScanQueries = 16;   // queries of a tile
constexpr int kScanFew = 4;        // in a round of few workgroups (its rows spread over more of them)
constexpr long kScanFewWgs = 512;  // fewer workgroups of 16-query tiles than this (two a CU): 4-query tiles
constexpr long kScanMaxWgs = 1L << 22;  // workgroups of a launch (a dispatch counts its threads in 32 bits)
// Queries that an XCD's row groups take in turn before the next ones: half of its 4 MB L2, the row groups
// in flight have the rest.  Whole searches, k = 10, without this limit -> 3, 2, 1 and 0.5 MB:
//   L1      300,000 x 128, 10,000 queries (5.1 MB)   22.0 ms -> 15.5, 15.3, 15.4, 15.5
//   L1      60,000 x 300,  4,000 queries (5.1 MB)     3.97   ->  3.19, 3.05, 3.08, 3.14;  1,000 queries 0.85 -> 0.84, 0.84, 0.88, 0.90
//   L1      20,000 x 1,000, 4,000 queries (16 MB)     4.00   ->  3.89, 3.83, 3.81, 3.81
//   Jaccard 300,000 x 128, 10,000 queries            42.7    -> 37.3, 37.2, 37.2, 37.2
constexpr long kScanQueryBytes = 2L << 20;
constexpr int kScanSlots = 16;     // LDS candidate slots per query and workgroup
constexpr int kScanWg = 256;       // rows per workgroup: 4 waves of 64 rows, one a lane

struct RowScanArgs {
    const void *base;     // rows of dpad floats, or of dpad code words
    const void *qry;      // queries in the same layout, zero rows up to a multiple of 128
    const float *shift;   // added to every base value as it is read, or null
    int dim, dpad, nq;
    long row_begin, row_end;
    const float *tau;     // FILTER: per-query thresholds
    uint2 *cand;
    uint32_t *cnt;        // FILTER: per-query candidate counters, cnt_stride words apart
    int cnt_stride, cap;
    long cand_row0;       // DENSE: row r goes to slot r - cand_row0
    int n_groups, n_qtiles, spread, chunk;  // row groups, query tiles, and how workgroups map to them
};

// (row group, query tile) of a workgroup.  spread: an XCD (workgroups b mod 8) takes every eighth row
// group; it runs `chunk` query tiles (the last chunk what is left) of its first group one after another,
// then of its next, and so through all its groups before the next chunk, so the group's rows and the
// chunk's queries stay in its L2.
__device__ __forceinline__ bool scan_tile(const RowScanArgs &a, int &group, int &qt) {
    const unsigned b = blockIdx.x;
    if (a.spread) {
        const unsigned seq = b >> 3, per_xcd = (unsigned)(a.n_groups + 7) / 8u;  // row groups of an XCD
        const unsigned first =
            a.chunk < a.n_qtiles ? seq / (per_xcd * (unsigned)a.chunk) * (unsigned)a.chunk : 0u;
        const unsigned tiles = min((unsigned)a.chunk, (unsigned)a.n_qtiles - first);
        const unsigned at = seq - per_xcd * first;
        group = (int)(at / tiles * 8u + (b & 7u));
        qt = (int)(first + at % tiles);
        return group < a.n_groups;
    }
    group = (int)(b % (unsigned)a.n_groups);
    qt = (int)(b / (unsigned)a.n_groups);
    return true;
}

// Candidates of one workgroup: passing pairs staged per query, written out once.
template <int NQ>
struct ScanSlots {
    uint32_t cnt[NQ];
    uint2 slot[NQ * kScanSlots];
};

template <int NQ>
__device__ __forceinline__ void scan_append(ScanSlots<NQ> &S, const RowScanArgs &a, int e, int q, uint32_t key,
                                            uint32_t row) {
    const uint32_t r = atomicAdd(&S.cnt[e], 1u);
    if (r < (uint32_t)kScanSlots) {
        S.slot[e * kScanSlots + r] = make_uint2(key, row);
    } else {
        const uint32_t at = __hip_atomic_fetch_add(a.cnt + (size_t)q * a.cnt_stride, 1u, __ATOMIC_RELAXED,
                                                   __HIP_MEMORY_SCOPE_AGENT);
        if (at < (uint32_t)a.cap) ((gu64 *)(a.cand + (size_t)q * a.cap))[at] = pack_u2(key, row);
    }
}

template <int NQ>
__device__ __forceinline__ void scan_flush(ScanSlots<NQ> &S, const RowScanArgs &a, int q0) {
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int e = wave; e < NQ; e += kScanWg / 64) {
        const int q = q0 + e;
        const uint32_t n = min(S.cnt[e], (uint32_t)kScanSlots);
        if (n == 0 || q >= a.nq) continue;
        uint32_t at = 0;
        if (lane == 0)
            at = __hip_atomic_fetch_add(a.cnt + (size_t)q * a.cnt_stride, n, __ATOMIC_RELAXED,
                                        __HIP_MEMORY_SCOPE_AGENT);
        at = __shfl(at, 0, 64);
        if (lane < (int)n && at + lane < (uint32_t)a.cap) {
            const uint2 v = S.slot[e * kScanSlots + lane];
            ((gu64 *)(a.cand + (size_t)q * a.cap))[at + lane] = pack_u2(v.x, v.y);
        }
    }
}

// Orders the LDS accesses of one wave's lanes (no other wave touches the region).
__device__ __forceinline__ void lanes_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Float rows.  A workgroup takes 256 rows of the round against NQ queries.  A wave copies 64 rows x 32 dimensions at a time into its own 8 KB of LDS (each
// load instruction 8 whole 128-byte row pieces, the next chunk's loads in flight under the current
// one's arithmetic) and reads them back one row a lane; slot c of row r sits at c ^ ((r >> 1) & 7),
// which spreads the 16 lanes of a ds_read_b128 pass over all 64 banks.  No barrier until the flush.
// A row's terms meet in two sums, added at the end: dimensions [0, 64) and [64, 128) for dpad 65..128,
// else the even and the odd runs of 32 (shorter chains round less; the order is that of the earlier
// kernel, whose scores these are bit for bit).  The running sum is swapped for the other one wherever
// the half changes.  A row's dimensions are read 32 at a time and summed 16 at a time, so the padding
// past the last 16 costs nothing (dim 100: 112 of 128).
template <int M, bool DENSE, int NQ>
__global__ __launch_bounds__(kScanWg) void k_valu_rows(RowScanArgs a) {
    __shared__ floatx4 tile[4][64 * 8];
    __shared__ ScanSlots<DENSE ? 1 : NQ> S;
    constexpr bool kTwo = M == JACC;  // the metric keeps two sums
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int group, qt;
    if (!scan_tile(a, group, qt)) return;
    const int q0 = qt * NQ;
    const int nk = a.dpad >> 5, nh = (a.dim + 15) >> 4;  // chunks of 32 dimensions, halves of 16 to sum
    const long r0 = a.row_begin + (long)group * kScanWg + 64 * wave;
    const long last = a.row_end - 1;
    if constexpr (!DENSE) {
        if (tid < NQ) S.cnt[tid] = 0;
        __syncthreads();
    }
    const float *base = (const float *)a.base;
    const cfloat *qp = (const cfloat *)((const float *)a.qry + (size_t)q0 * a.dpad);
    floatx4 *const my = tile[wave];

    // chunk kc of the wave's rows: lane l takes quad l & 7 of rows l / 8, l / 8 + 8, ... (rows past
    // the round repeat its last row, in bounds; they are not evaluated)
    floatx4 st[8];
    auto load = [&](int kc) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const long r = min(r0 + (lane >> 3) + 8 * i, last);
            st[i] = *(const floatx4 *)(base + (size_t)r * a.dpad + 32 * kc + 4 * (lane & 7));
        }
        if constexpr (M == L2) {
            if (a.shift) {
                const floatx4 sh = *(const floatx4 *)(a.shift + 32 * kc + 4 * (lane & 7));
#pragma unroll
                for (int i = 0; i < 8; ++i) st[i] += sh;
            }
        }
    };
    float s0[NQ], s1[NQ], t0[kTwo ? NQ : 1], t1[kTwo ? NQ : 1];
#pragma unroll
    for (int e = 0; e < NQ; ++e) {
        s0[e] = s1[e] = 0.0f;
        if constexpr (kTwo) t0[e] = t1[e] = 0.0f;
    }
    const int half_shift = (a.dpad > 64 && a.dpad <= 128) ? 1 : 0;  // chunks per half, log2
    // query e's dimensions [32 kc + 16 c, + 16)
    auto query = [&](int e, int kc, int c) -> floatx16 {
        return *(const cfloatx16 *)(qp + (size_t)e * a.dpad + 32 * kc + 16 * c);
    };
    load(0);
    floatx16 yn = query(0, 0, 0);
    for (int kc = 0; kc < nk; ++kc) {
        if (kc > 0 && ((kc >> half_shift) & 1) != (((kc - 1) >> half_shift) & 1)) {
#pragma unroll
            for (int e = 0; e < NQ; ++e) {
                const float x = s0[e];
                s0[e] = s1[e];
                s1[e] = x;
                if constexpr (kTwo) {
                    const float y = t0[e];
                    t0[e] = t1[e];
                    t1[e] = y;
                }
            }
        }
        lanes_sync();
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int r = (lane >> 3) + 8 * i;
            my[r * 8 + ((lane & 7) ^ ((r >> 1) & 7))] = st[i];
        }
        lanes_sync();
        load(min(kc + 1, nk - 1));  // branch-free: past the end it re-reads the last chunk
#pragma unroll
        for (int c = 0; c < 2; ++c) {  // 16 dimensions at a time
            if (2 * kc + c >= nh) break;  // uniform: the rest of the row is padding
            floatx4 x[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) x[i] = my[lane * 8 + ((4 * c + i) ^ ((lane >> 1) & 7))];
#pragma unroll
            for (int e = 0; e < NQ; ++e) {
                // the next step's query values are asked for before this step's arithmetic: scalar
                // loads return in any order, so a step waits for all of them
                const floatx16 y = yn;
                yn = e + 1 < NQ ? query(e + 1, kc, c) : (c == 0 ? query(0, kc, 1) : query(0, min(kc + 1, nk - 1), 0));
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int j = 0; j < 16; j += 2) {
                    float y0 = y[j], y1 = y[j + 1];
                    if constexpr (M == JACC) {
                        y0 = fabsf(y0);
                        y1 = fabsf(y1);
                    }
                    accum2<M>(s0[e], t0[kTwo ? e : 0], y0, y1, x[j >> 2][j & 3], x[j >> 2][(j & 3) + 1]);
                }
            }
        }
    }
    const long row = r0 + lane;
    const bool live = row < a.row_end;
#pragma unroll
    for (int e = 0; e < NQ; ++e) {
        const int q = q0 + e;
        if (q >= a.nq) break;  // uniform
        const float ta = M == LINF ? fmaxf(s0[e], s1[e]) : s0[e] + s1[e];
        const float tb = kTwo ? t0[kTwo ? e : 0] + t1[kTwo ? e : 0] : 0.0f;
        const float v = finish<M>(ta, tb);
        if constexpr (DENSE) {
            if (live)
                ((gu64 *)(a.cand + (size_t)q * a.cap))[row - a.cand_row0] = pack_u2(score_key(nan_last(v)), (uint32_t)row);
        } else {
            if (live && v <= a.tau[q]) scan_append<NQ>(S, a, e, q, score_key(v), (uint32_t)row);
        }
    }
    if constexpr (!DENSE) scan_flush<NQ>(S, a, q0);
}

// Packed codes of W words (a power of two): popcount of XOR, two VALU operations per word and query.
// A lane reads its rows' words straight into registers (32-byte rows are contiguous over the wave).
// Against the fp4 matrix-core scan it reads a quarter of the bytes, and v_xor + v_bcnt run at about 32 T
// operations a second: 4M x 256 bits, k = 10, whole search: 16 queries 231 -> 119 us; at 32 it takes 161
// where the fp4 scan takes 171, and at 1,024 bits 279 against 265, hence kHamSmallQueries = 16.
// FILTER takes R = 32 / W rows a lane (at most 4), 64 apart, so that the query words a wave reads
// serve R rows.
template <int W, bool DENSE>
constexpr int ham_rows_per_lane() { return DENSE ? 1 : (W >= 32 ? 1 : (W >= 16 ? 2 : 4)); }

template <int W, bool DENSE, int NQ>
__global__ __launch_bounds__(kScanWg) void k_ham_rows(RowScanArgs a) {
    __shared__ ScanSlots<DENSE ? 1 : NQ> S;
    constexpr int R = ham_rows_per_lane<W, DENSE>();
    constexpr int B = W < 8 ? W : 8;  // words per step
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    int group, qt;
    if (!scan_tile(a, group, qt)) return;
    const int q0 = qt * NQ;
    const long r0 = a.row_begin + ((long)group * 4 + wave) * 64 * R + lane;
    const cuint32 *qp = (const cuint32 *)((const uint32_t *)a.qry + (size_t)q0 * W);
    uint32_t xv[R][W];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const uint32_t *x = (const uint32_t *)a.base + (size_t)min(r0 + 64 * r, a.row_end - 1) * W;
        if constexpr (W >= 4) {
#pragma unroll
            for (int w = 0; w < W; w += 4) {
                const uint4 v = *(const uint4 *)(x + w);
                xv[r][w] = v.x;
                xv[r][w + 1] = v.y;
                xv[r][w + 2] = v.z;
                xv[r][w + 3] = v.w;
            }
        } else {
#pragma unroll
            for (int w = 0; w < W; ++w) xv[r][w] = x[w];
        }
    }
    if constexpr (!DENSE) {
        if (tid < NQ) S.cnt[tid] = 0;
        __syncthreads();
    }
    uint32_t d[R][NQ];
#pragma unroll
    for (int e = 0; e < NQ; ++e)
#pragma unroll
        for (int r = 0; r < R; ++r) d[r][e] = 0;
#pragma unroll
    for (int b = 0; b < W; b += B)
#pragma unroll
        for (int e = 0; e < NQ; ++e)
#pragma unroll
            for (int w = 0; w < B; ++w) {
                const uint32_t y = qp[e * W + b + w];
#pragma unroll
                for (int r = 0; r < R; ++r) d[r][e] += (uint32_t)__popc(xv[r][b + w] ^ y);
            }
#pragma unroll
    for (int e = 0; e < NQ; ++e) {
        const int q = q0 + e;
        if (q >= a.nq) break;  // uniform
        const float tq = DENSE ? 0.0f : a.tau[q];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const long row = r0 + 64 * r;
            const float v = (float)d[r][e];
            if constexpr (DENSE) {
                if (row < a.row_end)
                    ((gu64 *)(a.cand + (size_t)q * a.cap))[row - a.cand_row0] = pack_u2(score_key(v), (uint32_t)row);
            } else {
                if (row < a.row_end && v <= tq) scan_append<NQ>(S, a, e, q, score_key(v), (uint32_t)row);
            }
        }
    }
    if constexpr (!DENSE) scan_flush<NQ>(S, a, q0);
}

// Launches `kernel` over the rows of `a` in groups of `group_rows` against its query tiles of NQ.
template <class K>
static void launch_rows(K kernel, RowScanArgs a, int nq_tile, long group_rows, hipStream_t s) {
    a.n_qtiles = ceil_div(a.nq, nq_tile);
    a.chunk = (int)std::clamp(kScanQueryBytes / (4L * nq_tile * a.dpad), 1L, (long)a.n_qtiles);
    const long re = a.row_end;
    const long most = std::max(1L, kScanMaxWgs / a.n_qtiles / 8 * 8) * group_rows;  // rows of one launch
    for (long rb = a.row_begin; rb < re; rb += most) {
        a.row_begin = rb;
        a.row_end = std::min(re, rb + most);
        a.n_groups = (int)((a.row_end - rb + group_rows - 1) / group_rows);
        // Spread where the XCDs' shares differ by little: eight or more groups an XCD, or idle places at
        // most 8% of the groups.  Otherwise, in plain order, the whole chip shares them, and each XCD reads
        // every group.  (From 64 groups on alone: L1 20,000 x 128, whose filter rounds have 24 and 47
        // groups, 4,000 queries 682 us, with the second rule 575; spread over 16 places, the 12 groups of
        // 5,000 x 128 229 -> 250.)
        const long places = (a.n_groups + 7) / 8 * 8L;
        a.spread = a.n_qtiles > 1 && (a.n_groups >= 64 || (places - a.n_groups) * 100 <= a.n_groups * 8L);
        const long wgs = (a.spread ? places : (long)a.n_groups) * a.n_qtiles;
        scan_launch(kernel, dim3((unsigned)wgs), dim3(kScanWg), 0, s, a);
    }
}

// Whether a round takes 4-query tiles (see kScanFewWgs).
static bool few_tiles(const RowScanArgs &a, long group_rows) {
    const long groups = (a.row_end - a.row_begin + group_rows - 1) / group_rows;
    return a.nq <= kScanFew || groups * ceil_div(a.nq, kScanQueries) < kScanFewWgs;
}

template <int M>
static void launch_valu_m(const RowScanArgs &a, bool dense, hipStream_t s) {
    const bool few = few_tiles(a, kScanWg);
    if (dense && few) launch_rows(k_valu_rows<M, true, kScanFew>, a, kScanFew, kScanWg, s);
    else if (dense) launch_rows(k_valu_rows<M, true, kScanQueries>, a, kScanQueries, kScanWg, s);
    else if (few) launch_rows(k_valu_rows<M, false, kScanFew>, a, kScanFew, kScanWg, s);
    else launch_rows(k_valu_rows<M, false, kScanQueries>, a, kScanQueries, kScanWg, s);
}

template <int W>
static void launch_ham_w(const RowScanArgs &a, bool dense, hipStream_t s) {
    constexpr long kDense = (long)kScanWg * ham_rows_per_lane<W, true>();
    constexpr long kFilter = (long)kScanWg * ham_rows_per_lane<W, false>();
    if (dense) launch_rows(k_ham_rows<W, true, kScanFew>, a, kScanFew, kDense, s);
    else if (few_tiles(a, kFilter)) launch_rows(k_ham_rows<W, false, kScanFew>, a, kScanFew, kFilter, s);
    else launch_rows(k_ham_rows<W, false, kScanQueries>, a, kScanQueries, kFilter, s);
}

void launch_row_scan(int metric, bool dense, const void *base, const float *shift, const void *qry, const float *tau,
                     int nq, int dim, int dpad, long row_begin, long row_end, uint2 *cand, uint32_t *cnt,
                     int cnt_stride, int cap, hipStream_t s) {
    if (nq <= 0 || row_end <= row_begin) return;
    RowScanArgs a{};
    a.base = base;
    a.qry = qry;
    a.shift = shift;
    a.dim = dim;
    a.dpad = dpad;
    a.nq = nq;
    a.row_begin = row_begin;
    a.row_end = row_end;
    a.tau = tau;
    a.cand = cand;
    a.cnt = cnt;
    a.cnt_stride = cnt_stride;
    a.cap = cap;
    a.cand_row0 = row_begin;
    switch (metric) {
        case L2: launch_valu_m<L2>(a, dense, s); break;
        case L1: launch_valu_m<L1>(a, dense, s); break;
        case MINK: launch_valu_m<MINK>(a, dense, s); break;
        case LINF: launch_valu_m<LINF>(a, dense, s); break;
        case HAMF: launch_valu_m<HAMF>(a, dense, s); break;
        case MAHA: launch_valu_m<MAHA>(a, dense, s); break;
        case JACC: launch_valu_m<JACC>(a, dense, s); break;
        case HELL: launch_valu_m<HELL>(a, dense, s); break;
        case HAMMING_PACKED:
            switch (dpad) {
                case 1: launch_ham_w<1>(a, dense, s); break;
                case 2: launch_ham_w<2>(a, dense, s); break;
                case 4: launch_ham_w<4>(a, dense, s); break;
                case 8: launch_ham_w<8>(a, dense, s); break;
                case 16: launch_ham_w<16>(a, dense, s); break;
                default: launch_ham_w<32>(a, dense, s); break;
            }
            break;
        default: break;
    }
}

}  // namespace vh
