// pq_train.hip -- product-quantizer training and encoding with all sub-spaces in one launch.
//
// ProductQuantizer::train (vector-index/src/ivf/pq.rs:53-107) is one k-means per sub-space, encode
// (pq.rs:178-214) the nearest sub-centroid of each sub-vector.  A sub-space is narrow (a few dozen
// dimensions at most) and has at most 256 centroids, so the general engine (kmeans.hip) spends it on
// padding (rows padded to 32 dimensions, MFMA tiles) and on a dozen launches an iteration, one sub-space
// after another.  Here an iteration is three launches for all sub-spaces:
//   1. k_pq_assign -- a point a lane (two for narrow sub-vectors), its dimensions in registers; the
//      centroids are wave-uniform and come through the scalar cache, so an element costs one subtract
//      and one multiply-add.  The scores are the direct form the general engine's fix-up computes
//      (sequential over the dimensions, lowest index among equal ones), so every assignment is the one
//      its certified MFMA scan ends with.  (Its small-set kernel, for up to 1e6 (point, centroid) pairs,
//      adds slices of a row, so there a point between two centroids may go by another last bit);
//   2. k_pq_sums -- deviations x - c in 64-bit fixed point with the cluster's own scale, as in
//      kmeans.hip, summed with LDS integer atomics (exact in any order) and written per workgroup;
//   3. k_pq_finalize -- the workgroups' sums added up, new = old + sum / count, the centroid's shift.
// Bound: the vector ALUs in the assignment.  65,536 x 128 points, 8 sub-spaces of 256 centroids, 10
// iterations, host data in, codebooks out: 21 ms by sub-space k-means, 3.3 here (1.7 of it the upload and
// allocations, which vary by box); an assignment of all sub-spaces takes 129 us (94 at the rate of its subtracts and
// multiply-adds), the sums 18, the new centroids 8.  Encoding the same points: 524 us -> 134.
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <memory>
#include <vector>

#include "pq_scan.h"
#include "vh_runtime.h"

namespace vh {

namespace {

typedef __attribute__((address_space(4))) const float cfloat;  // read through the scalar cache

constexpr int kPqThreads = 256;
constexpr int kPqMaxK = 256;

template <int N>
struct Fixed {
    float v[N];
};

// N consecutive uniform floats.
template <int N>
__device__ __forceinline__ Fixed<N> uniform_row(const cfloat *p) {
    Fixed<N> r;
#pragma unroll
    for (int i = 0; i < N; ++i) r.v[i] = p[i];
    return r;
}

// Nearest of the k sub-centroids (rows of DSP floats at cent + m * k * DSP, zero past ds) of the points'
// sub-vectors m = blockIdx.y, which start at x + point * stride + m * ds (vec: 16-byte aligned).  Point
// i's index goes to out[i * out_stride + m * out_step].  TRAIN (squared L2) also counts each cluster's
// points and bounds their deviation |x_d - c_d| (count, devmax: k per sub-space); sub-spaces with
// active[m] == 0 are skipped.
template <int MT, int DSP, int P, bool TRAIN>
__global__ __launch_bounds__(kPqThreads) void k_pq_assign(const float *__restrict__ x, long n, long stride, long m_step,
                                                          int ds, int vec, const float *__restrict__ cent, int k,
                                                          uint8_t *__restrict__ out, long out_stride, long out_step,
                                                          uint32_t *__restrict__ count, uint32_t *__restrict__ devmax,
                                                          const uint32_t *__restrict__ active) {
    __shared__ uint32_t s_cnt[TRAIN ? kPqMaxK : 1], s_dev[TRAIN ? kPqMaxK : 1];
    constexpr bool hib = hib_metric(MT);
    constexpr int U = DSP <= 16 ? 2 : 1;  // centroids per step
    const int m = blockIdx.y, tid = threadIdx.x;
    if constexpr (TRAIN) {
        if (!active[m]) return;
        s_cnt[tid] = 0;
        s_dev[tid] = 0;
        __syncthreads();
    }
    const long i0 = (long)blockIdx.x * kPqThreads * P + tid;
    float xr[P][DSP];
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const float *xs = x + min(i0 + (long)p * kPqThreads, n - 1) * stride + m * m_step;
        if (vec) {
#pragma unroll
            for (int d = 0; d < DSP; d += 4) {
                const float4 v = d < ds ? *(const float4 *)(xs + d) : float4{0, 0, 0, 0};
                xr[p][d] = v.x;
                xr[p][d + 1] = v.y;
                xr[p][d + 2] = v.z;
                xr[p][d + 3] = v.w;
            }
        } else {
#pragma unroll
            for (int d = 0; d < DSP; ++d) xr[p][d] = d < ds ? xs[d] : 0.0f;
        }
    }
    float best[P];
    int bi[P];
#pragma unroll
    for (int p = 0; p < P; ++p) {
        best[p] = hib ? -INFINITY : INFINITY;
        bi[p] = 0;
    }
    const cfloat *cm = (const cfloat *)(cent + (size_t)m * k * DSP);
    auto score = [&](const Fixed<DSP> &c, int j) {
#pragma unroll
        for (int p = 0; p < P; ++p) {
            Acc<MT> acc;
#pragma unroll
            for (int d = 0; d < DSP; ++d) acc.step(xr[p][d], c.v[d]);
            const float v = acc.finish();
            if (hib ? v > best[p] : v < best[p]) {
                best[p] = v;
                bi[p] = j;
            }
        }
    };
    // the next step's centroids are asked for before this step's arithmetic (past the end: the last row)
    Fixed<DSP> nx[U];
#pragma unroll
    for (int u = 0; u < U; ++u) nx[u] = uniform_row<DSP>(cm + (size_t)min(u, k - 1) * DSP);
    for (int j = 0; j < k; j += U) {
        Fixed<DSP> c[U];
#pragma unroll
        for (int u = 0; u < U; ++u) c[u] = nx[u];
#pragma unroll
        for (int u = 0; u < U; ++u) nx[u] = uniform_row<DSP>(cm + (size_t)min(j + U + u, k - 1) * DSP);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < U; ++u) score(c[u], min(j + u, k - 1));  // a repeated last row never wins
    }
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const long i = i0 + (long)p * kPqThreads;
        if (i >= n) continue;
        out[i * out_stride + m * out_step] = (uint8_t)bi[p];
        if constexpr (TRAIN) {
            atomicAdd(&s_cnt[bi[p]], 1u);
            atomicMax(&s_dev[bi[p]], __float_as_uint(sqrtf(fmaxf(best[p], 0.0f)) * 1.0001f));
        }
    }
    if constexpr (TRAIN) {
        __syncthreads();
        if (tid < k && s_cnt[tid]) {
            atomicAdd(&count[m * k + tid], s_cnt[tid]);
            atomicMax(&devmax[m * k + tid], s_dev[tid]);
        }
    }
}

// Rows i0 .. i0 + rows of the n points, [rows][dim] at x, into sub-space-major rows [m][n][DSP] of the
// sub-spaces m0 .. m0 + m_sub, zero past ds; bad is set when some value is infinite (what the general
// engine's check rejects).
template <int DSP>
__global__ __launch_bounds__(256) void k_pq_split(const float *__restrict__ x, long rows, long i0, long n, int dim,
                                                  int ds, int m0, int m_sub, float *__restrict__ out,
                                                  uint32_t *__restrict__ bad) {
    const long total = rows * m_sub * DSP;
    for (long t = blockIdx.x * 256L + threadIdx.x; t < total; t += gridDim.x * 256L) {
        // consecutive threads write a row's DSP values, then the next sub-space of the same point, so that
        // a point's row is read once
        const int d = (int)(t % DSP);
        const long r = t / DSP;
        const int m = (int)(r % m_sub);
        const long i = r / m_sub;
        const float v = d < ds ? x[i * dim + (long)(m0 + m) * ds + d] : 0.0f;
        if (fabsf(v) == INFINITY) *bad = 1;
        out[((long)m * n + i0 + i) * DSP + d] = v;
    }
}

// Fixed-point exponent of a cluster (kmeans.hip, k_update_scales): no sum can overflow.
__device__ __forceinline__ int pq_exponent(float dev, uint32_t count) {
    if (!(dev > 0.0f) || count == 0) return 60;
    int e1, e2;
    (void)frexpf(dev, &e1);
    (void)frexp((double)count + 1.0, &e2);
    return min(60, 61 - e1 - e2);
}

// Workgroup (b, m): the deviations of points [b * per, + per) of sub-space m, into
// part[(m * gridDim.x + b) * k * DSP].  DSP consecutive lanes take a point's dimensions.
template <int DSP>
__global__ __launch_bounds__(kPqThreads) void k_pq_sums(const float *__restrict__ xs, long n, long per,
                                                        const float *__restrict__ cent, int k,
                                                        const uint8_t *__restrict__ assign,
                                                        const uint32_t *__restrict__ count,
                                                        const uint32_t *__restrict__ devmax,
                                                        unsigned long long *__restrict__ part,
                                                        const uint32_t *__restrict__ active) {
    extern __shared__ unsigned long long s_acc[];  // k * DSP sums, then k scales, then the k * DSP centroids
    const int m = blockIdx.y, tid = threadIdx.x, kd = k * DSP;
    if (!active[m]) return;
    double *s_scale = (double *)(s_acc + kd);
    float *s_cent = (float *)(s_scale + k);
    for (int t = tid; t < kd; t += kPqThreads) {
        s_acc[t] = 0ull;
        s_cent[t] = cent[(size_t)m * kd + t];
    }
    if (tid < k) s_scale[tid] = ldexp(1.0, pq_exponent(__uint_as_float(devmax[m * k + tid]), count[m * k + tid]));
    __syncthreads();
    constexpr int PTS = kPqThreads / DSP;  // points at a time
    constexpr int UN = 8;                  // of which this many rounds are in flight
    const int d = tid % DSP, slot = tid / DSP;
    const long b0 = blockIdx.x * per, b1 = min(n, b0 + per);
    const float *xm = xs + (size_t)m * n * DSP;
    const uint8_t *am = assign + (size_t)m * n;
    for (long i0 = b0 + slot; i0 < b1; i0 += PTS * UN) {
        float v[UN];
        int c[UN];
#pragma unroll
        for (int u = 0; u < UN; ++u) {
            const long i = min(i0 + u * PTS, b1 - 1);
            v[u] = xm[i * DSP + d];
            c[u] = am[i];
        }
#pragma unroll
        for (int u = 0; u < UN; ++u)
            if (i0 + u * PTS < b1) {
                const long long q = llrint(((double)v[u] - (double)s_cent[c[u] * DSP + d]) * s_scale[c[u]]);
                if (q) atomicAdd(&s_acc[c[u] * DSP + d], (unsigned long long)q);
            }
    }
    __syncthreads();
    unsigned long long *out = part + ((size_t)m * gridDim.x + blockIdx.x) * kd;
    for (int t = tid; t < kd; t += kPqThreads) out[t] = s_acc[t];
}

// New centroids of sub-space blockIdx.y, 256 / DSP clusters a workgroup: old + deviation sum / count, the
// squared shift (0 for an empty cluster, which keeps its centroid), and the counters cleared for the next
// iteration.
template <int DSP>
__global__ __launch_bounds__(kPqThreads) void k_pq_finalize(float *__restrict__ cent, int k, int parts,
                                                            const unsigned long long *__restrict__ part,
                                                            uint32_t *__restrict__ count, uint32_t *__restrict__ devmax,
                                                            float *__restrict__ shifts,
                                                            const uint32_t *__restrict__ active) {
    const int m = blockIdx.y, tid = threadIdx.x, kd = k * DSP;
    if (!active[m]) return;
    const int c = blockIdx.x * (kPqThreads / DSP) + tid / DSP, d = tid % DSP;
    const bool live = c < k;
    uint32_t cnt = 0;
    float dev = 0.0f;
    if (live) {
        cnt = count[m * k + c];
        dev = __uint_as_float(devmax[m * k + c]);
    }
    __syncthreads();
    if (live && d == 0) {
        count[m * k + c] = 0;
        devmax[m * k + c] = 0;
    }
    float sh = 0.0f;
    if (live && cnt) {
        const unsigned long long *p = part + (size_t)m * parts * kd + c * DSP + d;
        unsigned long long s0 = 0, s1 = 0, s2 = 0, s3 = 0;
        int b = 0;
        for (; b + 4 <= parts; b += 4) {
            s0 += p[(size_t)b * kd];
            s1 += p[(size_t)(b + 1) * kd];
            s2 += p[(size_t)(b + 2) * kd];
            s3 += p[(size_t)(b + 3) * kd];
        }
        for (; b < parts; ++b) s0 += p[(size_t)b * kd];
        const long long sum = (long long)(s0 + s1 + s2 + s3);
        const double inv = ldexp(1.0, -pq_exponent(dev, cnt)) / (double)cnt;
        float *cp = cent + ((size_t)m * k + c) * DSP + d;
        const float old = *cp, nv = (float)((double)old + (double)sum * inv);
        *cp = nv;
        sh = (nv - old) * (nv - old);
    }
#pragma unroll
    for (int o = DSP / 2; o > 0; o >>= 1) sh += __shfl_xor(sh, o, 64);
    if (live && d == 0) shifts[m * k + c] = sh;
}

// Dynamic LDS of k_pq_sums<dsp> for k clusters: sums, scales and centroids.
constexpr size_t pq_sums_lds(size_t dsp, size_t k) { return k * dsp * 8 + k * 8 + k * dsp * 4; }

static_assert(pq_sums_lds(16, kPqMaxK) <= 65536 && pq_sums_lds(32, kPqMaxK) <= 163840, "LDS of a workgroup");

int padded_ds(size_t ds) { return ds <= 4 ? 4 : (ds <= 8 ? 8 : (ds <= 16 ? 16 : 32)); }

// Codebooks [m_sub][rows of ds floats, `have` per sub-space at stride `ks`] into [m_sub][have][DSP].
std::vector<float> pad_codebooks(const float *cb, size_t m_sub, size_t ks, size_t have, size_t ds, int dsp) {
    std::vector<float> t(m_sub * have * dsp, 0.0f);
    for (size_t m = 0; m < m_sub; ++m)
        for (size_t j = 0; j < have; ++j)
            std::copy(cb + (m * ks + j) * ds, cb + (m * ks + j + 1) * ds, t.begin() + (m * have + j) * dsp);
    return t;
}

// Points per lane: two where a sub-vector takes at most 16 registers.
constexpr int pq_points(int dsp) { return dsp <= 16 ? 2 : 1; }

template <int MT, int DSP, bool TRAIN>
void launch_assign(const float *x, long n, long stride, long m_step, int ds, int vec, const float *cent, int k, int m_sub,
                   uint8_t *out, long out_stride, long out_step, uint32_t *count, uint32_t *devmax,
                   const uint32_t *active, hipStream_t s) {
    constexpr int P = pq_points(DSP);
    const long per = (long)kPqThreads * P;
    hipLaunchKernelGGL((k_pq_assign<MT, DSP, P, TRAIN>), dim3((unsigned)((n + per - 1) / per), (unsigned)m_sub),
                       dim3(kPqThreads), 0, s, x, n, stride, m_step, ds, vec, cent, k, out, out_stride, out_step, count,
                       devmax, active);
}

#define VH_DSP_SWITCH(dsp, CALL) \
    switch (dsp) {               \
        case 4: CALL(4); break;  \
        case 8: CALL(8); break;  \
        case 16: CALL(16); break; \
        default: CALL(32); break; \
    }

}  // namespace

// Sub-vectors this short are encoded by pq_encode_narrow and trained by pq_train_batched.
bool pq_narrow(size_t ds) { return ds <= 32; }

int pq_encode_narrow(const float *d_x, size_t n, size_t dim, size_t m_sub, size_t ks, int metric, const float *codebooks,
                     int dev, uint8_t *d_codes, DevBuf &cent, hipStream_t s) {
    if (n == 0) return VHIP_OK;
    const size_t ds = dim / m_sub;
    const int dsp = padded_ds(ds);
    const std::vector<float> t = pad_codebooks(codebooks, m_sub, ks, ks, ds, dsp);
    VH_CHECK(cent.ensure(dev, t.size() * sizeof(float)));
    VH_HIP(hipMemcpyAsync(cent.p, t.data(), t.size() * sizeof(float), hipMemcpyHostToDevice, s));
    VH_HIP(hipStreamSynchronize(s));  // t is released at return
    const int vec = ds % 4 == 0 && dim % 4 == 0 && (uintptr_t)d_x % 16 == 0 ? 1 : 0;
#define VH_ENC_DSP(DSP)                                                                                              \
    launch_assign<VH_ENC_MT, DSP, false>(d_x, (long)n, (long)dim, (long)ds, (int)ds, vec, cent.as<float>(), (int)ks, \
                                         (int)m_sub, d_codes, (long)m_sub, 1, nullptr, nullptr, nullptr, s)
#define VH_ENC(MT)                         \
    do {                                   \
        constexpr int VH_ENC_MT = MT;      \
        VH_DSP_SWITCH(dsp, VH_ENC_DSP)     \
    } while (0)
    VH_METRIC_SWITCH(metric, VH_ENC)
#undef VH_ENC
#undef VH_ENC_DSP
    VH_HIP(hipGetLastError());
    return VHIP_OK;
}

namespace {

// Device memory of `g` sub-spaces trained at once, uploaded `slab` rows at a time, in one allocation (freeing
// a large buffer takes about 0.24 ms): byte offsets of the uploaded rows, the points by sub-space, the partial
// sums, centroids, shifts, counters (counts, deviations, active flags, bad) and assignments.
struct PqGroupMem {
    size_t raw, xs, part, cent, shift, state, assign, total = 0;
    PqGroupMem(size_t n, size_t dim, size_t slab, size_t g, size_t ek, size_t dsp, size_t parts) {
        auto take = [&](size_t bytes) {
            const size_t o = total;
            total += round_up(bytes, 256);
            return o;
        };
        raw = take(slab * dim * sizeof(float));
        xs = take(n * g * dsp * sizeof(float));
        part = take(parts * g * ek * dsp * sizeof(unsigned long long));
        cent = take(g * ek * dsp * sizeof(float));
        shift = take(g * ek * sizeof(float));
        state = take((2 * g * ek + g + 1) * sizeof(uint32_t));
        assign = take(n * g);
    }
};

// Points of a workgroup of the sums of g sub-spaces: about two workgroups a CU in all, at least 256 points.
size_t pq_sum_points(int ordinal, size_t n, size_t g) {
    const size_t want = std::max<size_t>(1, (size_t)device_grid_cap(ordinal) / g);
    return std::max<size_t>(256, (n + want - 1) / want);
}

constexpr size_t kPqSlabBytes = (size_t)1 << 30;  // of an upload
constexpr size_t kPqMinSlabBytes = (size_t)16 << 20;
constexpr size_t kPqAskBytes = (size_t)1 << 30;   // a training set that takes less does not ask what is free
constexpr size_t kPqMaxGroup = 65535;             // sub-spaces are a grid dimension

// Device memory that training may take: half of what is free (the rest stays for the program's other
// objects), or VHIP_PQ_TRAIN_BYTES.
size_t pq_train_limit(size_t bytes) {
    if (const char *e = std::getenv("VHIP_PQ_TRAIN_BYTES")) return (size_t)std::strtoull(e, nullptr, 10);
    if (bytes <= kPqAskBytes) return bytes;
    size_t free_b = 0, total_b = 0;
    if (hipMemGetInfo(&free_b, &total_b) != hipSuccess) {
        (void)hipGetLastError();
        return bytes;
    }
    return free_b / 2;
}

}  // namespace

// ProductQuantizer::train under squared L2 for sub-vectors of at most 32 dimensions: the same codebooks as
// one vhip_kmeans_fit per sub-space (seed + 1 + m, shuffled start).  All sub-spaces at once where they fit
// the device memory (about 4 (dim + 1) bytes a point beside an upload of at most 1 GiB, more where ds is
// padded), else as many at a time as do, each group uploading the rows again; one at a time takes less
// than the general engine does for it.
int pq_train_batched(int ordinal, const float *data, size_t n, size_t dim, size_t m_sub, size_t ks, size_t max_iters,
                     float tol, const float *init_codebooks, uint64_t seed, float *out_codebooks) {
    if (n > 0x7fffffffull) return set_error(VHIP_ERR_INVALID_CONFIG, "k-means supports n < 2^31 points");
    const size_t ds = dim / m_sub, ek = std::min(ks, n);
    const int dsp = padded_ds(ds), k = (int)ek;
    const size_t kd = ek * dsp;
    VH_CHECK(open_device(ordinal));
    hipStream_t s;
    VH_HIP(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
    DevBuf mem;
    PinnedStager st;
    std::vector<float> start, sh, fin;
    std::vector<uint32_t> on;
    // declared after the buffers: the stream is drained and destroyed before they are released
    std::unique_ptr<ihipStream_t, void (*)(hipStream_t)> hold(s, [](hipStream_t q) {
        (void)hipStreamSynchronize(q);
        (void)hipStreamDestroy(q);
    });
    st.dev = ordinal;
    if (init_codebooks) {
        start = pad_codebooks(init_codebooks, m_sub, ks, ek, ds, dsp);
    } else {
        start.assign(m_sub * ek * dsp, 0.0f);
        for (size_t m = 0; m < m_sub; ++m) {
            const std::vector<uint32_t> idx = row_permutation(n, seed + 1 + m);
            for (size_t j = 0; j < ek; ++j) {
                const float *row = data + (size_t)idx[j] * dim + m * ds;
                std::copy(row, row + ds, start.begin() + (m * ek + j) * dsp);
            }
        }
    }
    // sub-spaces at a time and rows an upload: the most that the limit allows and the allocation gives
    size_t slab = std::min(n, std::max<size_t>(1, kPqSlabBytes / (dim * sizeof(float))));
    const size_t slab_min = std::min(n, std::max<size_t>(1, kPqMinSlabBytes / (dim * sizeof(float))));
    size_t group = std::min(m_sub, kPqMaxGroup);
    auto layout = [&](size_t g) {
        const size_t per = pq_sum_points(ordinal, n, g);
        return PqGroupMem(n, dim, slab, g, ek, dsp, (n + per - 1) / per);
    };
    auto shrink = [&]() {  // false when nothing is left to shrink
        if (group > 1) group = (group + 1) / 2;
        else if (slab > slab_min) slab = std::max(slab_min, slab / 2);
        else return false;
        return true;
    };
    const size_t limit = pq_train_limit(layout(group).total);
    while (layout(group).total > limit && shrink()) {}
    int rc = mem.ensure(ordinal, layout(group).total);
    while (rc != VHIP_OK && shrink()) rc = mem.ensure(ordinal, layout(group).total);
    VH_CHECK(rc);
    clear_error();
    group = (m_sub + (m_sub + group - 1) / group - 1) / ((m_sub + group - 1) / group);  // groups of like size
    // Only the widest kernel can need more than 64 KB of LDS.  Its limit is shared by every thread that
    // trains, so it is set to the most that any cluster count needs, not to this call's.
    const size_t lds = pq_sums_lds(dsp, ek);
    if (dsp == 32)
        VH_HIP(hipFuncSetAttribute((const void *)k_pq_sums<32>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                   (int)pq_sums_lds(32, kPqMaxK)));
    for (size_t m0 = 0; m0 < m_sub; m0 += group) {
        const size_t g = std::min(group, m_sub - m0);
        const size_t per = pq_sum_points(ordinal, n, g);
        const int parts = (int)((n + per - 1) / per);
        const PqGroupMem L(n, dim, slab, g, ek, dsp, (size_t)parts);
        VH_CHECK(mem.ensure(ordinal, L.total));  // a smaller last group may have more partial sums
        char *const p0 = mem.as<char>();
        float *raw = (float *)(p0 + L.raw), *xs = (float *)(p0 + L.xs), *cent = (float *)(p0 + L.cent),
              *shifts = (float *)(p0 + L.shift);
        unsigned long long *part = (unsigned long long *)(p0 + L.part);
        uint8_t *assign = (uint8_t *)(p0 + L.assign);
        uint32_t *count = (uint32_t *)(p0 + L.state), *devmax = count + g * ek, *active = devmax + g * ek,
                 *bad = active + g;
        launch_fill_u32(count, 2 * g * ek, 0u, s);
        launch_fill_u32(active, g, 1u, s);
        launch_fill_u32(bad, 1, 0u, s);
        for (size_t i0 = 0; i0 < n; i0 += slab) {
            const size_t rows = std::min(slab, n - i0);
            VH_CHECK(st.h2d_once(raw, data + i0 * dim, rows * dim * sizeof(float), s));
#define VH_SPLIT(DSP)                                                                                                   \
    hipLaunchKernelGGL(k_pq_split<DSP>, dim3((unsigned)std::min<size_t>(8192, (rows * g * DSP + 255) / 256)), dim3(256), \
                       0, s, raw, (long)rows, (long)i0, (long)n, (int)dim, (int)ds, (int)m0, (int)g, xs, bad)
            VH_DSP_SWITCH(dsp, VH_SPLIT)
#undef VH_SPLIT
        }
        VH_HIP(hipMemcpyAsync(cent, start.data() + m0 * kd, g * kd * sizeof(float), hipMemcpyHostToDevice, s));
        VH_HIP(hipGetLastError());
        uint32_t nonfinite = 0;
        VH_HIP(hipMemcpyAsync(&nonfinite, bad, sizeof(uint32_t), hipMemcpyDeviceToHost, s));
        VH_HIP(hipStreamSynchronize(s));
        if (nonfinite) return set_error(VHIP_ERR_INVALID_CONFIG, "data contains non-finite values");
        on.assign(g, 1u);
        sh.resize(g * ek);
        for (size_t it = 0; it < max_iters; ++it) {
#define VH_ITER(DSP)                                                                                                   \
    do {                                                                                                               \
        launch_assign<L2, DSP, true>(xs, (long)n, DSP, (long)n * DSP, DSP, 1, cent, k, (int)g, assign, 1, (long)n,      \
                                     count, devmax, active, s);                                                        \
        hipLaunchKernelGGL(k_pq_sums<DSP>, dim3((unsigned)parts, (unsigned)g), dim3(kPqThreads), lds, s, xs, (long)n,   \
                           (long)per, cent, k, assign, count, devmax, part, active);                                   \
        hipLaunchKernelGGL(k_pq_finalize<DSP>, dim3((unsigned)ceil_div((long)ek, kPqThreads / DSP), (unsigned)g),      \
                           dim3(kPqThreads), 0, s, cent, k, parts, part, count, devmax, shifts, active);               \
    } while (0)
            VH_DSP_SWITCH(dsp, VH_ITER)
#undef VH_ITER
            VH_HIP(hipGetLastError());
            if (tol >= 0.0f) {  // a sub-space stops when no centroid of it moved by more than tol
                VH_HIP(hipMemcpyAsync(sh.data(), shifts, sh.size() * sizeof(float), hipMemcpyDeviceToHost, s));
                VH_HIP(hipStreamSynchronize(s));
                bool changed = false, any = false;
                for (size_t m = 0; m < g; ++m) {
                    if (!on[m]) continue;
                    float mx = 0.0f;  // a NaN shift takes no part
                    for (size_t j = 0; j < ek; ++j) mx = std::max(mx, sh[m * ek + j]);
                    if (mx <= tol) {
                        on[m] = 0;
                        changed = true;
                    } else {
                        any = true;
                    }
                }
                if (!any) break;
                if (changed) {
                    VH_HIP(hipMemcpyAsync(active, on.data(), g * sizeof(uint32_t), hipMemcpyHostToDevice, s));
                    VH_HIP(hipStreamSynchronize(s));
                }
            }
        }
        fin.resize(g * kd);
        VH_HIP(hipMemcpyAsync(fin.data(), cent, fin.size() * sizeof(float), hipMemcpyDeviceToHost, s));
        VH_HIP(hipStreamSynchronize(s));
        for (size_t m = 0; m < g; ++m)
            for (size_t j = 0; j < ek; ++j)
                std::copy(fin.begin() + (m * ek + j) * dsp, fin.begin() + (m * ek + j) * dsp + ds,
                          out_codebooks + ((m0 + m) * ks + j) * ds);
    }
    return VHIP_OK;
}

}  // namespace vh
