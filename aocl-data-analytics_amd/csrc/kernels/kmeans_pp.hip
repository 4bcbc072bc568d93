// k-means++ initialisation for gfx950, without a host round trip per centre.
//
// The reference (source/core/clustering/kmeans/kmeans.cpp:1524-1664) keeps, per sample, the
// weight w = distance to the nearest chosen centre, draws 2 + ln k candidates per centre from
// the distribution w / sum(w), and takes the candidate with the smallest sum of min(w, d).
// Here a round is two launches on one stream, all decisions on the device:
//
//   kpp_draw (a workgroup per draw)  the previous round's costs -> its centre; that candidate's
//                                    block sums are the block sums of the new weights, so
//                                    their scan gives the total and the block of every draw;
//                                    then the sample within the block, and its row for the
//                                    cost pass (every workgroup repeats the first part);
//   kpp_cost (whole device)          the one pass over the data: the weights take in the
//                                    centre just chosen and each candidate's sum of min(w, d)
//                                    is formed.
//
// The chosen centre is not applied by a pass of its own: the cost pass of the next round reads
// every row anyway and computes its distance next to the candidates'; kpp_draw applies it to
// the rows of the few blocks it looks into. Distances are double direct differences (or
// 1 - cos for spherical k-means) summed over the features in order.
//
// Measured at 2,000,000 x 32 fp32, k = 256 (7 candidates): a round takes 73 us for the cost pass
// (288 MB: 4.0 TB/s) and 22 us for the draw, against 124 us (costs) + 64 us (update) + 43 us
// (scan) + 40 us (sums, searches, copies) and two host synchronisations before; the 256 rounds
// 90 -> 26 ms.
#include "launch.hpp"
#include <hip/hip_runtime.h>

namespace dagpu {

namespace {

constexpr int KPP_ROWS = 256; // rows staged at a time, one per thread

struct KppGeom {
    const double *inv; // inverse row norms (spherical k-means of normalised data) or null
};

__device__ __forceinline__ double kpp_cosine(double dot, const double *inv, int64_t i, int64_t j) {
    if (inv)
        dot = dot * inv[i] * inv[j];
    const double v = 1.0 - dot;
    return v > 0.0 ? v : 0.0;
}

// The weight of sample i after centre j at distance v was chosen (o: before).
__device__ __forceinline__ double kpp_min(double o, double v, bool self) {
    v = o < v ? o : v;
    v = v > 0.0 ? v : 0.0;
    return self ? 0.0 : v;
}
// The weight of a sample at distance v from the first centre.
__device__ __forceinline__ double kpp_first(double v, bool self) {
    return (!(v - v == 0.0) || v < 0.0 || self) ? 0.0 : v;
}

// LDS position of element e of a staged block of rows: one element of padding per 128 bytes,
// so that the 64 lanes of a wave, each reading its own row, do not meet in the banks.
template <typename T> __device__ __forceinline__ int kpp_pos(int e) {
    return e + e / (128 / (int)sizeof(T));
}

// Sums of the candidates over the rows of chunk blockIdx.x: part[t * nb + blockIdx.x]. Slot 0
// of crow ([feature][NT], doubles) is the centre chosen last, slots 1..nt the candidates. With
// `first` the weights are set from slot 0 and their sum goes to part[0].
// NV > 0: whole rows are staged, the 256 rows of a step being one contiguous run of memory read
// in at most NV 16-byte pieces per thread, the next step's while this one is computed; NV = 0:
// FB features of 256 rows at a time. The centres' values are the same for all lanes and come
// through scalar loads.
template <typename T, int NT, int NV, bool SPH>
__global__ __launch_bounds__(KPP_ROWS) void kpp_cost_kernel(
    const T *__restrict__ X, int n, int d, double *__restrict__ w,
    const double *__restrict__ crow, const KppState *__restrict__ st, int par, int nt, int chunk,
    double *__restrict__ part, int nb, int first, KppGeom g) {
    extern __shared__ double kpp_smem[];
    T *tile = reinterpret_cast<T *>(kpp_smem);
    __shared__ double red[KPP_ROWS / 64][NT];
    if (st->same)
        return;
    constexpr int FB = 128 / (int)sizeof(T);
    constexpr int VE = 16 / (int)sizeof(T);
    const int tid = threadIdx.x;
    const int64_t b0 = (int64_t)blockIdx.x * chunk;
    const int64_t b1 = b0 + chunk < n ? b0 + chunk : n;
    double sum[NT];
#pragma unroll
    for (int s = 0; s < NT; s++)
        sum[s] = 0.0;
    const int best = st->best;
    uint4 pre[NV > 0 ? NV : 1];
    double wpre = 0.0;
    // The step at row i0: its whole 16-byte pieces (piece p of the run goes to thread p % 256).
    auto fetch = [&](int64_t i0) {
        const int m = (int)(b1 - i0 < KPP_ROWS ? b1 - i0 : KPP_ROWS);
        const uint4 *src = reinterpret_cast<const uint4 *>(X + i0 * d);
        const int pieces = m * d / VE;
#pragma unroll
        for (int v = 0; v < (NV > 0 ? NV : 1); v++)
            if (v * KPP_ROWS + tid < pieces)
                pre[v] = src[v * KPP_ROWS + tid];
        wpre = (!first && tid < m) ? w[i0 + tid] : 0.0;
    };
    if constexpr (NV > 0)
        fetch(b0);
    for (int64_t i0 = b0; i0 < b1; i0 += KPP_ROWS) {
        const int m = (int)(b1 - i0 < KPP_ROWS ? b1 - i0 : KPP_ROWS);
        const int64_t i = i0 + tid;
        double acc[NT];
#pragma unroll
        for (int s = 0; s < NT; s++)
            acc[s] = 0.0;
        auto take = [&](double x, const double *__restrict__ c) {
#pragma unroll
            for (int s = 0; s < NT; s++) {
                if constexpr (SPH) {
                    acc[s] = fma(x, c[s], acc[s]);
                } else {
                    const double t = x - c[s];
                    acc[s] = fma(t, t, acc[s]);
                }
            }
        };
        double wi;
        if constexpr (NV > 0) {
            const int cnt = m * d, pieces = cnt / VE;
            __syncthreads();
#pragma unroll
            for (int v = 0; v < NV; v++) {
                const int p = v * KPP_ROWS + tid;
                if (p < pieces) {
                    // A piece never straddles a padding element: its first one is a multiple
                    // of VE elements.
                    T x[VE];
                    __builtin_memcpy(x, &pre[v], 16);
                    T *dst = tile + kpp_pos<T>(p * VE);
#pragma unroll
                    for (int u = 0; u < VE; u++)
                        dst[u] = x[u];
                }
            }
            if (pieces * VE + tid < cnt)
                tile[kpp_pos<T>(pieces * VE + tid)] = X[i0 * d + pieces * VE + tid];
            wi = wpre;
            __syncthreads();
            if (i0 + KPP_ROWS < b1)
                fetch(i0 + KPP_ROWS);
            if (tid < m) {
#pragma unroll 8
                for (int l = 0; l < d; l++)
                    take((double)tile[kpp_pos<T>(tid * d + l)], crow + (int64_t)l * NT);
            }
        } else {
            wi = (!first && tid < m) ? w[i] : 0.0;
            // The next FB features are read while these are computed: with few rows nothing else
            // hides the memory's latency (1,828 x 281 fp64, 8 workgroups: 118 -> 47 us).
            const int lc = tid % FB, lr = tid / FB;
            T next[FB];
            auto load = [&](int l0) {
#pragma unroll
                for (int u = 0; u < FB; u++) {
                    const int r = lr + u * (KPP_ROWS / FB);
                    next[u] = r < m && l0 + lc < d ? X[(i0 + r) * d + l0 + lc] : T(0);
                }
            };
            load(0);
            for (int l0 = 0; l0 < d; l0 += FB) {
                const int fl = d - l0 < FB ? d - l0 : FB;
                __syncthreads();
#pragma unroll
                for (int u = 0; u < FB; u++)
                    tile[(lr + u * (KPP_ROWS / FB)) * (FB + 1) + lc] = next[u];
                __syncthreads();
                if (l0 + FB < d)
                    load(l0 + FB);
                if (tid < m) {
#pragma unroll 8
                    for (int l = 0; l < fl; l++)
                        take((double)tile[tid * (FB + 1) + l], crow + (int64_t)(l0 + l) * NT);
                }
            }
        }
        if (tid < m) {
            if constexpr (SPH) {
                acc[0] = kpp_cosine(acc[0], g.inv, i, best);
#pragma unroll
                for (int s = 1; s < NT; s++)
                    if (s <= nt)
                        acc[s] = kpp_cosine(acc[s], g.inv, i, st->cand[par][s - 1]);
            }
            const double wn = first ? kpp_first(acc[0], i == best) : kpp_min(wi, acc[0], i == best);
            w[i] = wn;
            if (first) {
                sum[0] += wn;
            } else {
#pragma unroll
                for (int s = 1; s < NT; s++) {
                    const double v = wn < acc[s] ? wn : acc[s];
                    sum[s] += v > 0.0 ? v : 0.0;
                }
            }
        }
    }
#pragma unroll
    for (int s = 0; s < NT; s++) {
        double v = sum[s];
#pragma unroll
        for (int o = 32; o > 0; o >>= 1)
            v += __shfl_xor(v, o, 64);
        if ((tid & 63) == 0)
            red[tid >> 6][s] = v;
    }
    __syncthreads();
    if (tid < NT) {
        double v = 0.0;
#pragma unroll
        for (int q = 0; q < KPP_ROWS / 64; q++)
            v += red[q][tid];
        if (first) {
            if (tid == 0)
                part[blockIdx.x] = v;
        } else if (tid >= 1 && tid <= nt) {
            part[(int64_t)(tid - 1) * nb + blockIdx.x] = v;
        }
    }
}

// Round c. First, in every workgroup alike: centre c - 1 from the costs of its candidates
// (c = 1: the first centre, already in the weights), the scan of its block sums, one block per
// thread (nb <= 1,024). Then workgroup t finds draw t of centre c (u: its nt draws): the block,
// the first sample of the block at which the running sum of the weights reaches what is left of
// the draw (the sample after the block when rounding leaves none), and puts its row into slot
// 1 + t of crow, workgroup 0 the chosen centre's row into slot 0. c = k: only the choice.
template <typename T, bool SPH>
__global__ __launch_bounds__(1024) void kpp_draw_kernel(
    const T *__restrict__ X, int n, int d, const double *__restrict__ w,
    const double *__restrict__ part, int nb, int chunk, int nt, int c, int k,
    const double *__restrict__ u, double *__restrict__ crow, int NT, KppState *st,
    int *__restrict__ chosen, KppGeom g) {
    __shared__ double pre[1024];
    __shared__ double wsum[16], cost[KPP_TRIALS_MAX];
    __shared__ int old[KPP_TRIALS_MAX];
    __shared__ int best_s, row_s, first_t, found;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int t = blockIdx.x;
    if (c > 1 && st->same) {
        if (c == k)
            for (int j = tid; j < k; j += 1024)
                chosen[j] = j;
        return;
    }
    if (c > 1) {
        // The candidates of the previous round (the other half of cand is written below).
        if (tid < nt)
            old[tid] = st->cand[(c - 1) & 1][tid];
        for (int q = wv; q < nt; q += 16) {
            double x = 0.0;
#pragma unroll 4
            for (int b = lane; b < nb; b += 64)
                x += part[(int64_t)q * nb + b];
#pragma unroll
            for (int o = 32; o > 0; o >>= 1)
                x += __shfl_xor(x, o, 64);
            if (lane == 0)
                cost[q] = x;
        }
        __syncthreads();
        if (tid == 0) {
            // The first of the smallest finite costs among distinct candidates; row 0 when no
            // cost is finite.
            int row = 0, best = 0;
            double bc = __builtin_huge_val();
            for (int q = 0; q < nt; q++) {
                bool repeat = false;
                for (int j = 0; j < q; j++)
                    repeat |= old[j] == old[q];
                if (!repeat && cost[q] < bc) {
                    bc = cost[q];
                    best = old[q];
                    row = q;
                }
            }
            best_s = best;
            row_s = row;
        }
    } else if (tid == 0) {
        best_s = st->best;
        row_s = 0;
    }
    __syncthreads();
    const int best = best_s;
    if (t == 0 && tid == 0) {
        st->best = best;
        chosen[c - 1] = best;
    }
    if (c == k && c > 1)
        return;
    // Inclusive scan of the block sums: within waves, then over the wave totals.
    auto scan = [&](double x, double &excl) {
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const double y = __shfl_up(x, o, 64);
            if (lane >= o)
                x += y;
        }
        if (lane == 63)
            wsum[wv] = x;
        __syncthreads();
        double off = 0.0;
        for (int q = 0; q < wv; q++)
            off += wsum[q];
        x += off;
        excl = __shfl_up(x, 1, 64);
        if (lane == 0)
            excl = off;
        __syncthreads();
        return x;
    };
    double excl;
    pre[tid] = scan(tid < nb ? part[(int64_t)row_s * nb + tid] : 0.0, excl);
    __syncthreads();
    const double total = pre[nb - 1];
    if (c == 1 && !(total > 0.0)) {
        // All samples coincide with the first centre: the first k samples are taken.
        if (t == 0 && tid == 0) {
            st->same = 1;
            if (c == k)
                chosen[0] = 0;
        }
        return;
    }
    if (c == k)
        return;
    // The first block whose inclusive sum reaches u * total, and what is left of the draw there.
    // No weight left: sample 0; a total that overflowed: the last sample.
    int blk = 0;
    double rem = -1.0;
    if (total > 0.0) {
        const double target = u[t] * total;
        int lo = 0, hi = nb - 1;
        while (lo < hi) {
            const int mid = (lo + hi) / 2;
            if (pre[mid] < target)
                lo = mid + 1;
            else
                hi = mid;
        }
        blk = lo;
        rem = target - (lo > 0 ? pre[lo - 1] : 0.0);
        if (!(total < __builtin_huge_val())) {
            blk = nb - 1;
            rem = __builtin_huge_val();
        }
    }
    const int64_t b0 = (int64_t)blk * chunk;
    const int64_t b1 = b0 + chunk < n ? b0 + chunk : n;
    const int sub = (chunk + 1023) / 1024;
    const int64_t r0 = b0 + (int64_t)tid * sub, r1 = r0 + sub < b1 ? r0 + sub : b1;
    const T *cb = X + (int64_t)best * d;
    constexpr int VE = 16 / (int)sizeof(T);
    const bool vec = d % VE == 0 && (reinterpret_cast<uintptr_t>(X) & 15) == 0;
    // Weights of samples i and j (either may be the same sample), the centre chosen last taken
    // in; two rows at a time keep twice the loads in flight.
    auto weights = [&](int64_t i, int64_t j, double &wi, double &wj) {
        wi = w[i];
        wj = w[j];
        if (c == 1)
            return;
        double ai = 0.0, aj = 0.0;
        auto term = [&](double x, double y, double &a) {
            if constexpr (SPH) {
                a = fma(x, y, a);
            } else {
                const double v = x - y;
                a = fma(v, v, a);
            }
        };
        const T *x = X + i * d, *y = X + j * d;
        if (vec) {
#pragma unroll 8
            for (int l = 0; l < d; l += VE) {
                T a[VE], b[VE];
                const uint4 qa = *reinterpret_cast<const uint4 *>(x + l);
                const uint4 qb = *reinterpret_cast<const uint4 *>(y + l);
                __builtin_memcpy(a, &qa, 16);
                __builtin_memcpy(b, &qb, 16);
#pragma unroll
                for (int e = 0; e < VE; e++) {
                    term((double)a[e], (double)cb[l + e], ai);
                    term((double)b[e], (double)cb[l + e], aj);
                }
            }
        } else {
#pragma unroll 8
            for (int l = 0; l < d; l++) {
                term((double)x[l], (double)cb[l], ai);
                term((double)y[l], (double)cb[l], aj);
            }
        }
        if constexpr (SPH) {
            ai = kpp_cosine(ai, g.inv, i, best);
            aj = kpp_cosine(aj, g.inv, j, best);
        }
        wi = kpp_min(wi, ai, i == best);
        wj = kpp_min(wj, aj, j == best);
    };
    double x = 0.0;
    for (int64_t i = r0; i < r1; i += 2) {
        double wi, wj;
        weights(i, i + 1 < r1 ? i + 1 : i, wi, wj);
        x += wi;
        if (i + 1 < r1)
            x += wj;
    }
    if (tid == 0) {
        first_t = 1024;
        found = (int)(b1 < n ? b1 : n - 1);
    }
    const double incl = scan(x, excl);
    if (incl >= rem && r0 < r1)
        atomicMin(&first_t, tid);
    __syncthreads();
    if (tid == first_t) {
        double run = excl;
        int64_t hit = r1 - 1;
        for (int64_t i = r0; i < r1 - 1; i++) {
            double wi, wj;
            weights(i, i, wi, wj);
            run += wi;
            if (run >= rem) {
                hit = i;
                break;
            }
        }
        found = (int)hit;
    }
    __syncthreads();
    const int pick = found;
    if (tid == 0)
        st->cand[c & 1][t] = pick;
    for (int l = tid; l < d; l += 1024) {
        crow[(int64_t)l * NT + 1 + t] = (double)X[(int64_t)pick * d + l];
        if (t == 0)
            crow[(int64_t)l * NT] = (double)cb[l];
    }
}

template <typename T>
__global__ void kpp_begin_kernel(const T *__restrict__ X, int d, int first,
                                 double *__restrict__ crow, int NT, KppState *__restrict__ st) {
    for (int64_t e = threadIdx.x; e < (int64_t)d * NT; e += blockDim.x)
        crow[e] = e % NT == 0 ? (double)X[(int64_t)first * d + e / NT] : 0.0;
    if (threadIdx.x == 0) {
        st->best = first;
        st->same = 0;
    }
    if (threadIdx.x < KPP_TRIALS_MAX) {
        st->cand[0][threadIdx.x] = first;
        st->cand[1][threadIdx.x] = first;
    }
}

template <typename T, int NT, int NV>
hipError_t kpp_cost_nv(const T *X, int n, int d, double *w, const double *crow,
                       const KppState *st, int par, int nt, const KppPlan &p, double *part,
                       int first, hipStream_t s, int sph, const double *inv) {
    constexpr int FB = 128 / (int)sizeof(T);
    const size_t lds = NV > 0
                           ? ((size_t)KPP_ROWS * d + (size_t)KPP_ROWS * d / FB + 1) * sizeof(T)
                           : (size_t)KPP_ROWS * (FB + 1) * sizeof(T);
    auto kern = sph ? kpp_cost_kernel<T, NT, NV, true> : kpp_cost_kernel<T, NT, NV, false>;
    if (lds > 65536)
        (void)hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                                  (int)lds);
    hipLaunchKernelGGL(kern, dim3(p.nb), dim3(KPP_ROWS), lds, s, X, n, d, w, crow, st, par, nt,
                       p.chunk, part, p.nb, first, KppGeom{inv});
    return hipGetLastError();
}

// Rows of up to 256 bytes are staged whole (at most 68 KB of LDS, two workgroups per CU).
template <typename T, int NT>
hipError_t kpp_cost_nt(const T *X, int n, int d, double *w, const double *crow,
                       const KppState *st, int par, int nt, const KppPlan &p, double *part,
                       int first, hipStream_t s, int sph, const double *inv) {
    const size_t row = d * sizeof(T);
    const bool aligned = (reinterpret_cast<uintptr_t>(X) & 15) == 0;
#define DA_KPP_NV(NVV)                                                                           \
    return kpp_cost_nv<T, NT, NVV>(X, n, d, w, crow, st, par, nt, p, part, first, s, sph, inv)
    if (aligned && row <= 64)
        DA_KPP_NV(4);
    if (aligned && row <= 128)
        DA_KPP_NV(8);
    if (aligned && row <= 256)
        DA_KPP_NV(16);
    DA_KPP_NV(0);
#undef DA_KPP_NV
}

} // namespace

// Chunks of whole 256-row steps, at most 1,024 of them (kpp_draw scans them in one workgroup,
// and about four workgroups of the cost pass run on each of the 256 CUs at once, so one round of
// workgroups covers them). Slots: the chosen centre and nt candidates, padded to a kernel width.
KppPlan kpp_plan(int n, int nt) {
    KppPlan p;
    const int64_t rows = ((int64_t)n + 1023) / 1024;
    p.chunk = (int)((rows + KPP_ROWS - 1) / KPP_ROWS * KPP_ROWS);
    p.nb = (int)(((int64_t)n + p.chunk - 1) / p.chunk);
    p.slots = nt + 1 <= 4 ? 4 : nt + 1 <= 8 ? 8 : nt + 1 <= 16 ? 16 : 24;
    return p;
}

template <typename T>
hipError_t launch_kpp_begin(const T *X, int d, int first, double *crow, const KppPlan &p,
                            KppState *st, hipStream_t s) {
    hipLaunchKernelGGL(kpp_begin_kernel<T>, dim3(1), dim3(256), 0, s, X, d, first, crow, p.slots,
                       st);
    return hipGetLastError();
}

template <typename T>
hipError_t launch_kpp_cost(const T *X, int n, int d, double *w, const double *crow,
                           const KppState *st, int c, int nt, const KppPlan &p, double *part,
                           hipStream_t s, int sph, const double *inv) {
    if (n < 1 || d < 1 || nt < 0 || nt > KPP_TRIALS_MAX || nt + 1 > p.slots)
        return hipErrorInvalidValue;
    const int first = c == 0, par = c & 1;
    switch (p.slots) {
    case 4:
        return kpp_cost_nt<T, 4>(X, n, d, w, crow, st, par, nt, p, part, first, s, sph, inv);
    case 8:
        return kpp_cost_nt<T, 8>(X, n, d, w, crow, st, par, nt, p, part, first, s, sph, inv);
    case 16:
        return kpp_cost_nt<T, 16>(X, n, d, w, crow, st, par, nt, p, part, first, s, sph, inv);
    default:
        return kpp_cost_nt<T, 24>(X, n, d, w, crow, st, par, nt, p, part, first, s, sph, inv);
    }
}

template <typename T>
hipError_t launch_kpp_draw(const T *X, int n, int d, const double *w, const double *part, int nt,
                           int c, int k, const double *u, double *crow, const KppPlan &p,
                           KppState *st, int *chosen, hipStream_t s, int sph, const double *inv) {
    if (nt < 1 || nt > KPP_TRIALS_MAX || p.nb < 1 || p.nb > 1024)
        return hipErrorInvalidValue;
    auto kern = sph ? kpp_draw_kernel<T, true> : kpp_draw_kernel<T, false>;
    hipLaunchKernelGGL(kern, dim3(c < k ? nt : 1), dim3(1024), 0, s, X, n, d, w, part, p.nb,
                       p.chunk, nt, c, k, u, crow, p.slots, st, chosen, KppGeom{inv});
    return hipGetLastError();
}

#define DA_KPP_INST(T)                                                                           \
    template hipError_t launch_kpp_begin<T>(const T *, int, int, double *, const KppPlan &,     \
                                            KppState *, hipStream_t);                           \
    template hipError_t launch_kpp_cost<T>(const T *, int, int, double *, const double *,       \
                                           const KppState *, int, int, const KppPlan &,         \
                                           double *, hipStream_t, int, const double *);         \
    template hipError_t launch_kpp_draw<T>(const T *, int, int, const double *, const double *, \
                                           int, int, int, const double *, double *,             \
                                           const KppPlan &, KppState *, int *, hipStream_t, int, \
                                           const double *);
DA_KPP_INST(float)
DA_KPP_INST(double)
#undef DA_KPP_INST

} // namespace dagpu
