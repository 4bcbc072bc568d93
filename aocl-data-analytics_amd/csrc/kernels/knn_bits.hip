// k-nearest neighbours by hit bits on the fp16 matrix cores of gfx950, for the squared-euclidean
// metrics and rows of up to 128 features.
//
// A fused tile forms every key to the operand precision it certifies with and keeps the best of
// every split in lists, whose upkeep costs more than the products (100,003 x 100 fp32, 10,007
// queries, k = 20: 3.1 ms for 0.2 TFLOP). Here nothing is kept on the way:
//   1. scores against a sample of the rows give each query a threshold lim that a few times k rows
//      are expected to lie within. It is a guess: nothing depends on it but the work.
//   2. the sweep multiplies the rows' fp16 parts (one product, |x'||y'| 2^-10 of error) and leaves
//      one bit per pair: cleared only if |x' - y'|^2 > lim beyond the error bound. So every row
//      within lim is a hit; the error only adds hits.
//   3. the merge forms the exact keys of the hits (double, features in order, as the other paths
//      do). If k of them are within lim, the k smallest (key, row) are the neighbours.
// Queries with fewer than k rows within lim, more than BITS_KEEP hits or values beyond fp16's range
// are listed for the fused tile. When the error bound is wide against the distances (tight clusters
// far apart), the sample shows it: such queries are counted, and if they are more than a quarter the
// sweep does not run at all. (Sample and second search still cost 0.2 of 0.8 ms at 16,384 x 20 with
// 6,000 queries, so after a search that listed most of its queries the caller leaves some to the tile.)
//
// Bound: rows are centred and scaled by a power of two (knn_wide.hip); hi = x' (1 + 2^-11), so
// |hi.hi - x'.y'| <= 2^-10 (1 + 2^-11) |x'||y'|; the sum of Kp products from a start value of at most
// 1.5 (|x'|^2 + |y'|^2) where the outcome is open (lim <= 2 (|x'|^2 + |y'|^2) there) gamma_{Kp + 8}
// of 2 (|x'|^2 + |y'|^2), the rounded thresholds a few 2^-24. Together ce (|x'|^2 + |y'|^2) / 2, plus
// 2 alpha sqrt(d) (|x'| + max |y'|) for elements below fp16's normal range and the centring.
#include "launch.hpp"
#include "wave_rank.hpp"
#include <algorithm>
#include <cmath>
#include <hip/hip_runtime.h>

namespace dagpu {

namespace {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));

// One wave per query: the rank-th smallest of its 256 minima (at least the rank-th smallest score,
// and with rank well below 256 close to it).
__global__ __launch_bounds__(256) void bits_guess_kernel(
    const float *__restrict__ mins, int nq, int most_within, int d, int rank, double ce,
    const double *__restrict__ nrm, const WideScale *__restrict__ sc, float *__restrict__ A,
    double *__restrict__ lim, int *bad, int *__restrict__ count) {
    const int q = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    const double nn = nrm[q];
    if (lane == 0)
        count[q] = 0;
    if (q >= nq || !(nn < __builtin_huge_val())) {
        if (lane == 0) {
            A[q] = __builtin_huge_valf(); // no hits
            lim[q] = -1.0;
            if (q < nq)
                atomicAdd(bad, 1);
        }
        return;
    }
    const float4 m4 = reinterpret_cast<const float4 *>(mins + (int64_t)q * 256)[lane];
    const float m[4] = {m4.x, m4.y, m4.z, m4.w};
    const float pick = wave_rank_256(m, rank);
    // The sample's own rounding is covered, so that copies of a query pass.
    const double L = fmax(2.0 * (double)pick + nn * (1.0 + 0x1p-14), 0.0);
    int within = 0;
#pragma unroll
    for (int u = 0; u < 4; u++)
        within += __popcll(__builtin_amdgcn_ballot_w64((double)m[u] <= 0.5 * (L - nn) + ce * nn));
    if (lane == 0) {
        const bool hopeless = within > most_within;
        const double s = sc->scale, y2 = __longlong_as_double((long long)sc->ymax2);
        // A query that fits stays within 60,000 / s of the centre.
        const double alpha = 0x1p-24 + 0x1p-51 * (60000.0 + 2.0 * s * sc->big);
        const double ca = 2.0 * alpha * sqrt((double)d) * (sqrt(nn) + sqrt(y2));
        const double a = -(0.5 * (L - nn) + 0.5 * ce * nn + ca);
        A[q] = hopeless ? __builtin_huge_valf() : (float)(a - fabs(a) * 0x1p-22);
        lim[q] = hopeless ? -1.0 : L;
        if (hopeless)
            atomicAdd(bad, 1);
    }
}

constexpr int CTS = 4;

// Sample: the sweep below with a running maximum of -score per lane and row in place of the bits.
// Segment s, lane column r of a row make group 16 s + r. RT = 1 where RT = 4 would leave most CUs
// without a workgroup (1,024 queries, 65,536 sample rows of 96: 125 us in 64 workgroups).
template <int KS, int RT>
__global__ __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(2))) void bits_sample_kernel(
    const _Float16 *__restrict__ PA, const _Float16 *__restrict__ PB,
    const float *__restrict__ h, int cols, float *__restrict__ mins) {
    __shared__ __attribute__((aligned(16))) _Float16 sb[CTS * KS * 512];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int r = lane & 15, g = lane >> 4;
    const int seg = blockIdx.x & 15, row0 = ((int)(blockIdx.x >> 4) * 4 + w) * RT * 16;
    v8h a[RT][KS];
    v4f best[RT];
#pragma unroll
    for (int rt = 0; rt < RT; rt++) {
        const _Float16 *src = PA + (int64_t)(row0 / 16 + rt) * KS * 512 + lane * 8;
#pragma unroll
        for (int ks = 0; ks < KS; ks++)
            a[rt][ks] = *reinterpret_cast<const v8h *>(src + ks * 512);
#pragma unroll
        for (int i = 0; i < 4; i++)
            best[rt][i] = -__builtin_huge_valf();
    }
    for (int j0 = seg * cols; j0 < (seg + 1) * cols; j0 += 16 * CTS) {
        const _Float16 *src = PB + (int64_t)(j0 / 16) * KS * 512;
        v8h f[KS];
#pragma unroll
        for (int b = 0; b < KS; b++)
            f[b] = *reinterpret_cast<const v8h *>(src + (w * KS + b) * 512 + lane * 8);
        __syncthreads();
#pragma unroll
        for (int b = 0; b < KS; b++)
            *reinterpret_cast<v8h *>(sb + (w * KS + b) * 512 + lane * 8) = f[b];
        __syncthreads();
#pragma unroll
        for (int ct = 0; ct < CTS; ct++) {
            const float hv = -h[j0 + ct * 16 + r];
            v4f acc[RT];
#pragma unroll
            for (int rt = 0; rt < RT; rt++)
                acc[rt] = v4f{hv, hv, hv, hv};
#pragma unroll
            for (int ks = 0; ks < KS; ks++) {
                const v8h b = *reinterpret_cast<const v8h *>(sb + (ct * KS + ks) * 512 + lane * 8);
#pragma unroll
                for (int rt = 0; rt < RT; rt++)
                    acc[rt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[rt][ks], b, acc[rt], 0, 0, 0);
            }
#pragma unroll
            for (int rt = 0; rt < RT; rt++)
#pragma unroll
                for (int i = 0; i < 4; i++)
                    best[rt][i] = fmaxf(best[rt][i], acc[rt][i]);
        }
    }
#pragma unroll
    for (int rt = 0; rt < RT; rt++)
#pragma unroll
        for (int i = 0; i < 4; i++)
            mins[(int64_t)(row0 + rt * 16 + 4 * g + i) * 256 + seg * 16 + r] = -best[rt][i];
}

// The sweep, as that of radius_mfma.hip with one product for 32 features: a wave holds four tiles
// of 16 query rows in registers, training tiles pass through LDS four at a time, accumulators start
// at -A_x - B_y and their sign is shifted into the lane's word of the row. Bound by the matrix
// cores together with the two vector operations per pair. Bit order: word [row][j / 512][j % 16]
// holds column j at bit 31 - (j % 512) / 16.
constexpr int RT = 4;

template <int KS>
__global__ __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(2))) void bits_sweep_kernel(
    const _Float16 *__restrict__ PA, const _Float16 *__restrict__ PB,
    const float *__restrict__ A, const float *__restrict__ B, int nrb, int nblk, int segblk,
    const int *__restrict__ bad, int most_bad, unsigned *__restrict__ bits) {
    constexpr int STAGE = CTS * KS * 512; // fp16 elements of 16 CTS training rows
    __shared__ __attribute__((aligned(16))) _Float16 s0[STAGE];
    __shared__ __attribute__((aligned(16))) _Float16 s1[STAGE];
    if (*bad > most_bad)
        return;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int r = lane & 15, g = lane >> 4;
    // All row blocks of one segment first, so that the workgroups running at a time share it.
    const int segi = (int)blockIdx.x / nrb, rb = (int)blockIdx.x - segi * nrb;
    const int row0 = (rb * 4 + w) * RT * 16;
    const int b0 = segi * segblk, b1 = min(nblk, b0 + segblk);
    if (b0 >= b1)
        return;
    v8h a[RT][KS];
    float ax[RT][4];
    unsigned word[RT][4];
#pragma unroll
    for (int rt = 0; rt < RT; rt++) {
        const _Float16 *src = PA + (int64_t)(row0 / 16 + rt) * KS * 512 + lane * 8;
#pragma unroll
        for (int ks = 0; ks < KS; ks++)
            a[rt][ks] = *reinterpret_cast<const v8h *>(src + ks * 512);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            ax[rt][i] = A[row0 + rt * 16 + 4 * g + i];
            word[rt][i] = 0;
        }
    }
    float hv[CTS];
    auto stage = [&](int j0, _Float16 *dst) {
        const _Float16 *src = PB + (int64_t)(j0 / 16) * KS * 512;
#pragma unroll
        for (int b = 0; b < KS; b++) {
            const int blk = w * KS + b;
            __builtin_amdgcn_global_load_lds(
                (const __attribute__((address_space(1))) void *)(src + blk * 512 + lane * 8),
                (__attribute__((address_space(3))) void *)(dst + blk * 512), 16, 0, 0);
        }
#pragma unroll
        for (int ct = 0; ct < CTS; ct++)
            hv[ct] = B[j0 + ct * 16 + r];
    };
    auto compute = [&](const _Float16 *sb, const float (&bv)[CTS]) {
#pragma unroll
        for (int ct = 0; ct < CTS; ct++) {
            v4f acc[RT];
#pragma unroll
            for (int rt = 0; rt < RT; rt++)
#pragma unroll
                for (int i = 0; i < 4; i++)
                    acc[rt][i] = -bv[ct] - ax[rt][i];
#pragma unroll
            for (int ks = 0; ks < KS; ks++) {
                const v8h b = *reinterpret_cast<const v8h *>(sb + (ct * KS + ks) * 512 + lane * 8);
#pragma unroll
                for (int rt = 0; rt < RT; rt++)
                    acc[rt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[rt][ks], b, acc[rt], 0, 0, 0);
            }
#pragma unroll
            for (int rt = 0; rt < RT; rt++)
#pragma unroll
                for (int i = 0; i < 4; i++)
                    word[rt][i] = __builtin_amdgcn_alignbit(word[rt][i],
                                                            __float_as_uint(acc[rt][i]), 31);
        }
    };
    const int j1 = b1 * 512;
    stage(b0 * 512, s0);
    for (int blk = b0; blk < b1; blk++) {
        constexpr int ST = 16 * CTS;
        for (int j0 = blk * 512; j0 < blk * 512 + 512; j0 += 2 * ST) {
            // Rows j0 from s0, the next ST into s1; then the other way round.
            __builtin_amdgcn_s_waitcnt(0x0F70); // vmcnt(0): this wave's copies have landed
            __syncthreads();
            float bv[CTS];
#pragma unroll
            for (int ct = 0; ct < CTS; ct++)
                bv[ct] = hv[ct];
            stage(j0 + ST, s1);
            compute(s0, bv);
            __builtin_amdgcn_s_waitcnt(0x0F70);
            __syncthreads();
#pragma unroll
            for (int ct = 0; ct < CTS; ct++)
                bv[ct] = hv[ct];
            if (j0 + 2 * ST < j1)
                stage(j0 + 2 * ST, s0);
            compute(s1, bv);
        }
        // 32 sign bits per row and lane: set means miss.
#pragma unroll
        for (int rt = 0; rt < RT; rt++)
#pragma unroll
            for (int i = 0; i < 4; i++)
                bits[((int64_t)(row0 + rt * 16 + 4 * g + i) * nblk + blk) * 16 + r] = ~word[rt][i];
    }
}

// Set bits -> columns. A wave takes 1,024 words of a query's row (32,768 columns) in four loads a
// lane, adds up its set bits and appends their columns with one atomic. (Inside the merge, where a
// workgroup walked its row alone, the merge of 1,024 rows of 2,000,000 columns took 0.48 ms.)
__global__ __launch_bounds__(256) void bits_columns_kernel(const unsigned *__restrict__ bits, int nq,
                                                           int nvec, int parts,
                                                           const int *__restrict__ bad,
                                                           int most_bad, int *count,
                                                           int *__restrict__ cols) {
    if (*bad > most_bad)
        return;
    const int64_t wave = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const int64_t q = wave / parts;
    if (q >= nq)
        return;
    const int v0 = (int)(wave - q * parts) * 256;
    const uint4 *b = reinterpret_cast<const uint4 *>(bits) + q * nvec;
    uint4 v[4];
    int n = 0;
#pragma unroll
    for (int u = 0; u < 4; u++) {
        const int i = v0 + u * 64 + lane;
        v[u] = i < nvec ? b[i] : make_uint4(0, 0, 0, 0);
    }
#pragma unroll
    for (int u = 0; u < 4; u++)
        n += __popc(v[u].x) + __popc(v[u].y) + __popc(v[u].z) + __popc(v[u].w);
    int at = n;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int x = __shfl_up(at, o, 64);
        at += lane >= o ? x : 0;
    }
    const int all = __shfl(at, 63, 64);
    if (all == 0)
        return;
    int base = 0;
    if (lane == 0)
        base = atomicAdd(&count[q], all);
    at += __shfl(base, 0, 64) - n;
    if (n == 0)
        return;
    int *out = cols + q * BITS_KEEP;
    auto take = [&](unsigned x, int word) {
        while (x) {
            const int bit = __ffs(x) - 1;
            x &= x - 1;
            if (at < BITS_KEEP)
                out[at] = (word >> 4) * 512 + (31 - bit) * 16 + (word & 15);
            at++;
        }
    };
#pragma unroll
    for (int u = 0; u < 4; u++) {
        const int word = (v0 + u * 64 + lane) * 4;
        take(v[u].x, word);
        take(v[u].y, word + 1);
        take(v[u].z, word + 2);
        take(v[u].w, word + 3);
    }
}

// One workgroup per query: exact keys of the hits, one thread a hit. Bound by the latency of the
// row reads: a row of whole 16-byte pieces is read by four lanes, 64 bytes at a time, 256 bytes
// in flight, and reaches its thread through LDS (one lane per row touches 64 lines with every load).
// Keys within lim are kept, a histogram over [0, lim] finds the bin of the k-th, and only the keys
// up to that bin are ranked by counting.
constexpr int BITS_INSIDE = 1024;

template <typename T>
__global__ __launch_bounds__(256) void bits_merge_kernel(
    const int *__restrict__ count, const int *__restrict__ cols, const int *__restrict__ bad,
    int most_bad, const T *__restrict__ Q, const T *__restrict__ Y, int d, int k,
    const double *__restrict__ lim, const WideScale *__restrict__ sc, int post, int q0,
    T *__restrict__ out_dist, int *__restrict__ out_idx, int *__restrict__ fb_count,
    int *__restrict__ fb_list) {
    __shared__ double qrow[BITS_D];
    __shared__ int xi[BITS_INSIDE];
    __shared__ double xk[BITS_INSIDE];
    __shared__ v4u piece[4][64][5]; // a row's 64 bytes, padded against bank conflicts
    __shared__ __attribute__((aligned(16))) int hist[256];
    __shared__ int inside, near;
    const int q = blockIdx.x, t = threadIdx.x;
    const double L = lim[q];
    const int nh = count[q];
    if (*bad > most_bad || L < 0.0 || nh > BITS_KEEP || nh < k) {
        if (t == 0)
            fb_list[atomicAdd(fb_count, 1)] = q0 + q;
        return;
    }
    if (t == 0)
        inside = near = 0;
    hist[t] = 0;
    if (t < d)
        qrow[t] = (double)Q[(int64_t)q * d + t];
    __syncthreads();
    // The rounding of the exact keys leaves a margin far above it.
    const double s = sc->scale, top = L * (1.0 - 1e-10) / s / s;
    const double bins = 255.0 / top; // infinite or not a number for top 0: every key is 0
    constexpr int VE = 16 / (int)sizeof(T);
    const bool vec = d % VE == 0;
    const int lane = t & 63, w = t >> 6, np = d / VE;
    const int *col = cols + (int64_t)q * BITS_KEEP;
    for (int c0 = w * 64; c0 < nh; c0 += 256) {
        const int c = c0 + lane;
        const int j = col[min(c, nh - 1)];
        double acc = 0.0;
        if (vec) {
            const v4u *s0 = reinterpret_cast<const v4u *>(Y + (int64_t)__shfl(j, lane >> 2, 64) * d);
            const v4u *s1 =
                reinterpret_cast<const v4u *>(Y + (int64_t)__shfl(j, 16 + (lane >> 2), 64) * d);
            const v4u *s2 =
                reinterpret_cast<const v4u *>(Y + (int64_t)__shfl(j, 32 + (lane >> 2), 64) * d);
            const v4u *s3 =
                reinterpret_cast<const v4u *>(Y + (int64_t)__shfl(j, 48 + (lane >> 2), 64) * d);
            // One 64-byte step: from four registers through LDS to the rows' lanes.
            auto step = [&](int p0, v4u x0, v4u x1, v4u x2, v4u x3) {
                if (p0 >= np)
                    return;
                __builtin_amdgcn_wave_barrier();
                piece[w][lane >> 2][lane & 3] = x0;
                piece[w][16 + (lane >> 2)][lane & 3] = x1;
                piece[w][32 + (lane >> 2)][lane & 3] = x2;
                piece[w][48 + (lane >> 2)][lane & 3] = x3;
                __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
                __builtin_amdgcn_wave_barrier();
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    if (p0 + e < np) {
                        const v4u x = piece[w][lane][e];
                        T v[VE];
                        __builtin_memcpy(v, &x, 16);
#pragma unroll
                        for (int i = 0; i < VE; i++) {
                            const double dv = qrow[(p0 + e) * VE + i] - (double)v[i];
                            acc = fma(dv, dv, acc);
                        }
                    }
                }
                __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            };
            for (int pb = 0; pb < np; pb += 16) {
                const int l = lane & 3;
                const int a = min(pb + l, np - 1), b = min(pb + 4 + l, np - 1);
                const int c2 = min(pb + 8 + l, np - 1), e2 = min(pb + 12 + l, np - 1);
                const v4u a0 = s0[a], a1 = s1[a], a2 = s2[a], a3 = s3[a];
                const v4u b0 = s0[b], b1 = s1[b], b2 = s2[b], b3 = s3[b];
                const v4u x0 = s0[c2], x1 = s1[c2], x2 = s2[c2], x3 = s3[c2];
                const v4u y0 = s0[e2], y1 = s1[e2], y2 = s2[e2], y3 = s3[e2];
                step(pb, a0, a1, a2, a3);
                step(pb + 4, b0, b1, b2, b3);
                step(pb + 8, x0, x1, x2, x3);
                step(pb + 12, y0, y1, y2, y3);
            }
        } else {
            const T *y = Y + (int64_t)j * d;
#pragma unroll 8
            for (int l = 0; l < d; l++) {
                const double dv = qrow[l] - (double)y[l];
                acc = fma(dv, dv, acc);
            }
        }
        if (c < nh && acc <= top) {
            const int at = atomicAdd(&inside, 1);
            if (at < BITS_INSIDE) {
                xk[at] = acc;
                xi[at] = j;
            }
            atomicAdd(&hist[min(255, (int)(acc * bins))], 1);
        }
    }
    __syncthreads();
    const int m = inside;
    if (m < k || m > BITS_INSIDE) {
        if (t == 0)
            fb_list[atomicAdd(fb_count, 1)] = q0 + q;
        return;
    }
    // First bin whose running count reaches k.
    int last = 0;
    {
        const int4 h = reinterpret_cast<const int4 *>(hist)[lane];
        int sum = h.x + h.y + h.z + h.w, run = sum;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int x = __shfl_up(run, o, 64);
            run += lane >= o ? x : 0;
        }
        const unsigned long long full = __builtin_amdgcn_ballot_w64(run >= k);
        const int at = __ffsll((long long)full) - 1;
        int before = run - sum;
        int bin = 4 * lane;
        if ((before += h.x) < k) {
            bin++;
            if ((before += h.y) < k) {
                bin++;
                if ((before += h.z) < k)
                    bin++;
            }
        }
        last = __shfl(bin, at, 64);
    }
    // Keys up to that bin into the rows' buffer (free by now).
    __syncthreads();
    double *nk = reinterpret_cast<double *>(piece);
    int *ni = reinterpret_cast<int *>(nk + BITS_INSIDE);
    static_assert(sizeof(piece) >= BITS_INSIDE * 12, "ranked keys fit the row buffer");
    for (int c = t; c < m; c += 256)
        if (min(255, (int)(xk[c] * bins)) <= last) {
            const int at = atomicAdd(&near, 1);
            nk[at] = xk[c];
            ni[at] = xi[c];
        }
    __syncthreads();
    const int mk = near;
    for (int c = t; c < mk; c += 256) {
        const double v = nk[c];
        const int j = ni[c];
        int rank = 0;
#pragma unroll 4
        for (int o = 0; o < mk; o++)
            rank += nk[o] < v || (nk[o] == v && ni[o] < j);
        if (rank < k) {
            if (out_dist)
                out_dist[(int64_t)q * k + rank] = (T)(post == 1 ? sqrt(v) : v);
            out_idx[(int64_t)q * k + rank] = j;
        }
    }
}

} // namespace

double bits_relative_bound(int d) {
    const double terms = 32.0 * wide_ksteps(d) + 24, u = 0x1p-24;
    return 0x1p-10 * (1.0 + 0x1p-10) + 4.4 * terms * u / (1.0 - terms * u);
}

// A row is in the sample with probability p = ns / n, so of the k nearest about k p are, give or
// take sqrt(k p); a query falls short of k if as many as the rank are. Four deviations and three
// leave under one in 10^5 (three: one in 10^3 at k = 100, ns / n = 1 / 30, so that every other batch of
// 1,024 queries paid 0.25 ms for one of them).
int bits_rank(int k, int64_t n, int ns) {
    const double e = (double)k * ns / (double)n;
    return std::min(200, (int)std::ceil(e + 4.0 * std::sqrt(e)) + 3);
}

hipError_t launch_bits_sample(const void *PA, int nq, const void *PS, const float *hS, int ns, int d,
                              float *mins, hipStream_t s) {
    if (ns < BITS_SAMPLE || ns % BITS_SAMPLE != 0)
        return hipErrorInvalidValue;
    const bool wide = (nq + 255) / 256 * 16 >= 512;
    const dim3 grid((unsigned)(wide ? (nq + 255) / 256 * 16 : (nq + 63) / 64 * 16));
    const _Float16 *pa = static_cast<const _Float16 *>(PA), *pb = static_cast<const _Float16 *>(PS);
    auto run = [&](auto kern) {
        hipLaunchKernelGGL(kern, grid, dim3(256), 0, s, pa, pb, hS, ns / 16, mins);
        return hipGetLastError();
    };
    switch (wide_ksteps(d)) {
    case 1: return wide ? run(bits_sample_kernel<1, 4>) : run(bits_sample_kernel<1, 1>);
    case 2: return wide ? run(bits_sample_kernel<2, 4>) : run(bits_sample_kernel<2, 1>);
    case 3: return wide ? run(bits_sample_kernel<3, 4>) : run(bits_sample_kernel<3, 1>);
    case 4: return wide ? run(bits_sample_kernel<4, 4>) : run(bits_sample_kernel<4, 1>);
    }
    return hipErrorInvalidValue;
}

hipError_t launch_bits_guess(const float *mins, int nq, int ns, int64_t n, int d, int rank,
                             double ce, const double *nrm, const WideScale *sc, float *A,
                             double *lim, int *bad, int *count, hipStream_t s) {
    if (rank < 1 || rank > 256)
        return hipErrorInvalidValue;
    // Hits to expect: with a share f of the rows hit, a group of g sample rows holds none with
    // probability (1 - f)^g. (The number of groups with one, times the rows a group stands for, ends
    // at 256 groups, too few to tell below 24,577 rows.)
    const double f = 0.75 * BITS_KEEP / (double)n;
    const int most_within = (int)(256.0 * (1.0 - std::pow(1.0 - f, ns / 256.0)));
    hipLaunchKernelGGL(bits_guess_kernel, dim3((nq + 255) / 256 * 64), dim3(256), 0, s, mins, nq,
                       most_within, d, rank, ce, nrm, sc, A, lim, bad, count);
    return hipGetLastError();
}

hipError_t launch_bits_columns(const unsigned *bits, int nq, int n, const int *bad, int *count,
                               int *cols, hipStream_t s) {
    const int nvec = bits_rows(n) / 128, parts = (nvec + 255) / 256;
    hipLaunchKernelGGL(bits_columns_kernel, dim3((unsigned)(((int64_t)nq * parts + 3) / 4)),
                       dim3(256), 0, s, bits, nq, nvec, parts, bad, nq / 4, count, cols);
    return hipGetLastError();
}

hipError_t launch_bits_sweep(const void *PA, int nq, const void *P, int n, int d, const float *A,
                             const float *B, const int *bad, unsigned *bits, hipStream_t s) {
    const int nblk = bits_rows(n) / 512, nrb = (nq + 255) / 256;
    // About 1,024 workgroups (two per CU at a time), whole segments.
    const int want = std::max(1, std::min(nblk, (1024 + nrb - 1) / nrb));
    const int segblk = (nblk + want - 1) / want, nseg = (nblk + segblk - 1) / segblk;
    const dim3 grid((unsigned)nrb * nseg);
    const _Float16 *pa = static_cast<const _Float16 *>(PA), *pb = static_cast<const _Float16 *>(P);
    auto run = [&](auto kern) {
        hipLaunchKernelGGL(kern, grid, dim3(256), 0, s, pa, pb, A, B, nrb, nblk, segblk, bad, nq / 4,
                           bits);
        return hipGetLastError();
    };
    switch (wide_ksteps(d)) {
    case 1: return run(bits_sweep_kernel<1>);
    case 2: return run(bits_sweep_kernel<2>);
    case 3: return run(bits_sweep_kernel<3>);
    case 4: return run(bits_sweep_kernel<4>);
    }
    return hipErrorInvalidValue;
}

template <typename T>
hipError_t launch_bits_merge(const int *count, const int *cols, int nq, const int *bad, const T *Q,
                             const T *Y, int d, int k, const double *lim, const WideScale *sc,
                             int post, int q0, T *out_dist, int *out_idx, int *fb_count,
                             int *fb_list, hipStream_t s) {
    if (d > BITS_D || k > BITS_K || nq < 1)
        return hipErrorInvalidValue;
    hipLaunchKernelGGL(bits_merge_kernel<T>, dim3(nq), dim3(256), 0, s, count, cols, bad, nq / 4, Q,
                       Y, d, k, lim, sc, post, q0, out_dist, out_idx, fb_count, fb_list);
    return hipGetLastError();
}

#define DA_BITS_INST(T)                                                                          \
    template hipError_t launch_bits_merge<T>(const int *, const int *, int, const int *,         \
                                             const T *, const T *, int, int, const double *,     \
                                             const WideScale *, int, int, T *, int *, int *,     \
                                             int *, hipStream_t);
DA_BITS_INST(float)
DA_BITS_INST(double)
#undef DA_BITS_INST

} // namespace dagpu
