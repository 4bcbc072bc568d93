// k-nearest neighbours of rows too wide for the fused tile, and of the cosine metric, on the fp16
// matrix cores of gfx950.
//
// The general path forms every key with 3 d double operations. Here the keys are first formed
// approximately from rows held as hi + lo in fp16 (hi*hi + hi*lo + lo*hi on
// v_mfma_f32_16x16x32_f16, about 22 significant bits), the best of each query are selected with
// a margin, and only those get their exact key (double, features in order, as the general path
// forms it). A query is certified when every row left out has an approximate key above the k-th
// one by more than twice the error bound; the others are listed and searched exactly, so the
// result is that of the general path in every case.
//
// Euclidean: rows are centred on the middle of the training columns' ranges and scaled by a power
// of two to fp16's range; score v = |y'|^2/2 - x'.y' = (|x' - y'|^2 - |x'|^2) / 2. Cosine: rows
// are divided by their norms (the general path's, 1 for a zero row), v = -x'.y'.
//
// Error bound of a score: the products are summed in blocks of 256 features, whose sums are added
// up separately, so a block of 3 x 256 products carries gamma_{3*256+16} and the few block sums
// a few 2^-24; the split operands carry 2^-21 each, the dropped lo*lo 2^-22; |x'||y'| <=
// (|x'|^2 + |y'|^2) / 2. With ce = 1.05 gamma + 2^-18 and alpha the absolute error of an element
// (fp16 values below the normal range, the rounding of the centring):
//     E = ce (|x'|^2 + max |y'|^2) / 2 + 2 alpha sqrt(d) (|x'| + max |y'|).
#include "launch.hpp"
#include <algorithm>
#include <climits>
#include <cmath>
#include <limits>
#include <hip/hip_runtime.h>

namespace dagpu {

namespace {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));

__device__ __forceinline__ unsigned long long wide_order(double v) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    return (b >> 63) ? ~b : (b | 0x8000000000000000ull);
}
__device__ __forceinline__ double wide_value(unsigned long long k) {
    return __longlong_as_double((long long)((k >> 63) ? (k & 0x7FFFFFFFFFFFFFFFull) : ~k));
}

__global__ void wide_range_init_kernel(unsigned long long *range, int d, WideScale *sc) {
    for (int l = blockIdx.x * blockDim.x + threadIdx.x; l < d; l += gridDim.x * blockDim.x) {
        range[2 * l] = ~0ull;
        range[2 * l + 1] = 0ull;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        sc->bad = 0;
        sc->ymax2 = 0ull;
    }
}

// Column ranges: 64 columns per workgroup, its four waves taking every fourth row of a block.
template <typename T>
__global__ __launch_bounds__(256) void wide_range_kernel(const T *__restrict__ X, int rows, int d,
                                                         unsigned long long *range,
                                                         WideScale *sc) {
    __shared__ double lo[4][64], hi[4][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int l = blockIdx.x * 64 + lane;
    double mn = __builtin_huge_val(), mx = -__builtin_huge_val();
    bool nf = false;
    if (l < d) {
#pragma unroll 4
        for (int64_t i = (int64_t)blockIdx.y * 4 + w; i < rows; i += (int64_t)gridDim.y * 4) {
            const double v = (double)X[i * d + l];
            nf |= !(v - v == 0.0);
            mn = fmin(mn, v);
            mx = fmax(mx, v);
        }
    }
    lo[w][lane] = mn;
    hi[w][lane] = mx;
    if (__builtin_amdgcn_ballot_w64(nf) && lane == 0)
        atomicOr(&sc->bad, 1);
    __syncthreads();
    if (w == 0 && l < d) {
        for (int q = 1; q < 4; q++) {
            mn = fmin(mn, lo[q][lane]);
            mx = fmax(mx, hi[q][lane]);
        }
        if (mn <= mx) {
            atomicMin(&range[2 * l], wide_order(mn));
            atomicMax(&range[2 * l + 1], wide_order(mx));
        }
    }
}

// Centre and scale (one workgroup). Cosine: no centre, unit rows scaled to 2^14; inner product: no
// centre, the scale from the largest magnitude. kmax > 0: the largest value of the type that keys
// are rounded to; data whose keys could exceed it are marked bad.
__global__ __launch_bounds__(256) void wide_scale_kernel(const unsigned long long *range, int d,
                                                         int mode, double kmax, double *mu,
                                                         WideScale *sc) {
    __shared__ double half[256], big[256];
    const int t = threadIdx.x;
    double h = 0.0, a = 0.0;
    for (int l = t; l < d; l += 256) {
        double m = 0.0;
        if (mode != WIDE_COSINE && range[2 * l] <= range[2 * l + 1]) {
            const double lo = wide_value(range[2 * l]), hi = wide_value(range[2 * l + 1]);
            m = mode == WIDE_INNER ? 0.0 : lo + 0.5 * (hi - lo);
            h = fmax(h, fmax(hi - m, m - lo));
            a = fmax(a, fmax(fabs(lo), fabs(hi)));
        }
        mu[l] = m;
    }
    half[t] = h;
    big[t] = a;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (t < w) {
            half[t] = fmax(half[t], half[t + w]);
            big[t] = fmax(big[t], big[t + w]);
        }
        __syncthreads();
    }
    if (t == 0) {
        double s = 16384.0, b = 0.0;
        if (mode != WIDE_COSINE) {
            int E = 15;
            if (half[0] > 0.0)
                (void)frexp(half[0], &E);
            E = E < -200 ? -200 : (E > 200 ? 200 : E);
            s = ldexp(1.0, 15 - E); // training values stay below 2^15 (for E <= 200)
            b = big[0];
            // Queries reach twice the training range, so keys stay below 9 d half^2.
            if (!(b < 1e60) || (kmax > 0.0 && !(16.0 * d * half[0] * half[0] < kmax)))
                sc->bad = 1;
        }
        sc->scale = s;
        sc->big = b;
    }
}

// Operand rows, 16 a tile: [k step of 32][hi, lo][lane][8], lane 16 g + r holding features
// 32 ks + 8 g .. + 7 of row r (a fragment is 1 KB of contiguous memory). One workgroup per tile,
// its waves taking every blockDim / 64-th k step (1,066 queries of 784 features are 67 tiles: with
// one wave each the pass took 74 us).
// Training rows: h[row] = |y'|^2/2 (0 for cosine) and the largest |y'|^2; query rows: the error
// bound err[row] of their scores, +inf where a value is not finite or exceeds fp16's range.
// map: row i is row map[i] of X, -1 for padding (h = +inf). quantum: the rounding of keys below the
// normal range of the type they are rounded to. FORM PACK_ROWS: [row][k step][hi, lo][32] instead of
// tiles, for kernels that gather rows; PACK_HI: tiles of hi only, h = |y'|^2/2 (1 - ce), +inf for
// padding. nrm: |x'|^2 of query rows, +inf where they do not fit.
enum { PACK_TILES = 0, PACK_ROWS = 1, PACK_HI = 2 };
template <typename T, int FORM>
__global__ __launch_bounds__(1024) void wide_pack_kernel(
    const T *__restrict__ X, int rows, int d, int KS, const double *__restrict__ mu,
    WideScale *sc, const double *__restrict__ cosn, const int *__restrict__ map, int mode,
    double ce, double quantum, _Float16 *__restrict__ P,
    float *__restrict__ h, float *__restrict__ err, double *__restrict__ nrm) {
    __shared__ double rn[16][16], rb[16][16], rt[16][16];
    __shared__ int rf[16][16];
    const int t = blockIdx.x, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const int row = t * 16 + r;
    const int src = row < rows ? (map ? map[row] : row) : -1;
    const double s = sc->scale;
    const double inv = (cosn && src >= 0) ? 1.0 / cosn[src] : 1.0;
    double nn = 0.0, big = 0.0, top = 0.0;
    // A norm that overflowed makes a row of zeros here and keys of 1 or NaN there.
    bool nf = inv == 0.0;
    for (int ks = w; ks < KS; ks += nw) {
        v8h hi, lo;
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const int l = ks * 32 + g * 8 + e;
            double v = 0.0;
            if (src >= 0 && l < d) {
                const double x = (double)X[(int64_t)src * d + l];
                v = (x - mu[l]) * inv * s;
                big = fmax(big, fabs(x));
            }
            nf |= !(v - v == 0.0);
            top = fmax(top, fabs(v));
            const _Float16 hv = (_Float16)(float)v;
            hi[e] = hv;
            lo[e] = (_Float16)(float)(v - (double)(float)hv);
            nn = fma(v, v, nn);
        }
        if constexpr (FORM == PACK_HI) {
            *reinterpret_cast<v8h *>(P + ((int64_t)t * KS + ks) * 512 + lane * 8) = hi;
        } else {
            _Float16 *dst = FORM == PACK_ROWS ? P + ((int64_t)row * KS + ks) * 64 + g * 8
                                              : P + ((int64_t)t * KS + ks) * 1024 + lane * 8;
            *reinterpret_cast<v8h *>(dst) = hi;
            *reinterpret_cast<v8h *>(dst + (FORM == PACK_ROWS ? 32 : 512)) = lo;
        }
    }
#pragma unroll
    for (int o = 16; o <= 32; o <<= 1) {
        nn += __shfl_xor(nn, o, 64);
        big = fmax(big, __shfl_xor(big, o, 64));
        top = fmax(top, __shfl_xor(top, o, 64));
        nf |= __shfl_xor((int)nf, o, 64) != 0;
    }
    if (g == 0) {
        rn[w][r] = nn;
        rb[w][r] = big;
        rt[w][r] = top;
        rf[w][r] = nf;
    }
    __syncthreads();
    if (w != 0 || g != 0)
        return;
    for (int q = 1; q < nw; q++) {
        nn += rn[q][r];
        big = fmax(big, rb[q][r]);
        top = fmax(top, rt[q][r]);
        nf |= rf[q][r] != 0;
    }
    const bool fits = !nf && top < 60000.0;
    if (h) {
        h[row] = (map || FORM == PACK_HI) && src < 0 ? __builtin_huge_valf()
                 : FORM == PACK_HI                   ? (float)(0.5 * nn * (1.0 - ce))
                 : mode == WIDE_EUCLIDEAN ? (float)(0.5 * nn)
                                          : 0.0f;
        double top2 = fits ? nn : 0.0;
#pragma unroll
        for (int o = 1; o < 16; o <<= 1)
            top2 = fmax(top2, __shfl_xor(top2, o, 16));
        if (r == 0)
            atomicMax(&sc->ymax2, (unsigned long long)__double_as_longlong(top2));
        if (!fits)
            atomicOr(&sc->bad, 1);
    }
    if (nrm)
        nrm[row] = src >= 0 && fits ? nn : __builtin_huge_val();
    if (err) {
        const double y2 = __longlong_as_double((long long)sc->ymax2);
        // Centring: the double rounding of x - mu, relative to the larger of the two.
        const double alpha = ldexp(1.0, -24) +
                             (cosn ? ldexp(1.0, -50) * s : s * ldexp(1.0, -51) * (big + sc->big));
        // Inner product: queries and rows may differ in magnitude, so the product of the norms.
        const double p2 = mode == WIDE_INNER ? sqrt(nn) * sqrt(y2) : 0.5 * (nn + y2);
        const double E = ce * p2 + 2.0 * alpha * sqrt((double)d) * (sqrt(nn) + sqrt(y2)) +
                         s * s * quantum;
        err[row] = fits ? (float)(E * (1.0 + 1e-6)) : __builtin_huge_valf();
    }
}

__device__ __forceinline__ void wide_copy(const _Float16 *g, _Float16 *l) {
    // 16 bytes per lane from g (per lane) to l + 16 lane (l wave-uniform).
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)g,
                                     (__attribute__((address_space(3))) void *)l, 16, 0, 0);
}

// Scores of 128 queries x 128 training rows per workgroup, each wave 64 x 64. A k step's
// fragments (32 KB for the tile) are copied straight to LDS one step ahead of the products (two
// buffers, one barrier a step, two workgroups per CU). Bound by the matrix cores: 48 products a
// wave and step against 16 LDS reads. Work items are dealt to the XCDs in contiguous ranges,
// query blocks fastest, so a training panel is read by one XCD and stays in its L2 while the
// query blocks pass.
__global__ __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(2))) void wide_scores_kernel(
    const _Float16 *__restrict__ PA, const _Float16 *__restrict__ PB,
    const float *__restrict__ h, int KS, int nqb, int ntb, float *__restrict__ out, int64_t ldo) {
    __shared__ __attribute__((aligned(16))) _Float16 s0[32 * 512];
    __shared__ __attribute__((aligned(16))) _Float16 s1[32 * 512];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int r = lane & 15, g = lane >> 4;
    const int nwork = nqb * ntb, per_xcd = (nwork + 7) / 8;
    const int work = (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3);
    if (work >= nwork || (int)(blockIdx.x >> 3) >= per_xcd)
        return;
    const int tb = work / nqb, qb = work - tb * nqb;
    const int wr = w >> 1, wc = w & 1;
    v4f acc[4][4], sum[4][4];
#pragma unroll
    for (int ct = 0; ct < 4; ct++) {
        const float hv = -h[tb * 128 + (wc * 4 + ct) * 16 + r];
#pragma unroll
        for (int rt = 0; rt < 4; rt++) {
            sum[rt][ct] = v4f{hv, hv, hv, hv};
            acc[rt][ct] = v4f{0.f, 0.f, 0.f, 0.f};
        }
    }
    auto stage = [&](int ks, _Float16 *dst) {
#pragma unroll
        for (int b = 0; b < 8; b++) {
            const int blk = w * 8 + b; // 0..15 query fragments, 16..31 training fragments
            const int tile = (blk & 15) >> 1, half = blk & 1;
            const _Float16 *src = blk < 16 ? PA + ((int64_t)(qb * 8 + tile) * KS + ks) * 1024
                                           : PB + ((int64_t)(tb * 8 + tile) * KS + ks) * 1024;
            wide_copy(src + half * 512 + lane * 8, dst + blk * 512);
        }
    };
    auto compute = [&](const _Float16 *s) {
        v8h a[4][2];
#pragma unroll
        for (int rt = 0; rt < 4; rt++)
#pragma unroll
            for (int hf = 0; hf < 2; hf++)
                a[rt][hf] = *reinterpret_cast<const v8h *>(
                    s + ((wr * 4 + rt) * 2 + hf) * 512 + lane * 8);
#pragma unroll
        for (int ct = 0; ct < 4; ct++) {
            const _Float16 *p = s + (16 + (wc * 4 + ct) * 2) * 512 + lane * 8;
            const v8h bh = *reinterpret_cast<const v8h *>(p);
            const v8h bl = *reinterpret_cast<const v8h *>(p + 512);
#pragma unroll
            for (int rt = 0; rt < 4; rt++)
                acc[rt][ct] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[rt][0], bh, acc[rt][ct], 0, 0, 0);
#pragma unroll
            for (int rt = 0; rt < 4; rt++)
                acc[rt][ct] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[rt][0], bl, acc[rt][ct], 0, 0, 0);
#pragma unroll
            for (int rt = 0; rt < 4; rt++)
                acc[rt][ct] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[rt][1], bh, acc[rt][ct], 0, 0, 0);
        }
    };
    auto flush = [&]() {
#pragma unroll
        for (int rt = 0; rt < 4; rt++)
#pragma unroll
            for (int ct = 0; ct < 4; ct++) {
                sum[rt][ct] += acc[rt][ct];
                acc[rt][ct] = v4f{0.f, 0.f, 0.f, 0.f};
            }
    };
    stage(0, s0);
    for (int ks = 0; ks < KS; ks += 2) {
        __builtin_amdgcn_s_waitcnt(0x0F70); // vmcnt(0): this wave's copies have landed
        __syncthreads();
        if (ks + 1 < KS)
            stage(ks + 1, s1);
        compute(s0);
        if (ks + 1 < KS) {
            __builtin_amdgcn_s_waitcnt(0x0F70);
            __syncthreads();
            if (ks + 2 < KS)
                stage(ks + 2, s0);
            compute(s1);
        }
        if ((ks & 7) == 6)
            flush();
    }
    flush();
#pragma unroll
    for (int rt = 0; rt < 4; rt++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            float *o = out + (int64_t)(qb * 128 + (wr * 4 + rt) * 16 + 4 * g + i) * ldo +
                       tb * 128 + wc * 64 + r;
#pragma unroll
            for (int ct = 0; ct < 4; ct++)
                o[ct * 16] = -sum[rt][ct][i];
        }
}

// One wave per query: the kc selected scores (ascending, by (score, row)) -> exact keys of those
// within 2 E of the k-th, ordered by (key, row).
template <typename T, bool COS>
__global__ __launch_bounds__(64) void wide_merge_kernel(
    const float *__restrict__ skey, const int *__restrict__ sidx, int kc, int k,
    const T *__restrict__ Q, const T *__restrict__ Y, int d, const float *__restrict__ err,
    const double *__restrict__ qcos, const double *__restrict__ ycos, int post, int q0,
    T *__restrict__ out_dist, int *__restrict__ out_idx, int *__restrict__ fb_count,
    int *__restrict__ fb_list) {
    extern __shared__ double qrow[];
    __shared__ double xk[WIDE_KEEP];
    __shared__ int xi[WIDE_KEEP];
    const int q = blockIdx.x, lane = threadIdx.x;
    const float *kk = skey + (int64_t)q * kc;
    const int *ki = sidx + (int64_t)q * kc;
    const double E = (double)err[q];
    const double lim = (double)kk[k - 1] + 2.0 * E;
    const bool certified = E < __builtin_huge_val() && (double)kk[kc - 1] > lim;
    if (!certified) {
        if (lane == 0)
            fb_list[atomicAdd(fb_count, 1)] = q0 + q;
        return;
    }
    for (int l = lane; l < d; l += 64)
        qrow[l] = (double)Q[(int64_t)q * d + l];
    int nr = 0;
    for (int b = 0; b < kc; b += 64) {
        const bool in = b + lane < kc && (double)kk[b + lane] <= lim;
        nr += __popcll(__builtin_amdgcn_ballot_w64(in));
    }
    __syncthreads();
    constexpr int VE = 16 / (int)sizeof(T);
    const bool vec = d % VE == 0;
    for (int c = lane; c < nr; c += 64) {
        const int j = ki[c];
        const T *y = Y + (int64_t)j * d;
        double acc = 0.0;
        auto term = [&](double x, double yv) {
            if constexpr (COS) {
                acc = fma(x, yv, acc);
            } else {
                const double t = x - yv;
                acc = fma(t, t, acc);
            }
        };
        if (vec) {
#pragma unroll 16
            for (int l = 0; l < d; l += VE) {
                const uint4 u = *reinterpret_cast<const uint4 *>(y + l);
                T v[VE];
                __builtin_memcpy(v, &u, 16);
#pragma unroll
                for (int e = 0; e < VE; e++)
                    term(qrow[l + e], (double)v[e]);
            }
        } else {
            for (int l = 0; l < d; l++)
                term(qrow[l], (double)y[l]);
        }
        xk[c] = COS ? 1.0 - acc / (qcos[q] * ycos[j]) : acc;
        xi[c] = j;
    }
    __syncthreads();
    for (int c = lane; c < nr; c += 64) {
        const double v = xk[c];
        const int j = xi[c];
        int rank = 0;
        for (int o = 0; o < nr; o++)
            rank += xk[o] < v || (xk[o] == v && xi[o] < j);
        if (rank < k) {
            if (out_dist)
                out_dist[(int64_t)q * k + rank] = (T)(post == 1 ? sqrt(v < 0.0 ? 0.0 : v) : v);
            out_idx[(int64_t)q * k + rank] = j;
        }
    }
}

} // namespace

double wide_relative_bound(int products) {
    const double terms = products + 16.0, u = 1.0 / 16777216.0;
    return 1.05 * terms * u / (1.0 - terms * u) + 1.0 / 262144.0;
}

template <typename T, int FORM = PACK_TILES>
static void wide_prepare(const T *Y, int n, int d, int mode, const double *ycos, const int *map,
                         int rows, int tiles, double kmax, unsigned long long *range, double *mu,
                         WideScale *sc, void *P, float *h, hipStream_t s) {
    const int KS = wide_ksteps(d);
    hipLaunchKernelGGL(wide_range_init_kernel, dim3((d + 255) / 256), dim3(256), 0, s, range, d, sc);
    if (mode != WIDE_COSINE) {
        const int by = std::min(d > 512 ? 128 : 512, (n + 63) / 64);
        hipLaunchKernelGGL(wide_range_kernel<T>, dim3((d + 63) / 64, by), dim3(256), 0, s, Y, n, d,
                           range, sc);
    }
    hipLaunchKernelGGL(wide_scale_kernel, dim3(1), dim3(256), 0, s, range, d, mode, kmax, mu, sc);
    hipLaunchKernelGGL((wide_pack_kernel<T, FORM>), dim3(tiles), dim3(64 * std::min(16, KS)), 0, s,
                       Y, rows, d, KS, mu, sc, ycos, map, mode, 0.0, 0.0,
                       static_cast<_Float16 *>(P), h, (float *)nullptr, (double *)nullptr);
}

template <typename T>
hipError_t launch_wide_prepare(const T *Y, int n, int d, const double *ycos,
                               unsigned long long *range, double *mu, WideScale *sc, void *P,
                               float *h, hipStream_t s) {
    wide_prepare<T>(Y, n, d, ycos ? WIDE_COSINE : WIDE_EUCLIDEAN, ycos, nullptr, n,
                    wide_rows(n) / 16, 0.0, range, mu, sc, P, h, s);
    return hipGetLastError();
}

template <typename T>
hipError_t launch_wide_queries(const T *Q, int nq, int d, const double *qcos, const double *mu,
                               WideScale *sc, void *P, float *err, hipStream_t s) {
    const int KS = wide_ksteps(d), tiles = wide_rows(nq) / 16;
    hipLaunchKernelGGL((wide_pack_kernel<T, PACK_TILES>), dim3(tiles), dim3(64 * std::min(16, KS)), 0, s,
                       Q, nq, d, KS, mu, sc, qcos, (const int *)nullptr,
                       qcos ? WIDE_COSINE : WIDE_EUCLIDEAN, wide_relative_bound(3 * 256), 0.0,
                       static_cast<_Float16 *>(P), (float *)nullptr, err, (double *)nullptr);
    return hipGetLastError();
}

template <typename T>
hipError_t launch_bits_prepare(const T *Y, int n, int d, double ce, const int *smap, int ns,
                               unsigned long long *range, double *mu, WideScale *sc, void *PS,
                               float *hS, void *P, float *B, hipStream_t s) {
    const int KS = wide_ksteps(d);
    // The sample's operand first: it leaves the centre and scale; the whole set's pass leaves the
    // largest norm.
    wide_prepare<T, PACK_HI>(Y, n, d, WIDE_EUCLIDEAN, nullptr, smap, ns, ns / 16, 0.0, range, mu, sc, PS, hS,
                    s);
    hipLaunchKernelGGL((wide_pack_kernel<T, PACK_HI>), dim3(bits_rows(n) / 16), dim3(64 * KS), 0, s,
                       Y, n, d, KS, mu, sc, (const double *)nullptr, (const int *)nullptr,
                       WIDE_EUCLIDEAN, ce, 0.0, static_cast<_Float16 *>(P), B, (float *)nullptr,
                       (double *)nullptr);
    return hipGetLastError();
}

template <typename T>
hipError_t launch_bits_queries(const T *Q, int nq, int d, const double *mu, WideScale *sc, void *P,
                               double *nrm, hipStream_t s) {
    const int KS = wide_ksteps(d);
    hipLaunchKernelGGL((wide_pack_kernel<T, PACK_HI>), dim3((nq + 255) / 256 * 16),
                       dim3(64 * KS), 0, s, Q, nq, d, KS, mu, sc, (const double *)nullptr,
                       (const int *)nullptr, WIDE_EUCLIDEAN, 0.0, 0.0, static_cast<_Float16 *>(P),
                       (float *)nullptr, (float *)nullptr, nrm);
    return hipGetLastError();
}

template <typename T>
hipError_t launch_ivf_lists(const T *X, int n, int d, int ip, const int *map, int rows,
                            unsigned long long *range, double *mu, WideScale *sc, void *P, float *h,
                            hipStream_t s) {
    wide_prepare<T>(X, n, d, ip ? WIDE_INNER : WIDE_EUCLIDEAN, nullptr, map, rows, rows / 16,
                    (double)std::numeric_limits<T>::max(), range, mu, sc, P, h, s);
    return hipGetLastError();
}

template <typename T>
hipError_t launch_ivf_queries(const T *Q, int nq, int d, int ip, const double *mu, WideScale *sc,
                              void *P, float *err, hipStream_t s) {
    const int KS = wide_ksteps(d);
    // Keys are rounded to T: relative 2^-24 (fp32) of at most 2 (|x'|^2 + |y'|^2), covered by the
    // 2^-22 added to the relative bound, and the quantum below the normal range.
    const double quantum = sizeof(T) == 4 ? std::ldexp(1.0, -149) : 0.0;
    hipLaunchKernelGGL((wide_pack_kernel<T, PACK_ROWS>), dim3((nq + 15) / 16),
                       dim3(64 * std::min(16, KS)), 0, s, Q, nq, d, KS, mu, sc,
                       (const double *)nullptr, (const int *)nullptr,
                       ip ? WIDE_INNER : WIDE_EUCLIDEAN,
                       wide_relative_bound(3 * 32 * KS) + 1.0 / 4194304.0, quantum,
                       static_cast<_Float16 *>(P), (float *)nullptr, err, (double *)nullptr);
    return hipGetLastError();
}

hipError_t launch_wide_scores(const void *PA, int nq, const void *PB, int n, int d, const float *h,
                              float *out, hipStream_t s) {
    const int nqb = wide_rows(nq) / 128, ntb = wide_rows(n) / 128;
    const unsigned grid = (unsigned)(((int64_t)nqb * ntb + 7) / 8 * 8);
    hipLaunchKernelGGL(wide_scores_kernel, dim3(grid), dim3(256), 0, s,
                       static_cast<const _Float16 *>(PA), static_cast<const _Float16 *>(PB), h,
                       wide_ksteps(d), nqb, ntb, out, (int64_t)wide_rows(n));
    return hipGetLastError();
}

template <typename T>
hipError_t launch_wide_merge(const float *skey, const int *sidx, int nq, int kc, int k, const T *Q,
                             const T *Y, int d, const float *err, const double *qcos,
                             const double *ycos, int post, int q0, T *out_dist, int *out_idx,
                             int *fb_count, int *fb_list, hipStream_t s) {
    if (kc > WIDE_KEEP || k > kc || nq < 1 || (size_t)d * sizeof(double) > 60 * 1024)
        return hipErrorInvalidValue;
    auto kern = qcos ? wide_merge_kernel<T, true> : wide_merge_kernel<T, false>;
    hipLaunchKernelGGL(kern, dim3(nq), dim3(64), d * sizeof(double), s, skey, sidx, kc, k, Q,
                       Y, d, err, qcos, ycos, post, q0, out_dist, out_idx, fb_count, fb_list);
    return hipGetLastError();
}

#define DA_WIDE_INST(T)                                                                          \
    template hipError_t launch_wide_prepare<T>(const T *, int, int, const double *,              \
                                               unsigned long long *, double *, WideScale *,      \
                                               void *, float *, hipStream_t);                    \
    template hipError_t launch_wide_queries<T>(const T *, int, int, const double *,              \
                                               const double *, WideScale *, void *, float *,     \
                                               hipStream_t);                                     \
    template hipError_t launch_bits_prepare<T>(const T *, int, int, double, const int *, int,    \
                                               unsigned long long *, double *, WideScale *,      \
                                               void *, float *, void *, float *, hipStream_t);   \
    template hipError_t launch_bits_queries<T>(const T *, int, int, const double *, WideScale *, \
                                               void *, double *, hipStream_t);                   \
    template hipError_t launch_ivf_lists<T>(const T *, int, int, int, const int *, int,          \
                                            unsigned long long *, double *, WideScale *, void *, \
                                            float *, hipStream_t);                               \
    template hipError_t launch_ivf_queries<T>(const T *, int, int, int, const double *,          \
                                              WideScale *, void *, float *, hipStream_t);        \
    template hipError_t launch_wide_merge<T>(const float *, const int *, int, int, int,          \
                                             const T *, const T *, int, const float *,           \
                                             const double *, const double *, int, int, T *,      \
                                             int *, int *, int *, hipStream_t);
DA_WIDE_INST(float)
DA_WIDE_INST(double)
#undef DA_WIDE_INST

} // namespace dagpu
