// GEMM-form distance tiles on the fp64 matrix cores of gfx950 (v_mfma_f64_16x16x4f64), for
// the metrics whose value is a function of the dot product x.y: squared euclidean and
// euclidean (|x|^2 + |y|^2 - 2 x.y), their GEMM-form variants, cosine (1 - x.y/(|x||y|)) and
// the inner product. Both input precisions are widened to double when staged, so the cross
// term carries fp64 accuracy whatever the data type.
//
// The reference computes euclidean and squared euclidean with direct differences
// (source/core/metrics/metrics_kernels.hpp:413-1070), which are accurate to a few ulps of the
// distance itself; the GEMM form is accurate to a few ulps of |x|^2 + |y|^2 instead. Each
// element therefore carries the rounding bound of its GEMM form,
//     E = 2.01 gamma_{k+2} (|x|^2 + |y|^2),   gamma_n = n u / (1 - n u),  u = 2^-53,
// and an element whose value does not exceed E / rtol (rtol = 5e-13 for double output,
// 5e-7 for float output) is recomputed with direct differences in double: the distances keep
// the direct form's relative accuracy, the diagonal of X against itself is exactly zero.
// The GEMM-form variants, cosine and the inner product are GEMM products in the reference
// too (euclidean_gemm_distance.cpp:59-230, cosine_distance.cpp:66-161,
// inner_product_distance.cpp) and are stored as computed.
//
// Work decomposition: a 256-thread workgroup owns a TB x TB output tile, and each wave accumulates a
// quarter of it in 16 x 16 blocks on the matrix cores. 16-deep k slices of X and Y lie in LDS in the
// input type (widened when read) in two buffers: the next slice is loaded to registers before the
// products of this one and stored after them, with one barrier a slice. Bound by the matrix cores (a
// product occupies its SIMD for 64 cycles) and, for few features, by the epilogue. 8,192 x 8,192 x
// 256 fp32: 626 us; with one buffer and loads waited for between barriers 920. Operand
// layout of v_mfma_f64_16x16x4f64 for lane l: A[l % 16][l / 16], B[l / 16][l % 16]; the
// accumulator's register r holds C[4 r + l / 16][l % 16].
#include "launch.hpp"
#include <algorithm>
#include <cstdint>
#include <hip/hip_runtime.h>

namespace dagpu {

namespace {

constexpr int KC = 16; // k slice staged in LDS

typedef double v4d __attribute__((ext_vector_type(4)));

template <typename T, typename TY>
__device__ double direct_sqdist(const T *__restrict__ x, const TY *__restrict__ y, int k) {
    double acc = 0.0;
    for (int l = 0; l < k; l++) {
        const double d = (double)x[l] - (double)y[l];
        acc = fma(d, d, acc);
    }
    return acc;
}

// A thread's part of a TB x KC slice: VE consecutive k of TB * KC / (256 VE) rows. VE > 1 needs rows
// of whole 16-byte pieces.
template <typename T, int TB, int VE> struct Slice {
    static constexpr int PER = KC / VE, ROWS = 256 / PER, N = TB / ROWS;
    T v[N][VE];
    __device__ __forceinline__ void load(const T *__restrict__ X, int i0, int m, int k, int k0,
                                         int tid) {
        const int kk = k0 + (tid % PER) * VE, row = tid / PER;
#pragma unroll
        for (int s = 0; s < N; s++) {
            const int gi = i0 + row + s * ROWS;
            const bool in = kk < k && gi < m;
            if constexpr (VE > 1) {
                uint4 u = make_uint4(0, 0, 0, 0);
                if (in)
                    u = *reinterpret_cast<const uint4 *>(X + (int64_t)gi * k + kk);
                __builtin_memcpy(v[s], &u, 16);
            } else {
                v[s][0] = in ? X[(int64_t)gi * k + kk] : (T)0;
            }
        }
    }
    __device__ __forceinline__ void store(T (*S)[TB + 4], int tid) const {
        const int kk = (tid % PER) * VE, row = tid / PER;
#pragma unroll
        for (int s = 0; s < N; s++)
#pragma unroll
            for (int e = 0; e < VE; e++)
                S[kk + e][row + s * ROWS] = v[s][e];
    }
};

template <typename T, typename TY, typename U, int METRIC, int TB, bool VEC>
__global__ __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(2))) void pairwise_mfma_kernel(
    const T *__restrict__ X, const TY *__restrict__ Y, int m, int n, int k, U *__restrict__ D,
    int64_t ldd, const double *__restrict__ nx, const double *__restrict__ ny, int zero_diag,
    int diag_offset, double gam, double inv_rtol) {
    constexpr int RB = TB / 32; // blocks of 16 per wave and side
    __shared__ T Xs[2][KC][TB + 4];
    __shared__ TY Ys[2][KC][TB + 4];
    const int tid = threadIdx.x;
    const int lane = tid & 63, w = tid >> 6;
    const int wr = w >> 1, wc = w & 1;
    const int i0 = blockIdx.y * TB, j0 = blockIdx.x * TB;

    v4d acc[RB][RB];
#pragma unroll
    for (int a = 0; a < RB; a++)
#pragma unroll
        for (int b = 0; b < RB; b++)
            acc[a][b] = (v4d){0.0, 0.0, 0.0, 0.0};

    const int kq = lane >> 4, col = lane & 15;
    Slice<T, TB, VEC ? 16 / (int)sizeof(T) : 1> xs;
    Slice<TY, TB, VEC ? 16 / (int)sizeof(TY) : 1> ys;
    xs.load(X, i0, m, k, 0, tid);
    ys.load(Y, j0, n, k, 0, tid);
    xs.store(Xs[0], tid);
    ys.store(Ys[0], tid);
    int cur = 0;
    for (int k0 = 0; k0 < k; k0 += KC, cur ^= 1) {
        __syncthreads();
        const bool more = k0 + KC < k;
        if (more) {
            xs.load(X, i0, m, k, k0 + KC, tid);
            ys.load(Y, j0, n, k, k0 + KC, tid);
        }
#pragma unroll
        for (int q = 0; q < KC; q += 4) {
            double a[RB], b[RB];
#pragma unroll
            for (int t = 0; t < RB; t++) {
                a[t] = (double)Xs[cur][q + kq][wr * (TB / 2) + t * 16 + col];
                b[t] = (double)Ys[cur][q + kq][wc * (TB / 2) + t * 16 + col];
            }
#pragma unroll
            for (int ra = 0; ra < RB; ra++)
#pragma unroll
                for (int cb = 0; cb < RB; cb++)
                    acc[ra][cb] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[ra], b[cb], acc[ra][cb],
                                                                        0, 0, 0);
        }
        // The other buffer was last read before this slice's barrier.
        if (more) {
            xs.store(Xs[cur ^ 1], tid);
            ys.store(Ys[cur ^ 1], tid);
        }
    }

#pragma unroll
    for (int ra = 0; ra < RB; ra++) {
#pragma unroll
        for (int cb = 0; cb < RB; cb++) {
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int i = i0 + wr * (TB / 2) + ra * 16 + 4 * r + kq;
                const int j = j0 + wc * (TB / 2) + cb * 16 + col;
                if (i >= m || j >= n)
                    continue;
                const double g = acc[ra][cb][r];
                double v;
                if constexpr (METRIC == KM_SQEUCLIDEAN || METRIC == KM_EUCLIDEAN) {
                    const double s = nx[i] + ny[j];
                    v = s - 2.0 * g;
                    if (v <= 2.01 * gam * s * inv_rtol)
                        v = direct_sqdist(X + (int64_t)i * k, Y + (int64_t)j * k, k);
                    if constexpr (METRIC == KM_EUCLIDEAN)
                        v = sqrt(v);
                } else if constexpr (METRIC == KM_SQEUCLIDEAN_GEMM ||
                                     METRIC == KM_EUCLIDEAN_GEMM) {
                    v = nx[i] + ny[j] - 2.0 * g;
                    v = v < 0.0 ? 0.0 : v;
                    if constexpr (METRIC == KM_EUCLIDEAN_GEMM)
                        v = sqrt(v);
                } else if constexpr (METRIC == KM_COSINE) {
                    v = 1.0 - g / (nx[i] * ny[j]);
                } else {
                    v = g;
                }
                if (zero_diag && i + diag_offset == j)
                    v = 0.0;
                D[(int64_t)i * ldd + j] = (U)v;
            }
        }
    }
}

// Tile edge and load width of a call. Tiles of 128 halve the operand reads but leave fewer
// workgroups on a CU, so that epilogues overlap less with products: 8,192 x 8,192 fp32 euclidean
// by tiles of 64 and 128: 148 and 204 us with 3 features, 238 and 292 with 64, 626 and 676 with 256,
// equal with 512; inner products 1,205 and 1,169 with 512, 4,096 x 4,096 fp64 699 and 646 with 1,024.
template <typename T, typename TY, typename U, int METRIC>
void pairwise_mfma_run(const T *X, const TY *Y, int m, int n, int k, U *D, int64_t ldd,
                       const double *nx, const double *ny, int zero_diag, int diag_offset,
                       double gam, double inv_rtol, hipStream_t s) {
    auto run = [&](auto kern, int tb) {
        // At most 65,535 row tiles per launch (the grid's y extent).
        const int64_t step = (int64_t)65535 * tb;
        for (int64_t i0 = 0; i0 < m; i0 += step) {
            const int mm = (int)std::min<int64_t>(step, m - i0);
            hipLaunchKernelGGL(kern, dim3((n + tb - 1) / tb, (mm + tb - 1) / tb), dim3(256), 0, s,
                               X + i0 * k, Y, mm, n, k, D + i0 * ldd, ldd, nx ? nx + i0 : nx, ny,
                               zero_diag, diag_offset + (int)i0, gam, inv_rtol);
        }
    };
    auto aligned = [&](const void *p, size_t size) {
        return ((uintptr_t)p & 15) == 0 && k * size % 16 == 0;
    };
    const bool vec = aligned(X, sizeof(T)) && aligned(Y, sizeof(TY));
    const bool large = k >= 512 && (int64_t)((m + 127) / 128) * ((n + 127) / 128) >= 1024;
    if (large)
        run(vec ? pairwise_mfma_kernel<T, TY, U, METRIC, 128, true>
                : pairwise_mfma_kernel<T, TY, U, METRIC, 128, false>, 128);
    else
        run(vec ? pairwise_mfma_kernel<T, TY, U, METRIC, 64, true>
                : pairwise_mfma_kernel<T, TY, U, METRIC, 64, false>, 64);
}

} // namespace

bool pairwise_mfma_metric(int metric) {
    return metric == KM_SQEUCLIDEAN || metric == KM_EUCLIDEAN || metric == KM_COSINE ||
           metric == KM_INNER || metric == KM_SQEUCLIDEAN_GEMM || metric == KM_EUCLIDEAN_GEMM;
}

template <typename T, typename U>
hipError_t launch_pairwise_mfma(int metric, const T *X, const T *Y, int m, int n, int k, U *D,
                                int64_t ldd, const double *nx, const double *ny, int zero_diag,
                                int diag_offset, hipStream_t s) {
    if (!pairwise_mfma_metric(metric) || !nx || !ny)
        return hipErrorInvalidValue;
    if (m <= 0 || n <= 0)
        return hipSuccess;
    const double u = 1.0 / 9007199254740992.0; // 2^-53
    const double nk = (double)(k + 2);
    const double gam = nk * u / (1.0 - nk * u);
    const double inv_rtol = sizeof(U) == 8 ? 2e12 : 2e6;
#define DA_PWM_CASE(M)                                                                       \
    case M:                                                                                  \
        pairwise_mfma_run<T, T, U, M>(X, Y, m, n, k, D, ldd, nx, ny, zero_diag, diag_offset,  \
                                      gam, inv_rtol, s);                                      \
        break;
    switch (metric) {
        DA_PWM_CASE(KM_SQEUCLIDEAN)
        DA_PWM_CASE(KM_EUCLIDEAN)
        DA_PWM_CASE(KM_COSINE)
        DA_PWM_CASE(KM_INNER)
        DA_PWM_CASE(KM_SQEUCLIDEAN_GEMM)
        DA_PWM_CASE(KM_EUCLIDEAN_GEMM)
    default:
        return hipErrorInvalidValue;
    }
#undef DA_PWM_CASE
    return hipGetLastError();
}

template <typename TX, typename TY>
hipError_t launch_inner_mfma(const TX *X, const TY *Y, int m, int n, int k, float *D,
                             int64_t ldd, hipStream_t s) {
    if (m <= 0 || n <= 0)
        return hipSuccess;
    pairwise_mfma_run<TX, TY, float, KM_INNER>(X, Y, m, n, k, D, ldd, nullptr, nullptr, 0, 0, 0.0,
                                               0.0, s);
    return hipGetLastError();
}
template hipError_t launch_inner_mfma<double, float>(const double *, const float *, int, int,
                                                     int, float *, int64_t, hipStream_t);
template hipError_t launch_inner_mfma<double, double>(const double *, const double *, int, int,
                                                      int, float *, int64_t, hipStream_t);

template hipError_t launch_pairwise_mfma<float, float>(int, const float *, const float *, int,
                                                       int, int, float *, int64_t,
                                                       const double *, const double *, int, int,
                                                       hipStream_t);
template hipError_t launch_pairwise_mfma<double, double>(int, const double *, const double *,
                                                         int, int, int, double *, int64_t,
                                                         const double *, const double *, int,
                                                         int, hipStream_t);

} // namespace dagpu
