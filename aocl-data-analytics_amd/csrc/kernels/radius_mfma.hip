// Radius search on the fp16 matrix cores of gfx950: for every (query, training row) pair one
// bit, for the metrics that are a function of the squared euclidean distance.
//
// The key tile of the general path costs 3 d double operations and 2 x 4 or 8 bytes of HBM
// traffic per pair (written, then read by the selection), whatever the outcome. Here the
// product x.y of the rows, held as hi + lo in fp16 (hi*hi + hi*lo + lo*hi on
// v_mfma_f32_16x16x32_f16, three products for 32 features), rules out nearly every pair by an
// error bound, and only a bit leaves the kernel: cleared when |x|^2 + |y|^2 - 2 x.y is above the
// threshold by more than the bound. launch_radius_verify forms the key of every set bit as the
// general path does (double, features in order, rounded to T) and clears the bits of the pairs
// that miss, so the bits that remain are those of the general path. The rows are centred (the
// middle of each column's range) and scaled by a power of two to fp16's range first: distances
// do not change with the centre, and the bound shrinks with the norms. Values that are not
// finite, and searches that leave too many pairs set (a radius that holds some percent of the
// rows, or rows with outliers many orders of magnitude beyond it), are reported to the caller,
// which then takes the general path (radius_bits_most).
//
// Bound: with the scaled rows x', y', n(.) the squared norm and Kp the padded width, the sum of
// 3 Kp products and the start value in fp32 carries gamma_{3 Kp + 8} (|x'||y'| + ...), the split
// operands 2^-21 relative each and the dropped lo*lo 2^-22, and |x'||y'| <= (n(x') + n(y')) / 2;
// the rounded thresholds add a few 2^-24. Together: ce (n(x') + n(y')) with ce = gamma + 2^-19,
// plus a constant ca for values below fp16's normal range and the rounding of the centring. The
// threshold itself is the largest squared distance whose rounded key passes (radius_threshold2).
#include "launch.hpp"
#include <algorithm>
#include <hip/hip_runtime.h>

namespace dagpu {

namespace {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));

// Doubles as unsigned keys of the same order, for atomic minima and maxima.
__device__ __forceinline__ unsigned long long order_key(double v) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    return (b >> 63) ? ~b : (b | 0x8000000000000000ull);
}
__device__ __forceinline__ double order_value(unsigned long long k) {
    return __longlong_as_double(
        (long long)((k >> 63) ? (k & 0x7FFFFFFFFFFFFFFFull) : ~k));
}

// range[2 l], range[2 l + 1]: the order keys of column l's smallest and largest value;
// range[2 d]: set when a value is not finite.
__global__ void radius_range_init_kernel(unsigned long long *range, int d) {
    for (int l = threadIdx.x; l <= d; l += blockDim.x) {
        if (l < d) {
            range[2 * l] = ~0ull;
            range[2 * l + 1] = 0ull;
        } else {
            range[2 * d] = 0ull;
        }
    }
}

template <typename T>
__global__ __launch_bounds__(256) void radius_range_kernel(const T *__restrict__ X, int64_t rows,
                                                           int d, unsigned long long *range) {
    __shared__ unsigned long long lo[128], hi[128];
    __shared__ int bad;
    if (threadIdx.x < 128) {
        lo[threadIdx.x] = ~0ull;
        hi[threadIdx.x] = 0ull;
    }
    if (threadIdx.x == 0)
        bad = 0;
    __syncthreads();
    const int spp = 256 / d, sub = (int)threadIdx.x / d, l = (int)threadIdx.x - sub * d;
    if (sub < spp) {
        double mn = __builtin_huge_val(), mx = -__builtin_huge_val();
        bool nf = false;
        const int64_t step = (int64_t)gridDim.x * spp;
        int64_t i = (int64_t)blockIdx.x * spp + sub;
        auto take = [&](T x) {
            const double v = (double)x;
            nf |= !(v - v == 0.0);
            mn = fmin(mn, v);
            mx = fmax(mx, v);
        };
        for (; i + 3 * step < rows; i += 4 * step) {
            T v[4];
#pragma unroll
            for (int u = 0; u < 4; u++)
                v[u] = X[(i + u * step) * d + l];
#pragma unroll
            for (int u = 0; u < 4; u++)
                take(v[u]);
        }
        for (; i < rows; i += step)
            take(X[i * d + l]);
        if (mn <= mx) {
            atomicMin(&lo[l], order_key(mn));
            atomicMax(&hi[l], order_key(mx));
        }
        if (nf)
            bad = 1;
    }
    __syncthreads();
    if ((int)threadIdx.x < d) {
        atomicMin(&range[2 * threadIdx.x], lo[threadIdx.x]);
        atomicMax(&range[2 * threadIdx.x + 1], hi[threadIdx.x]);
    }
    if (threadIdx.x == 0 && bad)
        atomicMax(&range[2 * d], 1ull);
}

// Centre and scale from the column ranges (one workgroup of 128 threads, d <= 128).
__global__ __launch_bounds__(128) void radius_scale_kernel(const unsigned long long *range, int d,
                                                           int gemm, RadiusScale *out) {
    __shared__ double half[128], big[128];
    const int l = threadIdx.x;
    double h = 0.0, a = 0.0;
    if (l < d && range[2 * l] <= range[2 * l + 1]) {
        const double lo = order_value(range[2 * l]), hi = order_value(range[2 * l + 1]);
        const double mu = lo + 0.5 * (hi - lo);
        out->mu[l] = mu;
        h = fmax(hi - mu, mu - lo);
        a = fmax(fabs(lo), fabs(hi));
    } else if (l < 128) {
        out->mu[l] = 0.0;
    }
    half[l] = h;
    big[l] = a;
    __syncthreads();
    for (int w = 64; w > 0; w >>= 1) {
        if (l < w) {
            half[l] = fmax(half[l], half[l + w]);
            big[l] = fmax(big[l], big[l + w]);
        }
        __syncthreads();
    }
    if (l == 0) {
        int E = 0;
        (void)frexp(half[0], &E);
        if (!(half[0] > 0.0))
            E = 15;
        E = E < -200 ? -200 : E;
        const double s = ldexp(1.0, 15 - E); // scaled values stay below 2^15
        const double X = 32768.0 * sqrt((double)d);
        // Absolute error of an element: fp16 values below the normal range, the centring.
        const double alpha = ldexp(1.0, -24) + s * ldexp(1.0, -51) * big[0];
        double ca = 4.0 * alpha * sqrt((double)d) * X * 1.01;
        // The GEMM-form metrics' own keys are rounded relative to the norms of the rows as given.
        if (gemm)
            ca += 8.0 * (d + 4) * ldexp(1.0, -53) * d * (s * big[0]) * (s * big[0]);
        out->scale = s;
        out->ca = ca;
        out->bad = range[2 * d] != 0 || !(big[0] < 1e300) ? 1 : 0;
        out->probe = out->total = 0;
    }
}

// Operand layout: 16 rows a tile, [k step of 32][hi, lo][lane][8]: lane l = 16 g + r holds
// features 32 ks + 8 g .. + 7 of row r, so a wave reads a fragment as 1 KB of contiguous
// memory. One wave per tile; rows at or beyond `rows` are zero and never hit. A pair may be a hit
// when x'.y' - A_x - B_y >= 0.
template <typename T>
__global__ __launch_bounds__(256) void radius_pack_kernel(
    const T *__restrict__ X, int rows, int tiles, int d, int KS, const RadiusScale *__restrict__ sc,
    double thr, double ce, _Float16 *__restrict__ P, float *__restrict__ A,
    float *__restrict__ B) {
    const int t = blockIdx.x * 4 + (int)(threadIdx.x >> 6);
    if (t >= tiles)
        return;
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const int row = t * 16 + r;
    const double s = sc->scale;
    double nn = 0.0;
    for (int ks = 0; ks < KS; ks++) {
        v8h hi, lo;
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const int l = ks * 32 + g * 8 + e;
            double v = 0.0;
            if (row < rows && l < d)
                v = ((double)X[(int64_t)row * d + l] - sc->mu[l]) * s;
            const _Float16 h = (_Float16)(float)v;
            hi[e] = h;
            lo[e] = (_Float16)(float)(v - (double)(float)h);
            nn = fma(v, v, nn);
        }
        _Float16 *dst = P + ((int64_t)t * KS + ks) * 1024 + lane * 8;
        *reinterpret_cast<v8h *>(dst) = hi;
        *reinterpret_cast<v8h *>(dst + 512) = lo;
    }
    nn += __shfl_xor(nn, 16, 64);
    nn += __shfl_xor(nn, 32, 64);
    if (g == 0) {
        const float inf = __builtin_huge_valf();
        const bool in = row < rows;
        // Not below -2^100: with -inf here a padding column (B = inf) would give NaN, not a miss.
        if (A)
            A[row] = in ? (float)fmax(0.5 * (nn * (1.0 - ce) - thr * s * s * (1.0 + 0x1p-20) - sc->ca),
                                      -0x1p100)
                        : inf;
        if (B)
            B[row] = in ? (float)(0.5 * nn * (1.0 - ce)) : inf;
    }
}

__device__ __forceinline__ void copy_to_lds(const _Float16 *g, _Float16 *l) {
    // 16 bytes per lane from g (per lane) to l + 16 lane (l wave-uniform).
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)g,
                                     (__attribute__((address_space(3))) void *)l, 16, 0, 0);
}

// Row tiles per wave by k steps (registers), 16-row training tiles per stage.
constexpr int CTS = 4;
constexpr int rt_of(int ks) { return ks <= 2 ? 4 : 2; }
// The sweep. A wave holds RT tiles of 16 query rows in registers and takes the training rows of
// its segment 16 CTS at a time; their fragments are copied to LDS once for the workgroup's
// four waves, straight from memory, a step ahead (two buffers, one barrier a step). A tile's
// accumulators start at -A_x - B_y, so the sign of the result is the outcome, and one
// v_alignbit shifts it into the lane's word of the row: two vector operations per pair beside
// the products, no compare, no branch, no matter how many pairs hit. (With a branch per 64 x 64
// step that assembled words from ballots the kernel took 7.75 ms at 100,000 x 16, where nine
// steps in ten hold a hit; this form takes 1.8 ms, 0.55 PFLOP/s of products issued.)
//
// Bit order: a lane (r, g) sees columns 16 k + r of a row, so word [row][j / 512][j % 16] holds
// column j at bit 31 - (j % 512) / 16.
// Row block rb starts at row rb * rstep. Without bits only their number is left; with a probe above
// `most` nothing is done.
// Two waves per SIMD are asked for explicitly: with the whole register file to itself the
// compiler keeps the accumulators in accumulation registers and copies every element in and out.
template <int KS, int RT>
__global__ __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(2))) void radius_sweep_kernel(
    const _Float16 *__restrict__ PA, const _Float16 *__restrict__ PB,
    const float *__restrict__ A, const float *__restrict__ B, int nrb, int rstep, int nblk,
    int segblk, unsigned *__restrict__ bits, unsigned long long *total,
    const unsigned long long *probe, unsigned long long most) {
    constexpr int STAGE = CTS * KS * 1024; // fp16 elements of 16 CTS training rows
    __shared__ __attribute__((aligned(16))) _Float16 s0[STAGE];
    __shared__ __attribute__((aligned(16))) _Float16 s1[STAGE];
    if (probe && *probe > most)
        return;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int r = lane & 15, g = lane >> 4;
    // All row blocks of one segment first, so that the workgroups running at a time share it.
    const int segi = (int)blockIdx.x / nrb, rb = (int)blockIdx.x - segi * nrb;
    const int row0 = rb * rstep + w * RT * 16;
    const int b0 = segi * segblk, b1 = min(nblk, b0 + segblk);
    if (b0 >= b1)
        return;
    v8h a[RT][KS][2];
    float ax[RT][4];
    unsigned word[RT][4];
#pragma unroll
    for (int rt = 0; rt < RT; rt++) {
        const _Float16 *src = PA + (int64_t)(row0 / 16 + rt) * KS * 1024 + lane * 8;
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            a[rt][ks][0] = *reinterpret_cast<const v8h *>(src + ks * 1024);
            a[rt][ks][1] = *reinterpret_cast<const v8h *>(src + ks * 1024 + 512);
        }
#pragma unroll
        for (int i = 0; i < 4; i++) {
            ax[rt][i] = A[row0 + rt * 16 + 4 * g + i];
            word[rt][i] = 0;
        }
    }
    float hv[CTS];
    auto stage = [&](int j0, _Float16 *dst) {
        const _Float16 *src = PB + (int64_t)(j0 / 16) * KS * 1024;
#pragma unroll
        for (int b = 0; b < CTS / 2 * KS; b++) {
            const int blk = w * (CTS / 2 * KS) + b;
            copy_to_lds(src + blk * 512 + lane * 8, dst + blk * 512);
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
                const _Float16 *p = sb + (ct * KS + ks) * 1024 + lane * 8;
                const v8h bh = *reinterpret_cast<const v8h *>(p);
                const v8h bl = *reinterpret_cast<const v8h *>(p + 512);
#pragma unroll
                for (int rt = 0; rt < RT; rt++)
                    acc[rt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[rt][ks][0], bh, acc[rt], 0, 0, 0);
#pragma unroll
                for (int rt = 0; rt < RT; rt++)
                    acc[rt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[rt][ks][0], bl, acc[rt], 0, 0, 0);
#pragma unroll
                for (int rt = 0; rt < RT; rt++)
                    acc[rt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[rt][ks][1], bh, acc[rt], 0, 0, 0);
            }
#pragma unroll
            for (int rt = 0; rt < RT; rt++)
#pragma unroll
                for (int i = 0; i < 4; i++)
                    word[rt][i] = __builtin_amdgcn_alignbit(word[rt][i],
                                                            __float_as_uint(acc[rt][i]), 31);
        }
    };
    int set = 0;
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
            for (int i = 0; i < 4; i++) {
                const unsigned v = ~word[rt][i];
                if (bits)
                    bits[((int64_t)(row0 + rt * 16 + 4 * g + i) * nblk + blk) * 16 + r] = v;
                set += __popc(v);
            }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1)
        set += __shfl_xor(set, o, 64);
    if (lane == 0)
        atomicAdd(total, (unsigned long long)set);
}

// The key of a pair as the general path forms it.
template <typename T, int METRIC>
__device__ __forceinline__ T radius_key(const T *__restrict__ x, const T *__restrict__ y, int d,
                                        double nx, double ny) {
    double acc = 0.0;
    for (int l = 0; l < d; l++) {
        if constexpr (METRIC == KM_SQEUCLIDEAN_GEMM) {
            acc = fma((double)x[l], (double)y[l], acc);
        } else {
            const double t = (double)x[l] - (double)y[l];
            acc = fma(t, t, acc);
        }
    }
    if constexpr (METRIC == KM_EUCLIDEAN)
        acc = sqrt(acc);
    if constexpr (METRIC == KM_SQEUCLIDEAN_GEMM) {
        acc = nx + ny - 2.0 * acc;
        acc = acc < 0.0 ? 0.0 : acc;
    }
    return (T)acc;
}

// Words of a row per pass of a wave (64 lanes x 32 bits = 2,048 columns).
__device__ __forceinline__ int word_column(int word, int bit) {
    return (word >> 4) * 512 + (31 - bit) * 16 + (word & 15);
}

// One wave per row: the columns of its set bits are queued in LDS and their keys formed 64 at a
// time; bits whose key is above thr (or that are the row itself: column self0 + row) are cleared
// and cnt[row] is the number that remain.
template <typename T, int METRIC>
__global__ __launch_bounds__(256) void radius_verify_kernel(
    const T *__restrict__ X, const T *__restrict__ Y, int rows, int d,
    const double *__restrict__ nx, const double *__restrict__ ny, T thr, int self0, int nblk,
    unsigned *bits, int *__restrict__ cnt) {
    __shared__ int queue[4][2048 + 64];
    __shared__ int qcount[4];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int row = blockIdx.x * 4 + w;
    if (row >= rows)
        return;
    unsigned *b = bits + (int64_t)row * nblk * 16;
    const T *x = X + (int64_t)row * d;
    const double nxr = nx ? nx[row] : 0.0;
    const int self = self0 >= 0 ? self0 + row : -1;
    int *q = queue[w];
    int have = 0, count = 0;
    auto fence = [&]() {
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
    // Verifies entries [at, at + 64) of the queue.
    auto check = [&](int at) {
        bool pass = false;
        if (at + lane < have) {
            const int j = q[at + lane];
            pass = j != self &&
                   radius_key<T, METRIC>(x, Y + (int64_t)j * d, d, nxr, ny ? ny[j] : 0.0) <= thr;
            if (!pass) {
                const int wd = (j >> 9) * 16 + (j & 15);
                atomicAnd(&b[wd], ~(1u << (31 - ((j & 511) >> 4))));
            }
        }
        count += __popcll(__builtin_amdgcn_ballot_w64(pass));
    };
    const int nwords = nblk * 16;
    for (int w0 = 0; w0 < nwords; w0 += 256) {
        unsigned v[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int wd = w0 + u * 64 + lane;
            v[u] = wd < nwords ? b[wd] : 0u;
        }
#pragma unroll
        for (int u = 0; u < 4; u++) {
            if (__builtin_amdgcn_ballot_w64(v[u] != 0) == 0)
                continue;
            if (lane == 0)
                qcount[w] = have;
            fence();
            if (v[u]) {
                int p = atomicAdd(&qcount[w], __popc(v[u]));
                unsigned m = v[u];
                while (m) {
                    const int bit = 31 - __clz((int)m);
                    m &= ~(1u << bit);
                    q[p++] = word_column(w0 + u * 64 + lane, bit);
                }
            }
            fence();
            have = qcount[w];
            if (have >= 64) {
                int at = 0;
                for (; at + 64 <= have; at += 64)
                    check(at);
                // The rest (below 64) moves to the front.
                const int rest = have - at;
                const int keep = lane < rest ? q[at + lane] : 0;
                fence();
                if (lane < rest)
                    q[lane] = keep;
                have = rest;
                fence();
            }
        }
    }
    if (have > 0)
        check(0);
    if (lane == 0)
        cnt[row] = count;
}

// Indices of the set bits of every row, ascending, at offs[row]. One wave per row; the bits of
// 2,048 columns are put in column order through 32 words of LDS.
template <typename O>
__global__ __launch_bounds__(256) void radius_bits_fill_kernel(
    const unsigned *__restrict__ bits, int rows, int nblk, const O *__restrict__ offs,
    const int *__restrict__ cnt, int *__restrict__ ind) {
    __shared__ unsigned nat[4][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int row = blockIdx.x * 4 + w;
    if (row >= rows || cnt[row] == 0)
        return;
    const unsigned *b = bits + (int64_t)row * nblk * 16;
    const int nwords = nblk * 16;
    int64_t pos = (int64_t)offs[row];
    auto fence = [&]() {
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
    for (int w0 = 0; w0 < nwords; w0 += 256) {
        unsigned v[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int wd = w0 + u * 64 + lane;
            v[u] = wd < nwords ? b[wd] : 0u;
        }
#pragma unroll
        for (int u = 0; u < 4; u++) {
            if (__builtin_amdgcn_ballot_w64(v[u] != 0) == 0)
                continue;
            const int base = (w0 + u * 64) * 32; // first of the 2,048 columns
            nat[w][lane] = 0;
            fence();
            unsigned m = v[u];
            while (m) {
                const int bit = 31 - __clz((int)m);
                m &= ~(1u << bit);
                const int c = word_column(w0 + u * 64 + lane, bit) - base;
                atomicOr(&nat[w][c >> 5], 1u << (c & 31));
            }
            fence();
            unsigned x = nat[w][lane];
            const int mine = __popc(x);
            int incl = mine;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const int y = __shfl_up(incl, o, 64);
                if (lane >= o)
                    incl += y;
            }
            int64_t p = pos + incl - mine;
            while (x) {
                const int bit = __ffs((int)x) - 1;
                x &= x - 1;
                ind[p++] = base + lane * 32 + bit;
            }
            pos += __shfl(incl, 63, 64);
            fence();
        }
    }
}

// Keys of the listed neighbours: one wave per row, a lane per neighbour.
template <typename T, int METRIC>
__global__ __launch_bounds__(256) void radius_hit_keys_kernel(
    const T *__restrict__ X, const T *__restrict__ Y, int rows, int d,
    const double *__restrict__ nx, const double *__restrict__ ny, const int *__restrict__ offs,
    const int *__restrict__ ind, T *__restrict__ key) {
    const int lane = threadIdx.x & 63;
    const int row = blockIdx.x * 4 + (int)(threadIdx.x >> 6);
    if (row >= rows)
        return;
    const T *x = X + (int64_t)row * d;
    const int e = offs[row + 1];
    for (int p = offs[row] + lane; p < e; p += 64) {
        const int j = ind[p];
        key[p] = radius_key<T, METRIC>(x, Y + (int64_t)j * d, d, nx ? nx[row] : 0.0,
                                       ny ? ny[j] : 0.0);
    }
}


} // namespace

bool radius_bits_metric(int metric) {
    return metric == KM_SQEUCLIDEAN || metric == KM_EUCLIDEAN || metric == KM_SQEUCLIDEAN_GEMM;
}

RadiusPlan radius_plan(int d) {
    RadiusPlan p;
    p.ks = (d + 31) / 32;
    p.row_block = 64 * rt_of(p.ks);
    const double terms = 3.0 * 32 * p.ks + 8, u = 1.0 / 16777216.0;
    p.ce = terms * u / (1.0 - terms * u) + 1.0 / 524288.0;
    return p;
}

template <typename T>
hipError_t launch_radius_scale(const T *X, int64_t nx, const T *Y, int64_t ny, int d, int metric,
                               unsigned long long *range, RadiusScale *sc, hipStream_t s) {
    if (d < 1 || d > 128)
        return hipErrorInvalidValue;
    hipLaunchKernelGGL(radius_range_init_kernel, dim3(1), dim3(128), 0, s, range, d);
    for (int q = 0; q < 2; q++) {
        const T *p = q ? Y : X;
        const int64_t rows = q ? ny : nx;
        if (!p || rows <= 0)
            continue;
        const int64_t spp = 256 / d, blocks = std::min<int64_t>(512, (rows + spp - 1) / spp);
        hipLaunchKernelGGL(radius_range_kernel<T>, dim3((unsigned)blocks), dim3(256), 0, s, p,
                           rows, d, range);
    }
    hipLaunchKernelGGL(radius_scale_kernel, dim3(1), dim3(128), 0, s, range, d,
                       metric == KM_SQEUCLIDEAN_GEMM ? 1 : 0, sc);
    return hipGetLastError();
}

template <typename T>
hipError_t launch_radius_pack(const T *X, int rows, int rows_pad, int d, const RadiusPlan &p,
                              const RadiusScale *sc, double thr2, void *P, float *A, float *B,
                              hipStream_t s) {
    if (rows_pad % 16 != 0)
        return hipErrorInvalidValue;
    const int tiles = rows_pad / 16;
    hipLaunchKernelGGL(radius_pack_kernel<T>, dim3((tiles + 3) / 4), dim3(256), 0, s, X, rows,
                       tiles, d, p.ks, sc, thr2, p.ce, static_cast<_Float16 *>(P), A, B);
    return hipGetLastError();
}

static hipError_t radius_sweep(const RadiusPlan &p, const void *PA, int nrb, int rstep,
                               const void *PB, int n_pad, int segblk, const float *A,
                               const float *B, unsigned *bits, unsigned long long *total,
                               const unsigned long long *probe, unsigned long long most,
                               hipStream_t s) {
    const int nblk = n_pad / 512, nseg = (nblk + segblk - 1) / segblk;
    const _Float16 *pa = static_cast<const _Float16 *>(PA), *pb = static_cast<const _Float16 *>(PB);
#define DA_SWEEP(K)                                                                              \
    case K:                                                                                      \
        hipLaunchKernelGGL((radius_sweep_kernel<K, rt_of(K)>), dim3((unsigned)nrb * nseg),       \
                           dim3(256), 0, s, pa, pb, A, B, nrb, rstep, nblk, segblk, bits,        \
                           total, probe, most);                                                  \
        break;
    switch (p.ks) {
        DA_SWEEP(1)
        DA_SWEEP(2)
        DA_SWEEP(3)
        DA_SWEEP(4)
    default:
        return hipErrorInvalidValue;
    }
#undef DA_SWEEP
    return hipGetLastError();
}

hipError_t launch_radius_sweep(const RadiusPlan &p, const void *PA, int rows_pad, const void *PB,
                               int n_pad, const float *A, const float *B, unsigned *bits,
                               RadiusScale *sc, unsigned long long most, hipStream_t s) {
    if (rows_pad % p.row_block != 0 || n_pad % 512 != 0 || !bits)
        return hipErrorInvalidValue;
    const int nblk = n_pad / 512;
    const int nrb = rows_pad / p.row_block;
    // Column segments: about 1,024 workgroups (two run on a CU at a time), each of at least 1,024
    // training rows: a workgroup's start (its query rows) and end cost a few steps. 10,000 x
    // 100,000 pairs of 16 features: 222 us with 4,096 workgroups, 177 us with 512 to 2,048.
    const int nseg = std::max(1, std::min((nblk + 1) / 2, (1024 + nrb - 1) / nrb));
    return radius_sweep(p, PA, nrb, p.row_block, PB, n_pad, (nblk + nseg - 1) / nseg, A, B, bits,
                        &sc->total, &sc->probe, most, s);
}

// Four row blocks alone leave most CUs idle, so here the segments are short.
hipError_t launch_radius_probe(const RadiusPlan &p, const void *PA, int rows, const void *PB,
                               int n_pad, const float *A, const float *B, RadiusScale *sc,
                               hipStream_t s) {
    if (rows < radius_probe_rows(p) || n_pad % 512 != 0)
        return hipErrorInvalidValue;
    const int segblk = std::max(1, n_pad / 512 / 256);
    return radius_sweep(p, PA, 4, rows / 4 / p.row_block * p.row_block, PB, n_pad, segblk, A, B,
                        nullptr, &sc->probe, nullptr, 0, s);
}

template <typename T>
hipError_t launch_radius_verify(int metric, const T *X, const T *Y, int rows, int d,
                                const double *nx, const double *ny, T thr, int self0, int n_pad,
                                unsigned *bits, int *cnt, hipStream_t s) {
    if (rows <= 0)
        return hipSuccess;
    auto kern = metric == KM_EUCLIDEAN         ? radius_verify_kernel<T, KM_EUCLIDEAN>
                : metric == KM_SQEUCLIDEAN_GEMM ? radius_verify_kernel<T, KM_SQEUCLIDEAN_GEMM>
                                                : radius_verify_kernel<T, KM_SQEUCLIDEAN>;
    hipLaunchKernelGGL(kern, dim3((rows + 3) / 4), dim3(256), 0, s, X, Y, rows, d, nx, ny, thr,
                       self0, n_pad / 512, bits, cnt);
    return hipGetLastError();
}

template <typename O>
hipError_t launch_radius_bits_fill(const unsigned *bits, int rows, int n_pad, const O *offs,
                                   const int *cnt, int *ind, hipStream_t s) {
    if (rows <= 0)
        return hipSuccess;
    hipLaunchKernelGGL(radius_bits_fill_kernel<O>, dim3((rows + 3) / 4), dim3(256), 0, s, bits,
                       rows, n_pad / 512, offs, cnt, ind);
    return hipGetLastError();
}
template hipError_t launch_radius_bits_fill<int>(const unsigned *, int, int, const int *,
                                                 const int *, int *, hipStream_t);
template hipError_t launch_radius_bits_fill<long long>(const unsigned *, int, int,
                                                       const long long *, const int *, int *,
                                                       hipStream_t);

template <typename T>
hipError_t launch_radius_hit_keys(int metric, const T *X, const T *Y, int rows, int d,
                                  const double *nx, const double *ny, const int *offs,
                                  const int *ind, T *key, hipStream_t s) {
    if (rows <= 0)
        return hipSuccess;
    auto kern = metric == KM_EUCLIDEAN         ? radius_hit_keys_kernel<T, KM_EUCLIDEAN>
                : metric == KM_SQEUCLIDEAN_GEMM ? radius_hit_keys_kernel<T, KM_SQEUCLIDEAN_GEMM>
                                                : radius_hit_keys_kernel<T, KM_SQEUCLIDEAN>;
    hipLaunchKernelGGL(kern, dim3((rows + 3) / 4), dim3(256), 0, s, X, Y, rows, d, nx, ny, offs,
                       ind, key);
    return hipGetLastError();
}

#define DA_RM_INST(T)                                                                            \
    template hipError_t launch_radius_scale<T>(const T *, int64_t, const T *, int64_t, int, int, \
                                               unsigned long long *, RadiusScale *,              \
                                               hipStream_t);                                     \
    template hipError_t launch_radius_pack<T>(const T *, int, int, int, const RadiusPlan &,      \
                                              const RadiusScale *, double, void *, float *,      \
                                              float *, hipStream_t);                             \
    template hipError_t launch_radius_verify<T>(int, const T *, const T *, int, int,             \
                                                const double *, const double *, T, int, int,     \
                                                unsigned *, int *, hipStream_t);                 \
    template hipError_t launch_radius_hit_keys<T>(int, const T *, const T *, int, int,           \
                                                  const double *, const double *, const int *,   \
                                                  const int *, T *, hipStream_t);
DA_RM_INST(float)
DA_RM_INST(double)
#undef DA_RM_INST

} // namespace dagpu
