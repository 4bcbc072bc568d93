// Per-row k-smallest selection over a materialised key matrix.
//
// The reference selects with a "replace the current maximum" scan per query followed by
// a stable sort (source/core/nearest_neighbors/nearest_neighbors_utils.hpp:44-101). On the
// GPU one workgroup owns one row: each element is compared with a running threshold (the
// k-th best (key, index) pair kept so far) and, when it beats it, appended to an LDS
// candidate buffer with an LDS atomic. When the buffer is close to full the workgroup
// bitonic-sorts it, keeps the k best and tightens the threshold. Elements are ordered by
// (key, column index), so the result is deterministic, including at equal keys.
#include "launch.hpp"
#include <algorithm>
#include <climits>
#include <hip/hip_runtime.h>

namespace dagpu {

namespace {

template <typename K> __device__ __forceinline__ bool pair_less(K ka, int ia, K kb, int ib) {
    return ka < kb || (ka == kb && ia < ib);
}

// Sorts bkey/bidx[0..CAP) ascending by (key, index). All threads of the block must call.
template <typename K, int CAP>
__device__ void block_bitonic_sort(K *bkey, int *bidx) {
    for (int size = 2; size <= CAP; size <<= 1) {
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
            for (int t = threadIdx.x; t < CAP / 2; t += blockDim.x) {
                const int i = 2 * t - (t & (stride - 1));
                const int j = i + stride;
                const bool asc = (i & size) == 0;
                K ki = bkey[i], kj = bkey[j];
                int ii = bidx[i], ij = bidx[j];
                const bool gt = pair_less(kj, ij, ki, ii);
                if (gt == asc) {
                    bkey[i] = kj;
                    bkey[j] = ki;
                    bidx[i] = ij;
                    bidx[j] = ii;
                }
            }
            __syncthreads();
        }
    }
}

// The k smallest of rk[0..n), by (key, column), to out_key / out_idx (columns from c0 on).
// bkey, bidx: CAP entries of LDS. All threads of the block must call.
template <typename K, int CAP>
__device__ void row_select(const K *__restrict__ rk, int n, int k, int largest, int c0, K *bkey,
                           int *bidx, K *__restrict__ out_key, int *__restrict__ out_idx) {
    __shared__ int count;
    __shared__ K thr_k;
    __shared__ int thr_i;
    const K inf = (K)__builtin_huge_val();
    if (threadIdx.x == 0) {
        count = 0;
        thr_k = inf;
        thr_i = INT_MAX;
    }
    __syncthreads();
    for (int base = 0; base < n; base += 256) {
        const int j = base + threadIdx.x;
        if (j < n) {
            K v = rk[j];
            if (largest)
                v = -v;
            if (v != v)
                v = inf;
            if (pair_less(v, j, thr_k, thr_i)) {
                const int pos = atomicAdd(&count, 1);
                bkey[pos] = v;
                bidx[pos] = j;
            }
        }
        __syncthreads();
        const int c = count;
        // Every thread must read the count before any thread appends again.
        __syncthreads();
        if (c > CAP - 256) {
            for (int t = c + threadIdx.x; t < CAP; t += blockDim.x) {
                bkey[t] = inf;
                bidx[t] = INT_MAX;
            }
            __syncthreads();
            block_bitonic_sort<K, CAP>(bkey, bidx);
            if (threadIdx.x == 0) {
                count = c < k ? c : k;
                if (c >= k) {
                    thr_k = bkey[k - 1];
                    thr_i = bidx[k - 1];
                }
            }
            __syncthreads();
        }
    }
    const int c = count;
    for (int t = c + threadIdx.x; t < CAP; t += blockDim.x) {
        bkey[t] = inf;
        bidx[t] = INT_MAX;
    }
    __syncthreads();
    block_bitonic_sort<K, CAP>(bkey, bidx);
    for (int t = threadIdx.x; t < k; t += blockDim.x) {
        K v = bkey[t];
        out_key[t] = largest ? -v : v;
        out_idx[t] = bidx[t] == INT_MAX ? INT_MAX : c0 + bidx[t];
    }
}

template <typename K, int CAP>
__global__ __launch_bounds__(256) void row_topk_kernel(const K *__restrict__ keys, int64_t ld,
                                                       int n, int k, int largest,
                                                       K *__restrict__ out_key,
                                                       int *__restrict__ out_idx) {
    __shared__ K bkey[CAP];
    __shared__ int bidx[CAP];
    const int64_t row = blockIdx.x;
    row_select<K, CAP>(keys + row * ld, n, k, largest, 0, bkey, bidx, out_key + row * k,
                       out_idx + row * k);
}

} // namespace

namespace {

// The same selection for k <= 128: thread t keeps the smallest of elements t, t + 256, ..., and
// the k-th smallest of the 256 group minima, attained by k elements of the row, bounds the k-th
// key from above. A second pass collects the elements at or below it, -256 ln(1 - k / 256) on
// average (5 for k = 5, 127 for k = 100), and one sort of those ends the row: two barriers-free
// sweeps instead of two barriers per 256 elements and a 512-entry sort whenever the buffer fills.
// Rows with more than SEL_CAP elements at or below the bound (ties) are selected from by the
// general way, in the same launch (a launch of its own behind this one: 5 us of a small search).
// Segment blockIdx.y of `seg` columns (the whole row when there is one); the results of
// (row, segment) pairs lie one after another.
constexpr int SEL_CAP = 1024;
template <typename K>
__global__ __launch_bounds__(256) void row_topk_bound_kernel(const K *__restrict__ keys,
                                                             int64_t ld, int n, int k,
                                                             int largest, K *__restrict__ out_key,
                                                             int *__restrict__ out_idx, int seg) {
    __shared__ K bkey[SEL_CAP];
    __shared__ int bidx[SEL_CAP];
    __shared__ int count;
    __shared__ K bound;
    const K inf = (K)__builtin_huge_val();
    const int tid = threadIdx.x;
    const int64_t o = ((int64_t)blockIdx.x * gridDim.y + blockIdx.y) * k;
    const int c0 = (int)blockIdx.y * seg;
    const K *rk = keys + (int64_t)blockIdx.x * ld + c0;
    n = n - c0 < seg ? n - c0 : seg;
    auto value = [&](K v) {
        v = largest ? -v : v;
        return v != v ? inf : v;
    };
    K mn = inf;
    int j = tid;
    for (; j + 7 * 256 < n; j += 8 * 256) {
        K v[8];
#pragma unroll
        for (int u = 0; u < 8; u++)
            v[u] = rk[j + u * 256];
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const K x = value(v[u]);
            mn = x < mn ? x : mn;
        }
    }
    for (; j < n; j += 256) {
        const K x = value(rk[j]);
        mn = x < mn ? x : mn;
    }
    // The k-th smallest minimum: the one with rank k - 1 (ties by thread).
    bkey[tid] = mn;
    if (tid == 0)
        count = 0;
    __syncthreads();
    int rank = 0;
#pragma unroll 8
    for (int t = 0; t < 256; t++) {
        const K o = bkey[t];
        rank += o < mn || (o == mn && t < tid);
    }
    if (rank == k - 1)
        bound = mn;
    __syncthreads();
    const K bd = bound;
    __syncthreads();
    auto take = [&](K x, int jj) {
        if (x <= bd) {
            const int p = atomicAdd(&count, 1);
            if (p < SEL_CAP) {
                bkey[p] = x;
                bidx[p] = jj;
            }
        }
    };
    j = tid;
    for (; j + 7 * 256 < n; j += 8 * 256) {
        K v[8];
#pragma unroll
        for (int u = 0; u < 8; u++)
            v[u] = rk[j + u * 256];
#pragma unroll
        for (int u = 0; u < 8; u++)
            take(value(v[u]), j + u * 256);
    }
    for (; j < n; j += 256)
        take(value(rk[j]), j);
    __syncthreads();
    const int c = count;
    if (c > SEL_CAP) {
        row_select<K, 512>(rk, n, k, largest, c0, bkey, bidx, out_key + o, out_idx + o);
        return;
    }
    int cap = 2;
    while (cap < c || cap < k)
        cap <<= 1;
    for (int t = c + tid; t < cap; t += 256) {
        bkey[t] = inf;
        bidx[t] = INT_MAX;
    }
    __syncthreads();
    for (int size = 2; size <= cap; size <<= 1) {
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
            for (int t = tid; t < cap / 2; t += 256) {
                const int a = 2 * t - (t & (stride - 1));
                const int b = a + stride;
                const bool asc = (a & size) == 0;
                const K ka = bkey[a], kb = bkey[b];
                const int ia = bidx[a], ib = bidx[b];
                if (pair_less(kb, ib, ka, ia) == asc) {
                    bkey[a] = kb;
                    bkey[b] = ka;
                    bidx[a] = ib;
                    bidx[b] = ia;
                }
            }
            __syncthreads();
        }
    }
    for (int t = tid; t < k; t += 256) {
        const K v = bkey[t];
        out_key[o + t] = largest ? -v : v;
        out_idx[o + t] = bidx[t] == INT_MAX ? INT_MAX : c0 + bidx[t];
    }
}

// idx[e] = cols[row of e][idx[e]]: the columns behind the positions of a second selection.
__global__ void row_topk_map_kernel(int *__restrict__ idx, const int *__restrict__ cols, int rows,
                                    int k, int width) {
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= (int64_t)rows * k)
        return;
    const int p = idx[e];
    if (p != INT_MAX)
        idx[e] = cols[e / k * width + p];
}

} // namespace

// The selection over (row, segment) pairs: rows x nseg results of k (segments only for k <= 128).
template <typename K>
static hipError_t topk_level(const K *keys, int64_t ld, int rows, int n, int k, int largest,
                             K *out_key, int *out_idx, int seg, int nseg, hipStream_t s) {
    dim3 grid(rows, nseg), block(256);
    if (k <= 128) {
        hipLaunchKernelGGL(row_topk_bound_kernel<K>, grid, block, 0, s, keys, ld, n, k, largest,
                           out_key, out_idx, seg);
        return hipGetLastError();
    }
    auto kern = k + 256 <= 512    ? row_topk_kernel<K, 512>
                : k + 256 <= 1024 ? row_topk_kernel<K, 1024>
                : k + 256 <= 2048 ? row_topk_kernel<K, 2048>
                                  : row_topk_kernel<K, 4096>;
    hipLaunchKernelGGL(kern, dim3(rows), block, 0, s, keys, ld, n, k, largest, out_key, out_idx);
    return hipGetLastError();
}

// Few long rows (one workgroup each would leave the chip idle: a row of 2,000,000 keys takes one
// workgroup some 2 ms) are cut into segments of 8,192 columns or more, about 1,024 workgroups in
// all, each segment's k best selected, then the best of those.
int row_topk_segments(int rows, int n, int k) {
    if (k > 128 || rows >= 512 || n < 32768)
        return 1;
    return std::max(1, std::min({n / 8192, 1024 / rows, 256}));
}

template <typename K>
hipError_t launch_row_topk(const K *keys, int64_t ld, int rows, int n, int k, int largest,
                           K *out_key, int *out_idx, hipStream_t s, K *tmp_key, int *tmp_idx) {
    if (k < 1 || k > 3840 || rows < 1)
        return hipErrorInvalidValue;
    const int want = tmp_key && tmp_idx ? row_topk_segments(rows, n, k) : 1;
    if (want <= 1)
        return topk_level<K>(keys, ld, rows, n, k, largest, out_key, out_idx, n, 1, s);
    const int seg = (n + want - 1) / want, nseg = (n + seg - 1) / seg;
    hipError_t e = topk_level<K>(keys, ld, rows, n, k, largest, tmp_key, tmp_idx, seg, nseg, s);
    if (e != hipSuccess)
        return e;
    // Among equal keys the earlier segment and, within it, the earlier column come first, so the
    // order of the positions is that of the columns.
    e = topk_level<K>(tmp_key, (int64_t)nseg * k, rows, nseg * k, k, largest, out_key, out_idx,
                      nseg * k, 1, s);
    if (e != hipSuccess)
        return e;
    hipLaunchKernelGGL(row_topk_map_kernel, dim3((unsigned)(((int64_t)rows * k + 255) / 256)),
                       dim3(256), 0, s, out_idx, tmp_idx, rows, k, nseg * k);
    return hipGetLastError();
}

template hipError_t launch_row_topk<float>(const float *, int64_t, int, int, int, int, float *,
                                           int *, hipStream_t, float *, int *);
template hipError_t launch_row_topk<double>(const double *, int64_t, int, int, int, int,
                                            double *, int *, hipStream_t, double *, int *);

} // namespace dagpu

namespace dagpu {
namespace {
template <typename T>
__global__ void knn_finalize_kernel(const double *__restrict__ keys, const int *__restrict__ idx,
                                    int rows, int k, int post, double p, T *__restrict__ out_dist,
                                    int *__restrict__ out_idx, int64_t ldo) {
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= (int64_t)rows * k)
        return;
    const int64_t q = e / k, j = e - q * k;
    double v = keys[e];
    if (post == 1)
        v = sqrt(v < 0.0 ? 0.0 : v);
    else if (post == 2)
        v = pow(v, 1.0 / p);
    if (out_dist)
        out_dist[q * ldo + j] = (T)v;
    out_idx[q * ldo + j] = idx[e];
}
} // namespace

template <typename T>
hipError_t launch_knn_finalize(const double *keys, const int *idx, int rows, int k, int post,
                               double p, T *out_dist, int *out_idx, int64_t ldo,
                               hipStream_t s) {
    const int64_t total = (int64_t)rows * k;
    hipLaunchKernelGGL(knn_finalize_kernel<T>, dim3((unsigned)((total + 255) / 256)), dim3(256),
                       0, s, keys, idx, rows, k, post, p, out_dist, out_idx, ldo);
    return hipGetLastError();
}
template hipError_t launch_knn_finalize<float>(const double *, const int *, int, int, int,
                                               double, float *, int *, int64_t, hipStream_t);
template hipError_t launch_knn_finalize<double>(const double *, const int *, int, int, int,
                                                double, double *, int *, int64_t, hipStream_t);
} // namespace dagpu

namespace dagpu {
namespace {
template <typename E>
__global__ void gather_scatter_kernel(const E *__restrict__ src, E *__restrict__ dst,
                                      const int *__restrict__ idx, int m, int cols, int scatter) {
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= (int64_t)m * cols)
        return;
    const int64_t i = e / cols, c = e - i * cols;
    const int64_t row = idx[i];
    if (scatter)
        dst[row * cols + c] = src[i * cols + c];
    else
        dst[i * cols + c] = src[row * cols + c];
}
} // namespace
hipError_t launch_gather_scatter(const void *src, void *dst, const int *idx, int m, int cols,
                                 int elem, int scatter, hipStream_t s) {
    const int64_t total = (int64_t)m * cols;
    dim3 grid((unsigned)((total + 255) / 256)), block(256);
    if (elem == 8)
        hipLaunchKernelGGL(gather_scatter_kernel<long long>, grid, block, 0, s,
                           static_cast<const long long *>(src), static_cast<long long *>(dst), idx,
                           m, cols, scatter);
    else
        hipLaunchKernelGGL(gather_scatter_kernel<int>, grid, block, 0, s,
                           static_cast<const int *>(src), static_cast<int *>(dst), idx, m, cols,
                           scatter);
    return hipGetLastError();
}
} // namespace dagpu
