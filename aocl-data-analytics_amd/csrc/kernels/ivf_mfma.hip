// IVF-Flat search on the fp16 matrix cores of gfx950: list by list instead of query by query.
//
// A scan per (query, probe) reads a list once for each query that probes it and forms every key in
// double. Here the queries of a block are grouped by probed list; a workgroup takes up to 128 of a
// list's queries and a run of its vectors, held as hi + lo fp16 tiles (layout, scores and error
// bound E as in knn_wide.hip), and writes approximate scores into each query's row at the probed
// list's columns (lists ascending, each padded to 16 columns of +inf). The selection bounds the
// k-th score of a row from above, collects what lies within 2 E of the bound, and orders those by
// their exact keys, summed and rounded as the scan does: (key, column) decides there as here, so the
// results are the scan's in every case. A query whose collection overflows or whose values leave
// fp16's range is listed for the scan.
#include "ivf_keys.hpp"
#include "launch.hpp"
#include "wave_rank.hpp"
#include <algorithm>
#include <climits>
#include <hip/hip_runtime.h>

namespace dagpu {

namespace {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));

// One wave per query: its probes in ascending list number, their first columns and its place in
// each list's group.
__global__ __launch_bounds__(256) void ivf_place_kernel(IvfTiles p, const int *__restrict__ probes,
                                                        int nq) {
    const int q = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (q >= nq)
        return;
    const int np = p.n_probe;
    const int *pr = probes + (int64_t)q * np;
    for (int a = lane; a < np; a += 64) {
        const int c = pr[a];
        int rank = 0, start = 0;
        for (int o = 0; o < np; o++) {
            const int co = pr[o];
            if (co < c) {
                rank++;
                start += p.tile_off[co + 1] - p.tile_off[co];
            }
        }
        const int64_t at = (int64_t)q * np + rank;
        p.slist[at] = c;
        p.sseg[at] = start * 16;
        p.place[at] = atomicAdd(&p.cnt[c], 1);
        if (rank == np - 1)
            p.rowlen[q] = (start + p.tile_off[c + 1] - p.tile_off[c]) * 16;
    }
}

// Vectors of each list's operand rows, -1 for padding.
__global__ __launch_bounds__(256) void ivf_map_kernel(const int *__restrict__ perm,
                                                      const int *__restrict__ list_off,
                                                      const int *__restrict__ tile_off,
                                                      int *__restrict__ map) {
    const int c = blockIdx.x;
    const int b = list_off[c], n = list_off[c + 1] - b, t0 = tile_off[c];
    const int rows = (tile_off[c + 1] - t0) * 16;
    for (int i = threadIdx.x; i < rows; i += 256)
        map[(int64_t)t0 * 16 + i] = i < n ? perm[b + i] : -1;
}

__global__ __launch_bounds__(1024) void ivf_zero_kernel(int *cnt, int n) {
    for (int c = threadIdx.x; c < n; c += 1024)
        cnt[c] = 0;
}

// One workgroup: group offsets, and a work item per 128 queries of a list.
__global__ __launch_bounds__(1024) void ivf_items_kernel(IvfTiles p) {
    __shared__ int a[1024], b[1024];
    const int t = threadIdx.x;
    int ca = 0, cb = 0;
    for (int c0 = 0; c0 < p.n_list; c0 += 1024) {
        const int c = c0 + t;
        const int n = c < p.n_list ? p.cnt[c] : 0;
        const int tiles = c < p.n_list ? p.tile_off[c + 1] - p.tile_off[c] : 0;
        const int w = tiles > 0 ? (n + 127) / 128 : 0;
        a[t] = n;
        b[t] = w;
        __syncthreads();
        for (int o = 1; o < 1024; o <<= 1) {
            const int x = t >= o ? a[t - o] : 0, y = t >= o ? b[t - o] : 0;
            __syncthreads();
            a[t] += x;
            b[t] += y;
            __syncthreads();
        }
        if (c < p.n_list) {
            p.qoff[c] = ca + a[t] - n;
            for (int i = 0; i < w; i++)
                p.items[cb + b[t] - w + i] = make_int2(c, i);
        }
        ca += a[1023];
        cb += b[1023];
        __syncthreads();
    }
    if (t == 0)
        *p.n_items = cb;
}

__global__ __launch_bounds__(256) void ivf_group_kernel(IvfTiles p, int64_t pairs) {
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (t < pairs)
        p.group[p.qoff[p.slist[t]] + p.place[t]] = (int)t;
}

// Scores. Each wave holds 32 queries' fragments (hi, lo, all k steps) in registers; a list's tiles
// pass through LDS two at a time, copied straight there one step ahead (two buffers, one barrier
// per step). The list vectors are the rows of the product, so a lane holds four consecutive
// columns of one query: a store instruction writes 64 contiguous bytes for each of 16 queries.
// Bound by the score stores: 4 bytes a pair against 6 d operations. With the selection below
// 10,000 queries, 16 of 1,024 lists of 1,000,000 x 96 fp32 take 1.4 ms (scans and row selection: 28).
constexpr int IVF_RUN = 16; // tiles per workgroup and pass

template <int KS>
__global__ __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(2))) void ivf_scores_kernel(IvfTiles p,
                                                               const _Float16 *__restrict__ QP,
                                                               float *__restrict__ out,
                                                               int64_t ld) {
    __shared__ __attribute__((aligned(16))) _Float16 s0[2 * KS * 1024];
    __shared__ __attribute__((aligned(16))) _Float16 s1[2 * KS * 1024];
    if ((int)blockIdx.x >= *p.n_items)
        return;
    const int2 it = p.items[blockIdx.x];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int r = lane & 15, g = lane >> 4;
    const int c = it.x, t0 = p.tile_off[c], tiles = p.tile_off[c + 1] - t0;
    if ((int)blockIdx.y * IVF_RUN >= tiles)
        return;
    const int nq = p.cnt[c], first = it.y * 128 + w * 32;
    const bool live = first < nq; // wave-uniform
    v8h x[2][KS][2];
    float *dst[2];
    bool on[2];
#pragma unroll
    for (int rt = 0; rt < 2; rt++) {
        const int place = first + rt * 16 + r;
        on[rt] = place < nq;
        const int pair = p.group[p.qoff[c] + min(place, nq - 1)];
        const int q = pair / p.n_probe;
        dst[rt] = out + (int64_t)q * ld + p.sseg[pair] + g * 4;
        const _Float16 *src = QP + (int64_t)q * KS * 64 + g * 8;
#pragma unroll
        for (int ks = 0; ks < KS; ks++)
#pragma unroll
            for (int hf = 0; hf < 2; hf++)
                x[rt][ks][hf] = *reinterpret_cast<const v8h *>(src + ks * 64 + hf * 32);
    }
    const _Float16 *op = static_cast<const _Float16 *>(p.op);
    for (int b0 = blockIdx.y * IVF_RUN; b0 < tiles; b0 += gridDim.y * IVF_RUN) {
        const int be = min(b0 + IVF_RUN, tiles);
        // Two tiles are 4 KS blocks of 1 KB; the last tile of an odd run is read twice.
        auto stage = [&](int b, _Float16 *s) {
#pragma unroll
            for (int i = 0; i < KS; i++) {
                const int blk = w * KS + i, tile = blk / (2 * KS);
                const _Float16 *src = op + (int64_t)(t0 + min(b + tile, be - 1)) * KS * 1024 +
                                      (blk - tile * 2 * KS) * 512 + lane * 8;
                __builtin_amdgcn_global_load_lds(
                    (const __attribute__((address_space(1))) void *)src,
                    (__attribute__((address_space(3))) void *)(s + blk * 512), 16, 0, 0);
            }
        };
        auto compute = [&](int b, const _Float16 *s) {
#pragma unroll
            for (int tt = 0; tt < 2; tt++) {
                if (b + tt >= be)
                    break;
                const float4 hv = *reinterpret_cast<const float4 *>(
                    p.h + (int64_t)(t0 + b + tt) * 16 + g * 4);
                v4f acc[2];
                acc[0] = acc[1] = v4f{-hv.x, -hv.y, -hv.z, -hv.w};
#pragma unroll
                for (int ks = 0; ks < KS; ks++) {
                    const _Float16 *f = s + (tt * KS + ks) * 1024 + lane * 8;
                    const v8h yh = *reinterpret_cast<const v8h *>(f);
                    const v8h yl = *reinterpret_cast<const v8h *>(f + 512);
#pragma unroll
                    for (int rt = 0; rt < 2; rt++)
                        acc[rt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(yh, x[rt][ks][0], acc[rt], 0, 0, 0);
#pragma unroll
                    for (int rt = 0; rt < 2; rt++)
                        acc[rt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(yh, x[rt][ks][1], acc[rt], 0, 0, 0);
#pragma unroll
                    for (int rt = 0; rt < 2; rt++)
                        acc[rt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(yl, x[rt][ks][0], acc[rt], 0, 0, 0);
                }
#pragma unroll
                for (int rt = 0; rt < 2; rt++)
                    if (on[rt])
                        *reinterpret_cast<v4f *>(dst[rt] + (b + tt) * 16) = -acc[rt];
            }
        };
        stage(b0, s0);
        for (int b = b0; b < be; b += 4) {
            __builtin_amdgcn_s_waitcnt(0x0F70); // vmcnt(0): this wave's copies have landed
            __syncthreads();
            if (b + 2 < be)
                stage(b + 2, s1);
            if (live)
                compute(b, s0);
            if (b + 2 < be) {
                __builtin_amdgcn_s_waitcnt(0x0F70);
                __syncthreads();
                if (b + 4 < be)
                    stage(b + 4, s0);
                if (live)
                    compute(b + 2, s1);
            }
        }
        __syncthreads(); // the next run refills the buffers
    }
}

// One workgroup per query. The k-th smallest of the 256 threads' minima is at least the k-th
// smallest score; with fewer than k non-empty threads the row is collected whole. Bound by the two passes over the row, the second of them out of the caches.
constexpr int IVF_KEEP = 1024;

template <typename T, bool IP>
__global__ __launch_bounds__(256) void ivf_tile_select_kernel(
    IvfTiles p, const float *__restrict__ scores, int64_t ld, const float *__restrict__ err,
    const T *__restrict__ Q, const T *__restrict__ X, int d, int k, int post, int q0,
    T *__restrict__ dist, int *__restrict__ ind, int *__restrict__ fb_count,
    int *__restrict__ fb_list) {
    __shared__ __attribute__((aligned(16))) float mins[256];
    __shared__ float bound;
    __shared__ int kept;
    __shared__ T xk[IVF_KEEP];
    __shared__ int col[IVF_KEEP], id[IVF_KEEP];
    const int q = blockIdx.x, t = threadIdx.x;
    const float E = err[q];
    const int len = p.rowlen[q], nv = len / 4;
    const float4 *row = reinterpret_cast<const float4 *>(scores + (int64_t)q * ld);
    if (!(E < __builtin_huge_valf())) {
        if (t == 0)
            fb_list[atomicAdd(fb_count, 1)] = q0 + q;
        return;
    }
    float m = __builtin_huge_valf();
#pragma unroll 8
    for (int i = t; i < nv; i += 256) {
        const float4 v = row[i];
        m = fminf(m, fminf(fminf(v.x, v.y), fminf(v.z, v.w)));
    }
    mins[t] = m;
    if (t == 0)
        kept = 0;
    __syncthreads();
    if (t < 64) {
        const float4 m4 = reinterpret_cast<const float4 *>(mins)[t];
        const float v[4] = {m4.x, m4.y, m4.z, m4.w};
        const float kth = wave_rank_256(v, k);
        if (t == 0)
            bound = __double2float_ru((double)kth + 2.0 * (double)E);
    }
    __syncthreads();
    const float lim = bound;
    auto take = [&](float v, int c) {
        if (v <= lim && v < __builtin_huge_valf()) { // not the padding
            const int at = atomicAdd(&kept, 1);
            if (at < IVF_KEEP)
                col[at] = c;
        }
    };
#pragma unroll 4
    for (int i = t; i < nv; i += 256) {
        const float4 v = row[i];
        if (fminf(fminf(v.x, v.y), fminf(v.z, v.w)) <= lim) {
            take(v.x, 4 * i);
            take(v.y, 4 * i + 1);
            take(v.z, 4 * i + 2);
            take(v.w, 4 * i + 3);
        }
    }
    __syncthreads();
    const int nc = kept;
    if (nc > IVF_KEEP) {
        if (t == 0)
            fb_list[atomicAdd(fb_count, 1)] = q0 + q;
        return;
    }
    // Columns -> vectors: the last probed list that starts at or before the column (an empty list
    // starts where the next one does).
    for (int i = t; i < nc; i += 256) {
        const int *seg = p.sseg + (int64_t)q * p.n_probe;
        int lo = 0, hi = p.n_probe - 1;
        while (lo < hi) {
            const int mid = (lo + hi + 1) / 2;
            if (seg[mid] <= col[i])
                lo = mid;
            else
                hi = mid - 1;
        }
        const int c = p.slist[(int64_t)q * p.n_probe + lo];
        id[i] = p.map[(int64_t)p.tile_off[c] * 16 + col[i] - seg[lo]];
    }
    __syncthreads();
    // Exact keys, summed as the scans sum them.
    const T *qv = Q + (int64_t)q * d;
    if (ivf_chunked<T>(d)) {
        using CT = Chunk16<T>;
        using ch_t = typename CT::type;
        constexpr int G = 8;
        const int dc = d / (16 / (int)sizeof(T)), sub = t & (G - 1);
        for (int i = t / G; i < nc; i += 256 / G) {
            const int j = id[i];
            double acc = 0.0;
            const ch_t *a = reinterpret_cast<const ch_t *>(qv);
            const ch_t *b = reinterpret_cast<const ch_t *>(X + (int64_t)j * d);
            for (int ch = sub; ch < dc; ch += G) {
                if constexpr (IP)
                    CT::dot(acc, a[ch], b[ch]);
                else
                    CT::acc(acc, a[ch], b[ch]);
            }
#pragma unroll
            for (int o = G / 2; o > 0; o >>= 1)
                acc += __shfl_xor(acc, o, G);
            if (sub == 0)
                xk[i] = (T)(IP ? -acc : acc);
        }
    } else {
        constexpr int G = 16;
        const int sub = t & (G - 1);
        for (int i = t / G; i < nc; i += 256 / G) {
            const int j = id[i];
            double acc = 0.0;
            const T *b = X + (int64_t)j * d;
            for (int l = sub; l < d; l += G) {
                if constexpr (IP) {
                    acc += (double)qv[l] * (double)b[l];
                } else {
                    const double u = (double)qv[l] - (double)b[l];
                    acc += u * u;
                }
            }
#pragma unroll
            for (int o = G / 2; o > 0; o >>= 1)
                acc += __shfl_xor(acc, o, G);
            if (sub == 0)
                xk[i] = (T)(IP ? -acc : acc);
        }
    }
    __syncthreads();
    for (int i = t; i < nc; i += 256) {
        const T v = xk[i];
        int above = 0;
        for (int o = 0; o < nc; o++)
            above += xk[o] < v || (xk[o] == v && col[o] < col[i]);
        if (above < k) {
            T o = v;
            if (post == 1 && o >= (T)0)
                o = sqrt(o);
            else if (post == 2)
                o = (T)1 + o;
            else if (post == 3)
                o = -o;
            dist[(int64_t)q * k + above] = o;
            ind[(int64_t)q * k + above] = id[i];
        }
    }
    // Fewer vectors than k in the probed lists: index -1 at infinite distance.
    const T inf = (T)__builtin_huge_val();
    for (int i = nc + t; i < k; i += 256) {
        dist[(int64_t)q * k + i] = post == 3 ? -inf : inf;
        ind[(int64_t)q * k + i] = -1;
    }
}

} // namespace

hipError_t launch_ivf_map(const int *perm, const int *list_off, const int *tile_off, int n_list,
                          int *map, hipStream_t s) {
    hipLaunchKernelGGL(ivf_map_kernel, dim3(n_list), dim3(256), 0, s, perm, list_off, tile_off, map);
    return hipGetLastError();
}

hipError_t launch_ivf_tile_scores(const IvfTiles &p, const int *probes, const void *QP, int nq,
                                  int d, float *out, int64_t ld, hipStream_t s) {
    const int64_t pairs = (int64_t)nq * p.n_probe;
    if (d < 1 || d > IVF_TILE_D || p.n_probe > IVF_TILE_PROBE || p.n_probe > p.n_list ||
        pairs > INT_MAX || nq < 1)
        return hipErrorInvalidValue;
    hipLaunchKernelGGL(ivf_zero_kernel, dim3(1), dim3(1024), 0, s, p.cnt, p.n_list);
    hipLaunchKernelGGL(ivf_place_kernel, dim3((nq + 3) / 4), dim3(256), 0, s, p, probes, nq);
    hipLaunchKernelGGL(ivf_items_kernel, dim3(1), dim3(1024), 0, s, p);
    hipLaunchKernelGGL(ivf_group_kernel, dim3((unsigned)((pairs + 255) / 256)), dim3(256), 0, s, p,
                       pairs);
    // Workgroups without an item or a run end at once; a list longer than 64 runs takes several
    // passes.
    const dim3 grid((unsigned)ivf_items(pairs, p.n_list),
                    (unsigned)std::min(64, std::max(1, (p.max_tiles + IVF_RUN - 1) / IVF_RUN)));
    const _Float16 *qp = static_cast<const _Float16 *>(QP);
    switch (wide_ksteps(d)) {
    case 1: hipLaunchKernelGGL(ivf_scores_kernel<1>, grid, dim3(256), 0, s, p, qp, out, ld); break;
    case 2: hipLaunchKernelGGL(ivf_scores_kernel<2>, grid, dim3(256), 0, s, p, qp, out, ld); break;
    case 3: hipLaunchKernelGGL(ivf_scores_kernel<3>, grid, dim3(256), 0, s, p, qp, out, ld); break;
    default: hipLaunchKernelGGL(ivf_scores_kernel<4>, grid, dim3(256), 0, s, p, qp, out, ld); break;
    }
    return hipGetLastError();
}

template <typename T>
hipError_t launch_ivf_tile_select(const IvfTiles &p, const float *scores, int64_t ld,
                                  const float *err, const T *Q, const T *X, int nq, int d, int k,
                                  int ip, int post, int q0, T *dist, int *ind, int *fb_count,
                                  int *fb_list, hipStream_t s) {
    if (k < 1 || k > IVF_TILE_K || d > IVF_TILE_D || nq < 1)
        return hipErrorInvalidValue;
    auto kern = ip ? ivf_tile_select_kernel<T, true> : ivf_tile_select_kernel<T, false>;
    hipLaunchKernelGGL(kern, dim3(nq), dim3(256), 0, s, p, scores, ld, err, Q, X, d, k, post, q0,
                       dist, ind, fb_count, fb_list);
    return hipGetLastError();
}

#define DA_IVF_TILE_INST(T)                                                                      \
    template hipError_t launch_ivf_tile_select<T>(const IvfTiles &, const float *, int64_t,      \
                                                  const float *, const T *, const T *, int, int, \
                                                  int, int, int, int, T *, int *, int *, int *,  \
                                                  hipStream_t);
DA_IVF_TILE_INST(float)
DA_IVF_TILE_INST(double)
#undef DA_IVF_TILE_INST

} // namespace dagpu
