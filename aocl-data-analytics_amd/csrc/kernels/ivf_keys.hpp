// Terms of the exact IVF-Flat keys, shared by the list scans and the selection of the matrix-core
// search, which must round alike.
#pragma once
#include <hip/hip_runtime.h>

namespace dagpu {

// 16-byte chunks of a row: four floats or two doubles. acc adds the squared differences of
// a chunk's elements in element order, dot their products.
template <typename T> struct Chunk16;
template <> struct Chunk16<float> {
    using type = float4;
    __device__ static type zero() { return make_float4(0.f, 0.f, 0.f, 0.f); }
    __device__ static void acc(double &a, const type &q, const type &x) {
        const double t0 = (double)q.x - (double)x.x, t1 = (double)q.y - (double)x.y;
        const double t2 = (double)q.z - (double)x.z, t3 = (double)q.w - (double)x.w;
        a += t0 * t0;
        a += t1 * t1;
        a += t2 * t2;
        a += t3 * t3;
    }
    __device__ static void dot(double &a, const type &q, const type &x) {
        a += (double)q.x * (double)x.x;
        a += (double)q.y * (double)x.y;
        a += (double)q.z * (double)x.z;
        a += (double)q.w * (double)x.w;
    }
};
template <> struct Chunk16<double> {
    using type = double2;
    __device__ static type zero() { return make_double2(0.0, 0.0); }
    __device__ static void acc(double &a, const type &q, const type &x) {
        const double t0 = q.x - x.x, t1 = q.y - x.y;
        a += t0 * t0;
        a += t1 * t1;
    }
    __device__ static void dot(double &a, const type &q, const type &x) {
        a += q.x * x.x;
        a += q.y * x.y;
    }
};

// Rows of whole 16-byte chunks (the buffers are allocated 256-byte aligned) up to 128 elements are
// summed chunk by chunk over eight lanes, others element by element over sixteen.
template <typename T> __host__ __device__ constexpr bool ivf_chunked(int d) {
    return d % (16 / (int)sizeof(T)) == 0 && d <= 128;
}

} // namespace dagpu
