// What kernels that take a row a workgroup share: several elements an access, and the sum over the workgroup.
#pragma once
#include "common.h"
#include "lane_moves.h"

// V neighbouring elements as one access.
template <class T, int V> struct alignas(V * sizeof(T)) Pack { T v[V]; };
template <class T, int V> __device__ __forceinline__ void load_as_f32(const T *p, float *out) {
    const Pack<T, V> in = *(const Pack<T, V> *)p;
#pragma unroll
    for (int e = 0; e < V; ++e) out[e] = to_f32(in.v[e]);
}
template <class T, int V> __device__ __forceinline__ void store_f32(T *p, const float *in) {
    Pack<T, V> out;
#pragma unroll
    for (int e = 0; e < V; ++e) out.v[e] = from_f32<T>(in[e]);
    *(Pack<T, V> *)p = out;
}

// The same where the address may lie at any element: V accesses unless WIDE.
template <class T, int V, bool WIDE> __device__ __forceinline__ void load_some(const T *p, float *out) {
    if constexpr (WIDE) {
        load_as_f32<T, V>(p, out);
    } else {
#pragma unroll
        for (int e = 0; e < V; ++e) out[e] = to_f32(p[e]);
    }
}
template <class T, int V, bool WIDE> __device__ __forceinline__ void store_some(T *p, const float *in) {
    if constexpr (WIDE) {
        store_f32<T, V>(p, in);
    } else {
#pragma unroll
        for (int e = 0; e < V; ++e) p[e] = from_f32<T>(in[e]);
    }
}

// The sum over a workgroup of up to 16 waves; `scratch` (16 floats) is not in use by an earlier call.
__device__ __forceinline__ float row_sum(float v, float *scratch) {
    v = wave_sum_in_place(v);
    if ((threadIdx.x & 63) == 0) scratch[threadIdx.x >> 6] = v;
    __syncthreads();
    float t = 0.f;
    for (int i = 0; i < (int)blockDim.x / WAVE; ++i) t += scratch[i];
    return t;
}

// Whether four elements at a time may be read and written at p (null: nothing is).
static bool four_ok(const void *p, int type) { return ((uintptr_t)p & (type == LCU_BF16 ? 7 : 15)) == 0; }
