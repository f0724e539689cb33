// The sum of a token's experts' outputs where it is used: by the kernel that adds nothing else (moe.hip), or by the norm that adds it to the residual
// stream, which then takes one trip to memory for what a kernel in front of it would have written and it read again.
#pragma once
#include "common.h"

typedef __attribute__((ext_vector_type(4))) float pair_f32x4;
template <class T> struct alignas(4 * sizeof(T)) PairQuad { T v[4]; };

// row t: base[t] (null: 0) + sum_k wts[t, k] * y[t * top + k]  (in the order of k; wts null: ones)  + gate[t] * (shared[t] or shared32[t])  (gate null: 1).
// A pair's product is rounded before it is added, the shared row's is not.
// ids (null: none), real, h: a pair whose expert is `real` or beyond is an identity expert, whose output is the token's input row h[t] itself.
// shared and h are of the model's type, all else 32-bit; all rows are contiguous and aligned for four of their elements.
struct PairSum {
    const float *base, *y, *wts;
    const void *shared;
    const float *shared32, *gate;
    const int *ids;
    const void *h;
    int top, real;
};

// Columns c .. c + 3 of row t of width d.
template <class T>
__device__ __forceinline__ pair_f32x4 pair_sum4(const PairSum &p, size_t t, int c, int d) {
#pragma clang fp contract(off)
    auto four = [](const void *base, size_t at) {
        const PairQuad<T> q = *(const PairQuad<T> *)((const T *)base + at);
        return pair_f32x4{to_f32(q.v[0]), to_f32(q.v[1]), to_f32(q.v[2]), to_f32(q.v[3])};
    };
    const size_t at = t * d + c;
    pair_f32x4 acc = {0.f, 0.f, 0.f, 0.f}, own = acc, s = acc;
    if (p.base) acc = *(const pair_f32x4 *)(p.base + at);
    if (p.ids) own = four(p.h, at);
    if (p.shared) s = four(p.shared, at);
    else if (p.shared32) s = *(const pair_f32x4 *)(p.shared32 + at);
    const float g = p.gate ? p.gate[t] : 1.f;
    for (int k0 = 0; k0 < p.top; k0 += 2) {              // (two pairs' loads together; an identity expert's row of y is memory that nobody wrote, and dropped)
        pair_f32x4 row[2];
        float w[2];
        bool mine[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const size_t pair = t * p.top + min(k0 + u, p.top - 1);
            row[u] = *(const pair_f32x4 *)(p.y + pair * d + c);
            w[u] = p.wts ? p.wts[pair] : 1.f;
            mine[u] = p.ids && p.ids[pair] >= p.real;
        }
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            if (k0 + u >= p.top) break;
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[e] += w[u] * (mine[u] ? own[e] : row[u][e]);
        }
    }
    if (p.shared || p.shared32) {
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[e] = __builtin_fmaf(g, s[e], acc[e]);
    }
    return acc;
}

// Whether every row may be read four elements at a time.
static bool pair_sum_ok(const PairSum &p, int type, int d) {
    const uintptr_t narrow = (uintptr_t)p.shared | (uintptr_t)p.h;
    return d > 0 && d % 4 == 0 && p.y && p.top > 0 && (!p.ids || p.h) && (narrow & (type == LCU_BF16 ? 7 : 15)) == 0 &&
           (((uintptr_t)p.base | (uintptr_t)p.y | (uintptr_t)p.shared32) & 15) == 0;
}
