// The sum of a token's experts' outputs where it is used: by the kernel that adds nothing else (moe.hip), or by the norm that adds it to the residual
// stream, which then takes one trip to memory for what a kernel in front of it would have written and it read again.
#pragma once
#include "common.h"

typedef __attribute__((ext_vector_type(4))) float pair_f32x4;
typedef __attribute__((ext_vector_type(2))) uint32_t pair_u32x2;
// Rows may begin at any element (a caller's part of a larger tensor): one load of four elements all the same, which the hardware takes at any address.
typedef pair_f32x4 __attribute__((aligned(4))) pair_f32x4_at;
typedef pair_u32x2 __attribute__((aligned(2))) pair_u32x2_at;
__device__ __forceinline__ pair_f32x4 pair_four(const float *p) { return *(const pair_f32x4_at *)p; }
__device__ __forceinline__ pair_f32x4 pair_four(const bf16_t *p) {
    const pair_u32x2 v = *(const pair_u32x2_at *)p;
    return pair_f32x4{__uint_as_float(v[0] << 16), __uint_as_float(v[0] & 0xffff0000u), __uint_as_float(v[1] << 16), __uint_as_float(v[1] & 0xffff0000u)};
}

// row t: base[t] (null: 0) + sum_k wts[t, k] * y[t * top + k]  (in the order of k; wts null: ones)  + gate[t] * (shared[t] or shared32[t])  (gate null: 1).
// A pair's product is rounded before it is added, the shared row's is not.
// ids (null: none), real, h: a pair whose expert is `real` or beyond is an identity expert, whose output is the token's input row h[t] itself.
// shared and h are of the model's type, all else 32-bit; all rows are contiguous.
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
    auto four = [](const void *base, size_t at) { return pair_four((const T *)base + at); };
    const size_t at = t * d + c;
    pair_f32x4 acc = {0.f, 0.f, 0.f, 0.f}, own = acc, s = acc;
    if (p.base) acc = pair_four(p.base + at);
    if (p.ids) own = four(p.h, at);
    if (p.shared) s = four(p.shared, at);
    else if (p.shared32) s = pair_four(p.shared32 + at);
    const float g = p.gate ? p.gate[t] : 1.f;
    for (int k0 = 0; k0 < p.top; k0 += 2) {              // (two pairs' loads together; an identity expert's row of y is memory that nobody wrote, and dropped)
        pair_f32x4 row[2];
        float w[2];
        bool mine[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const size_t pair = t * p.top + min(k0 + u, p.top - 1);
            row[u] = pair_four(p.y + pair * d + c);
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

static bool pair_sum_ok(const PairSum &p, int d) { return d > 0 && d % 4 == 0 && p.y && p.top > 0 && (!p.ids || p.h); }
