// A norm BEHIND a sublayer, the residual sum, and the norm in front of the next sublayer, in one pass:
//
//   x <- x + a * rsqrt(mean(a^2) + eps_post) * w_post          (a: the sublayer's output; x: the 32-bit residual stream)
//   h  = x * rsqrt(mean(x^2) + eps_pre) * w_pre                (only if w_pre is given; with out but no w_pre: h = x, the
//                                                              stream itself rounded to out's type, for a sublayer that reads it so)
//
// One block per row; sums, factors and the stream are 32-bit, one rounding where h is stored.  The weights are the
// factors themselves (a model that stores them around zero adds the one when it loads them).  The order of the sums
// depends on the width and the block size only.
#include "rows.h"
#include "pair_sum.h"

constexpr int NP_KEEP = 8;          // elements of a row that a thread keeps in registers: rows up to 8 x the block's threads are read once

// THREADS: 256, or 1024 where a step has few rows (what counts then is how many loads a row has in flight).  All loads of
// the kept elements go out before anything waits for one.
template <class TA, class TO, int THREADS>
__global__ void __launch_bounds__(THREADS)
norm_post_kernel(float *__restrict__ x, const TA *__restrict__ a, const float *__restrict__ a_bias, const float *__restrict__ w_post, float eps_post,
                 const float *__restrict__ w_pre, float eps_pre, TO *__restrict__ out, int d) {
    __shared__ float scratch[16];
    float *xr = x + (size_t)blockIdx.x * d;
    const TA *ar = a + (size_t)blockIdx.x * d;
    float keep[NP_KEEP], xs[NP_KEEP], wp[NP_KEEP], wq[NP_KEEP];
    float acc = 0.f;
#pragma unroll
    for (int e = 0; e < NP_KEEP; ++e) {
        const int c = threadIdx.x + e * THREADS;
        const bool in = c < d;
        keep[e] = in ? to_f32(ar[c]) + (a_bias ? a_bias[c] : 0.f) : 0.f;
        xs[e] = in ? xr[c] : 0.f;
        wp[e] = in ? w_post[c] : 0.f;
        wq[e] = (in && w_pre) ? w_pre[c] : 0.f;
    }
#pragma unroll
    for (int e = 0; e < NP_KEEP; ++e) acc += keep[e] * keep[e];
    for (int c = threadIdx.x + NP_KEEP * THREADS; c < d; c += THREADS) {
        const float v = to_f32(ar[c]) + (a_bias ? a_bias[c] : 0.f);
        acc += v * v;
    }
    const float f_post = rsqrtf(block_sum(acc, scratch) / (float)d + eps_post);
    acc = 0.f;
#pragma unroll
    for (int e = 0; e < NP_KEEP; ++e) {
        const int c = threadIdx.x + e * THREADS;
        if (c < d) {
            keep[e] = xs[e] + keep[e] * f_post * wp[e];
            xr[c] = keep[e];
            acc += keep[e] * keep[e];
        }
    }
    for (int c = threadIdx.x + NP_KEEP * THREADS; c < d; c += THREADS) {
        const float v = xr[c] + (to_f32(ar[c]) + (a_bias ? a_bias[c] : 0.f)) * f_post * w_post[c];
        xr[c] = v;
        acc += v * v;
    }
    if (!out) return;
    TO *o = out + (size_t)blockIdx.x * d;
    if (!w_pre) {                            // the stream itself, rounded once
#pragma unroll
        for (int e = 0; e < NP_KEEP; ++e) {
            const int c = threadIdx.x + e * THREADS;
            if (c < d) o[c] = from_f32<TO>(keep[e]);
        }
        for (int c = threadIdx.x + NP_KEEP * THREADS; c < d; c += THREADS) o[c] = from_f32<TO>(xr[c]);
        return;
    }
    const float f_pre = rsqrtf(block_sum(acc, scratch) / (float)d + eps_pre);
#pragma unroll
    for (int e = 0; e < NP_KEEP; ++e) {
        const int c = threadIdx.x + e * THREADS;
        if (c < d) o[c] = from_f32<TO>(keep[e] * f_pre * wq[e]);
    }
    for (int c = threadIdx.x + NP_KEEP * THREADS; c < d; c += THREADS)      // (a thread reads what it wrote itself)
        o[c] = from_f32<TO>(xr[c] * f_pre * w_pre[c]);
}

// Rows of up to 4 * THREADS * PT elements, a multiple of 4, with every pointer aligned for four: 512 threads whatever the number of
// rows, all loads first, two barriers.  (With 1,024 threads and single elements one row of 2,048 took 3.7 us, now 2.2, 16 rows 4.7, now 3.1; 2,048 rows
// 10.8, now 9.2.)
constexpr int NP_ROW_THREADS = 512;
// A: where the sublayer's output comes from: rows, or a token's experts.  (Their sum in a kernel in front was 4.7 us a layer in a step of 16 tokens and 11.7 in one of
// 2,040, most of it the way through memory: ralepel 12.54 -> 12.12 ms a pass without it.)
template <class T> struct RowsOf {
    const T *p;
    __device__ __forceinline__ void four(size_t row, int c, int d, float *out) const { load_as_f32<T, 4>(p + row * d + c, out); }
};
template <class T> struct PairsOf {
    PairSum p;
    __device__ __forceinline__ void four(size_t row, int c, int d, float *out) const {
        const pair_f32x4 v = pair_sum4<T>(p, row, c, d);
#pragma unroll
        for (int e = 0; e < 4; ++e) out[e] = v[e];
    }
};
template <class A, class TO, int PT>
__global__ void __launch_bounds__(NP_ROW_THREADS)
norm_post_row_kernel(float *__restrict__ x, const A a, const float *__restrict__ a_bias, const float *__restrict__ w_post, float eps_post,
                     const float *__restrict__ w_pre, float eps_pre, TO *__restrict__ out, int d) {
    __shared__ float scratch[2][16];
    float *xr = x + (size_t)blockIdx.x * d;
    float v[PT][4], xs[PT][4], wp[PT][4], wq[PT][4], acc = 0.f;
#pragma unroll
    for (int i = 0; i < PT; ++i) {
        const int c = (threadIdx.x + NP_ROW_THREADS * i) * 4;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[i][e] = 0.f;
        if (c >= d) continue;
        load_as_f32<float, 4>(xr + c, xs[i]);
        load_as_f32<float, 4>(w_post + c, wp[i]);
        if (w_pre) load_as_f32<float, 4>(w_pre + c, wq[i]);
        a.four(blockIdx.x, c, d, v[i]);
        if (a_bias) {
            float b[4];
            load_as_f32<float, 4>(a_bias + c, b);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[i][e] += b[e];
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) acc += v[i][e] * v[i][e];
    }
    const float f_post = rsqrtf(row_sum(acc, scratch[0]) / (float)d + eps_post);
    acc = 0.f;
#pragma unroll
    for (int i = 0; i < PT; ++i) {
        const int c = (threadIdx.x + NP_ROW_THREADS * i) * 4;
        if (c >= d) continue;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            v[i][e] = xs[i][e] + v[i][e] * f_post * wp[i][e];
            acc += v[i][e] * v[i][e];
        }
        store_f32<float, 4>(xr + c, v[i]);
    }
    if (!out) return;
    const float f_pre = w_pre ? rsqrtf(row_sum(acc, scratch[1]) / (float)d + eps_pre) : 1.f;
    TO *o = out + (size_t)blockIdx.x * d;
#pragma unroll
    for (int i = 0; i < PT; ++i) {
        const int c = (threadIdx.x + NP_ROW_THREADS * i) * 4;
        if (c >= d) continue;
        if (w_pre) {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[i][e] = v[i][e] * f_pre * wq[i][e];
        }                                    // (else the stream itself, rounded once)
        store_f32<TO, 4>(o + c, v[i]);
    }
}

// x: [n, d] float32, updated in place.  a: [n, d] of a_type.  w_post, w_pre: float32 [d]; w_pre and out may be null.
// a_bias: null, or float32 [d] that the sublayer's output still lacks (a bias of its last product): a + a_bias is normed.
LCU_API int lcu_norm_post(float *x, const void *a, int a_type, const float *a_bias, const float *w_post, float eps_post, const float *w_pre,
                          float eps_pre, void *out, int out_type, int n, int d, hipStream_t stream) {
    if (n <= 0) return LCU_OK;
    if (d <= 0 || !x || !a || !w_post || (w_pre && !out)) return LCU_BAD_ARGUMENT;
    // few rows of some width: 1024 threads a row (a row's sums are then added in another order than with 256: a
    // difference of rounding between steps of few and of many rows)
    const bool wide = n <= 64 && d >= 1024;
    dim3 grid(n);
    const bool four = d % 4 == 0 && d <= 8 * NP_ROW_THREADS && four_ok(x, LCU_F32) && four_ok(a, a_type) && four_ok(a_bias, LCU_F32) &&
                      four_ok(w_post, LCU_F32) && four_ok(w_pre, LCU_F32) && four_ok(out, out_type);
#define FOUR(TA, TO, PT) norm_post_row_kernel<RowsOf<TA>, TO, PT><<<grid, dim3(NP_ROW_THREADS), 0, stream>>>(x, RowsOf<TA>{(const TA *)a}, a_bias, w_post, eps_post, w_pre, eps_pre, (TO *)out, d)
#define GO(TA, TO) do { if (four && d <= 4 * NP_ROW_THREADS) FOUR(TA, TO, 1); else if (four) FOUR(TA, TO, 2); \
                        else if (wide) norm_post_kernel<TA, TO, 1024><<<grid, dim3(1024), 0, stream>>>(x, (const TA *)a, a_bias, w_post, eps_post, w_pre, eps_pre, (TO *)out, d); \
                        else norm_post_kernel<TA, TO, 256><<<grid, dim3(256), 0, stream>>>(x, (const TA *)a, a_bias, w_post, eps_post, w_pre, eps_pre, (TO *)out, d); } while (0)
    if (a_type == LCU_F32 && out_type == LCU_F32) GO(float, float);
    else if (a_type == LCU_F32 && out_type == LCU_BF16) GO(float, bf16_t);
    else if (a_type == LCU_BF16 && out_type == LCU_BF16) GO(bf16_t, bf16_t);
    else if (a_type == LCU_BF16 && out_type == LCU_F32) GO(bf16_t, float);
    else return LCU_BAD_ARGUMENT;
#undef GO
#undef FOUR
    LCU_LAUNCH_CHECK();
    return LCU_OK;
}

// The same with a token's experts' sum (in host memory; type: of the model, and of out) in the place of a.  d a multiple of 4, at most 8 * NP_ROW_THREADS.
LCU_API int lcu_norm_post_pairs(float *x, const PairSum *pairs, int type, const float *w_post, float eps_post, const float *w_pre, float eps_pre, void *out, int n,
                                int d, hipStream_t stream) {
    if (n <= 0) return LCU_OK;
    if (!x || !pairs || !w_post || (w_pre && !out) || !pair_sum_ok(*pairs, d) || d > 8 * NP_ROW_THREADS || !four_ok(x, LCU_F32) || !four_ok(w_post, LCU_F32) ||
        !four_ok(w_pre, LCU_F32) || !four_ok(out, type) || (type != LCU_F32 && type != LCU_BF16))
        return LCU_BAD_ARGUMENT;
#define GO(T, PT) norm_post_row_kernel<PairsOf<T>, T, PT><<<dim3(n), dim3(NP_ROW_THREADS), 0, stream>>>(x, PairsOf<T>{*pairs}, nullptr, w_post, eps_post, w_pre, eps_pre, (T *)out, d)
    if (type == LCU_BF16) { if (d <= 4 * NP_ROW_THREADS) GO(bf16_t, 1); else GO(bf16_t, 2); }
    else { if (d <= 4 * NP_ROW_THREADS) GO(float, 1); else GO(float, 2); }
#undef GO
    LCU_LAUNCH_CHECK();
    return LCU_OK;
}

// acc = (first ? 0 : acc) + scale * x over `count` floats: the 32-bit sum of several branches' outputs.
template <class TX>
__global__ void scaled_sum_kernel(float *__restrict__ acc, const TX *__restrict__ x, float scale, long long count, int first) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) acc[i] = (first ? 0.f : acc[i]) + scale * to_f32(x[i]);
}

LCU_API int lcu_scaled_sum(float *acc, const void *x, int x_type, float scale, long long count, int first, hipStream_t stream) {
    if (count <= 0) return LCU_OK;
    if (!acc || !x) return LCU_BAD_ARGUMENT;
    dim3 grid((unsigned)((count + 255) / 256)), block(256);
    if (x_type == LCU_F32) scaled_sum_kernel<float><<<grid, block, 0, stream>>>(acc, (const float *)x, scale, count, first);
    else if (x_type == LCU_BF16) scaled_sum_kernel<bf16_t><<<grid, block, 0, stream>>>(acc, (const bf16_t *)x, scale, count, first);
    else return LCU_BAD_ARGUMENT;
    LCU_LAUNCH_CHECK();
    return LCU_OK;
}

// rows[t, c] += bias[c] in place (rows: [n, d] of `type`, the sum in 32-bit, one rounding): the bias of a product whose
// kernel adds none.
template <class T>
__global__ void row_bias_kernel(T *__restrict__ rows, const float *__restrict__ bias, long long count, int d) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) rows[i] = from_f32<T>(to_f32(rows[i]) + bias[i % d]);
}

LCU_API int lcu_row_bias(void *rows, int type, const float *bias, int n, int d, hipStream_t stream) {
    if (n <= 0) return LCU_OK;
    if (d <= 0 || !rows || !bias) return LCU_BAD_ARGUMENT;
    const long long count = (long long)n * d;
    dim3 grid((unsigned)((count + 255) / 256)), block(256);
    if (type == LCU_F32) row_bias_kernel<float><<<grid, block, 0, stream>>>((float *)rows, bias, count, d);
    else if (type == LCU_BF16) row_bias_kernel<bf16_t><<<grid, block, 0, stream>>>((bf16_t *)rows, bias, count, d);
    else return LCU_BAD_ARGUMENT;
    LCU_LAUNCH_CHECK();
    return LCU_OK;
}
