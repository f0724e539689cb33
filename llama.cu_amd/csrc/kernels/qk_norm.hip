// What stands between the q, k, v product and an attention that has no rotation: a norm
// over the whole query projection and over the whole key projection (all heads at once, a
// weight per column), a factor on the queries that grows with the logarithm of the position,
// and the write of keys and values into their pages.  Each piece is optional.
//
//   q <- q * rsqrt(mean(q^2) + eps) * qw          (mean over all nh * dh columns, or over q_count of them where heads
//                                                   were filled up with columns of zeros; qw null: no norm)
//   q <- q * (1 + coef * ln(floor((p + 1) / every) + 1))      (p the row's position; coef 0: none)
//   k <- k * rsqrt(mean(k^2) + eps) * kw          (over all nkvh * dh columns), into the cache
//   v into the cache as it is (head size dv)
// Sums, norms and factors are 32-bit; one rounding where q is written back and where k
// is stored.
//
// A row's queries, keys and values are a workgroup each, and a row is read once, four columns at a time where the addresses allow it, the
// weights on their way with it: one trip to memory and one sum.  One MI355X, 4 rows of 16 heads of 128 over 4, bfloat16: 9.5 us with
// one workgroup a row that did the three one after the other and read each twice; 4.7 us now.
#include "rows.h"
#include "kv_layout.h"

constexpr int QK_THREADS = 512, QK_KEEP = 2;      // accesses of a thread that stay in registers between the sum and the product

// Workgroups (row, part) of qkv = [q (nh*dh) | k (nkvh*dh) | v (nkvh*dv)]: the parts are the queries, the keys and the values (only the
// queries if !store_kv).  V: columns an access.
template <class T, int V>
__global__ void __launch_bounds__(QK_THREADS)
qk_norm_store_kernel(T *__restrict__ qkv, int row_stride, const int *__restrict__ positions,
                     const int *__restrict__ slots, const float *__restrict__ qw, const float *__restrict__ kw,
                     T *__restrict__ cache, int nh, int nkvh, int dh, int dv, int page, float eps, float coef,
                     int every, int q_count, int k_count) {
    __shared__ float scratch[16];
    const int t = blockIdx.x, part = blockIdx.y, nq = nh * dh, nk = nkvh * dh, nv = nkvh * dv;
    T *row = qkv + (size_t)t * row_stride;
    const int slot = part > 0 ? slots[t] : 0;
    if (slot < 0) return;
    T *pg = part > 0 ? cache + (size_t)(slot / page) * kv_page_elems(nkvh, dh, dv, page) : nullptr;
    const int tok = slot % page;
    if (part == 2) {
        for (int c = threadIdx.x; c < nv; c += QK_THREADS) pg[kv_value_offset(nkvh, c / dv, tok, c % dv, dh, dv, page)] = row[nq + nk + c];
        return;
    }
    const int nc = part == 0 ? nq : nk;
    T *src = part == 0 ? row : row + nq;
    const float *w = part == 0 ? qw : kw;
    if (part == 0 && !w && coef == 0.f) return;
    float x[QK_KEEP][V], f[QK_KEEP][V], factor = 1.f;
    auto load = [&](int c, float *xs, float *fs) {
        load_as_f32<T, V>(src + c, xs);
        if (w) {
            load_as_f32<float, V>(w + c, fs);
        } else {
#pragma unroll
            for (int e = 0; e < V; ++e) fs[e] = 1.f;
        }
    };
    auto store = [&](int c, float *xs, const float *fs) {
#pragma unroll
        for (int e = 0; e < V; ++e) xs[e] = xs[e] * factor * fs[e];
        store_f32<T, V>(part == 0 ? src + c : pg + kv_key_offset(c / dh, tok, c % dh, dh, page), xs);     // (V divides eight: within a piece of eight dims)
    };
    const int c0 = threadIdx.x * V;
    constexpr int STEP = QK_THREADS * V;
#pragma unroll
    for (int i = 0; i < QK_KEEP; ++i)
        if (c0 + i * STEP < nc) load(c0 + i * STEP, x[i], f[i]);
    const int p = part == 0 && coef != 0.f ? positions[t] : 0;
    if (w) {
        float acc = 0.f;
#pragma unroll
        for (int i = 0; i < QK_KEEP; ++i)
            if (c0 + i * STEP < nc)
#pragma unroll
                for (int e = 0; e < V; ++e) acc += x[i][e] * x[i][e];
        for (int c = c0 + QK_KEEP * STEP; c < nc; c += STEP) {
            float v[V];
            load_as_f32<T, V>(src + c, v);
#pragma unroll
            for (int e = 0; e < V; ++e) acc += v[e] * v[e];
        }
        factor = rsqrtf(row_sum(acc, scratch) / (float)(part == 0 ? q_count : k_count) + eps);
    }
    if (part == 0 && coef != 0.f) factor *= 1.0f + coef * logf((float)((p + 1) / every) + 1.0f);
#pragma unroll
    for (int i = 0; i < QK_KEEP; ++i)
        if (c0 + i * STEP < nc) store(c0 + i * STEP, x[i], f[i]);
    for (int c = c0 + QK_KEEP * STEP; c < nc; c += STEP) {
        float xs[V], fs[V];
        load(c, xs, fs);
        store(c, xs, fs);
    }
}

LCU_API int lcu_qk_norm_store(void *qkv, int type, int n, int row_stride, const int *positions, const int *slots,
                              const float *qw, const float *kw, void *cache, int nh, int nkvh, int dh, int dv, int page,
                              float eps, float coef, int every, int store_kv, int q_count, int k_count, hipStream_t stream) {
    if (n <= 0) return LCU_OK;
    if (nh <= 0 || nkvh <= 0 || dh <= 0 || dh % 8 || dv <= 0 || page <= 0 || (coef != 0.f && (every <= 0 || !positions)) ||
        (store_kv && (!cache || !slots)))
        return LCU_BAD_ARGUMENT;
    // the columns that a mean runs over: fewer than the rows hold where heads were filled up with columns of zeros
    if (q_count <= 0) q_count = nh * dh;
    if (k_count <= 0) k_count = nkvh * dh;
    const dim3 grid(n, store_kv ? 3 : 1), block(QK_THREADS);
    // four columns at a time: queries and keys are whole pieces of eight columns, so only the addresses decide
    const bool four = four_ok(qkv, type) && four_ok(qw, LCU_F32) && four_ok(kw, LCU_F32) && (!store_kv || four_ok(cache, type)) && row_stride % 4 == 0 && page % 4 == 0;
#define GO(T, V) qk_norm_store_kernel<T, V><<<grid, block, 0, stream>>>((T *)qkv, row_stride, positions, slots, qw, kw, (T *)cache, nh, nkvh, dh, dv, page, eps, coef, every, q_count, k_count)
    if (type == LCU_F32) { if (four) GO(float, 4); else GO(float, 1); }
    else if (type == LCU_BF16) { if (four) GO(bf16_t, 4); else GO(bf16_t, 1); }
    else return LCU_BAD_ARGUMENT;
#undef GO
    LCU_LAUNCH_CHECK();
    return LCU_OK;
}
