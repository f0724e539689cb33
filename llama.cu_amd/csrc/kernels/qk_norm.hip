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
// A row is read once, four columns at a time where the addresses allow it, the weights on their way with it: one trip to memory and one sum.
// A sum is made of those of stretches of 64 accesses, in their order, however many waves they are dealt to: a row's bits do not depend on
// how many rows there are.  Up to QK_FEW rows, which latency bounds, a row's queries, keys and values are a workgroup of eight waves each; beyond
// them they share a workgroup, with two accesses a lane (the most that a lane keeps).  One MI355X, bfloat16, 16 heads of 128 over 4, with
// norms, us at 4 / 256 / 2,048 rows: 3.1 / 4.3 / 12.5; workgroups of their own throughout 3.0 / 4.4 / 17.6; one workgroup that did the three one
// after the other and read each twice 6.6 / 7.5 / 16.3.
#include "rows.h"
#include "kv_layout.h"

constexpr int QK_KEEP = 2;                        // accesses of a thread that stay in registers between the sum and the product
constexpr int QK_MAX_Q = 8, QK_MAX_K = 4, QK_MAX_V = 2;       // waves of a part, powers of two
constexpr int QK_SUMS = 128;                      // stretches with a sum of their own (a wave's number modulo this is its own stretches')
constexpr int QK_FEW = 128;

// Row blockIdx.x of qkv = [q (nh*dh) | k (nkvh*dh) | v (nkvh*dv)]: q_waves waves for the queries, then k_waves for the keys (0: the row
// holds queries only), the rest for the values; q_waves 0: workgroup (row, part), all waves for that part.  V: columns an access.
template <class T, int V>
__global__ void __launch_bounds__((QK_MAX_Q + QK_MAX_K + QK_MAX_V) * WAVE)
qk_norm_store_kernel(T *__restrict__ qkv, int row_stride, const int *__restrict__ positions,
                     const int *__restrict__ slots, const float *__restrict__ qw, const float *__restrict__ kw,
                     T *__restrict__ cache, int nh, int nkvh, int dh, int dv, int page, float eps, float coef,
                     int every, int q_count, int k_count, int q_waves, int k_waves) {
    __shared__ float sums[2][QK_SUMS];
    const int t = blockIdx.x, nq = nh * dh, nk = nkvh * dh, nv = nkvh * dv;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const bool apart = q_waves == 0;                 // every part a workgroup of its own
    const int part = apart ? (int)blockIdx.y : wave < q_waves ? 0 : wave < q_waves + k_waves ? 1 : 2;
    const int wave0 = apart || part == 0 ? 0 : part == 1 ? q_waves : q_waves + k_waves;
    const int waves = apart || part == 2 ? (int)blockDim.x / WAVE - wave0 : part == 0 ? q_waves : k_waves;
    const int tid = threadIdx.x - wave0 * WAVE, threads = waves * WAVE;
    T *row = qkv + (size_t)t * row_stride;
    const int slot = part > 0 ? slots[t] : 0;
    T *pg = part > 0 && slot >= 0 ? cache + (size_t)(slot / page) * kv_page_elems(nkvh, dh, dv, page) : nullptr;
    const int tok = slot % page;
    if (part == 2) {
        if (slot >= 0)
#pragma unroll 4
            for (int c = tid; c < nv; c += threads) pg[kv_value_offset(nkvh, c / dv, tok, c % dv, dh, dv, page)] = row[nq + nk + c];
        if (!apart && (qw || kw)) __syncthreads();   // (the parts with a norm wait for their sums)
        return;
    }
    const int nc = part == 0 ? nq : nk;
    T *src = part == 0 ? row : row + nq;
    const float *w = part == 0 ? qw : kw;
    const bool writes = part == 0 ? w || coef != 0.f : slot >= 0;
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
    const int c0 = tid * V, step = threads * V;
    if (writes)
#pragma unroll
        for (int i = 0; i < QK_KEEP; ++i)
            if (c0 + i * step < nc) load(c0 + i * step, x[i], f[i]);
    const int p = part == 0 && coef != 0.f ? positions[t] : 0;
    const int stretches = (nc + WAVE * V - 1) / (WAVE * V);
    if (w && writes) {
        for (int i = wave - wave0, k = 0; i < stretches; i += waves, ++k) {
            float acc = 0.f, v[V];
            const int c = (i * WAVE + tid % WAVE) * V;
            if (c < nc) {
                if (k >= QK_KEEP) load_as_f32<T, V>(src + c, v);
#pragma unroll
                for (int e = 0; e < V; ++e) {
                    const float one = k == 0 ? x[0][e] : k == 1 ? x[1][e] : v[e];
                    acc = fmaf(one, one, acc);        // (as it stands: which product the compiler would fuse is not the same for all stretches)
                }
            }
            acc = wave_sum_in_place(acc);
            if (tid % WAVE == 0) sums[part][i % QK_SUMS] = (i < QK_SUMS ? 0.f : sums[part][i % QK_SUMS]) + acc;
        }
    }
    if (qw || kw) __syncthreads();
    if (!writes) return;
    if (w) {
        float total = 0.f;
        for (int i = 0; i < min(stretches, QK_SUMS); ++i) total += sums[part][i];
        factor = rsqrtf(total / (float)(part == 0 ? q_count : k_count) + eps);
    }
    if (part == 0 && coef != 0.f) factor *= 1.0f + coef * logf((float)((p + 1) / every) + 1.0f);
#pragma unroll
    for (int i = 0; i < QK_KEEP; ++i)
        if (c0 + i * step < nc) store(c0 + i * step, x[i], f[i]);
    for (int c = c0 + QK_KEEP * step; c < nc; c += step) {
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
    // four columns at a time: queries and keys are whole pieces of eight columns, so only the addresses decide
    const bool four = four_ok(qkv, type) && four_ok(qw, LCU_F32) && four_ok(kw, LCU_F32) && (!store_kv || four_ok(cache, type)) && row_stride % 4 == 0 && page % 4 == 0;
    auto waves = [&](int columns, int a_wave, int most) {          // the power of two of waves that take a_wave columns each
        int x = 1;
        while (x < most && x * a_wave < columns) x *= 2;
        return x;
    };
    const int a_wave = WAVE * (four ? 4 : 1) * QK_KEEP;
    const bool apart = n <= QK_FEW;
    const int q_waves = apart ? 0 : waves(nh * dh, a_wave, QK_MAX_Q), k_waves = apart || !store_kv ? 0 : waves(nkvh * dh, a_wave, QK_MAX_K);
    const int v_waves = apart || !store_kv ? 0 : waves(nkvh * dv, 4 * WAVE, QK_MAX_V);
    const dim3 grid(n, apart && store_kv ? 3 : 1), block((apart ? QK_MAX_Q : q_waves + k_waves + v_waves) * WAVE);
#define GO(T, V) qk_norm_store_kernel<T, V><<<grid, block, 0, stream>>>((T *)qkv, row_stride, positions, slots, qw, kw, (T *)cache, nh, nkvh, dh, dv, page, eps, coef, every, q_count, k_count, q_waves, k_waves)
    if (type == LCU_F32) { if (four) GO(float, 4); else GO(float, 1); }
    else if (type == LCU_BF16) { if (four) GO(bf16_t, 4); else GO(bf16_t, 1); }
    else return LCU_BAD_ARGUMENT;
#undef GO
    LCU_LAUNCH_CHECK();
    return LCU_OK;
}
