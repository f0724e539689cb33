// Causal attention over the paged key/value cache: the kernel that takes every
// shape (any head counts and groups, head sizes in steps of 8 up to 256, any page
// size that is a multiple of 8, a window or none), for 32-bit and bfloat16 storage.
//
// A workgroup of eight waves per (token, head).  A token's request, its absolute position p and the
// keys it sees, [lo, p] with lo = max(0, p - window + 1) (0 without a window; with
// chunk > 0 instead lo = p - p % chunk: the keys of the query's own chunk, chunks counted
// from the request's position 0), come from the batch arrays.  Keys are walked in chunks of 128 that start at multiples of
// 128, sixteen keys a wave: four lanes share a key's dims, then every lane holds dims of the values and takes them sixteen keys
// at a time, and a wave has all these loads on their way together.  The waves share nothing while they walk; their maxima,
// sums (online softmax) and outputs, all 32-bit, meet at the end, added in the waves' order.  What a (token, head) computes,
// and the order it adds in, depends on p and the cache's contents only: not on how the step's tokens were cut,
// not on other requests in the batch, not on which pages hold the keys.
//
// Latency bounds it: one MI355X, 2 requests of 53 keys, 8 heads of 128 over 2, 32-bit, inside a step: 6.7 us (23.6 with one wave a
// (token, head) that walked 64 keys at a time, a lane a key, and then the values key by key).
//
// head_slopes (may be null): a bias inside the scores that grows with the distance, for position
// encodings of that kind: slope[h] * (j - p) is added to the scaled score of key j for the query at p.
// dv: the values' head size (the keys' is dh); out is [n, nh * dv].
// sinks (may be null): a number per head that stands in the softmax's denominator as exp(sink[h]) beside the keys'
// terms; it has no key, no value, no scale and no bias, and counts once for every query.
// softcap (0: none): a scaled score s becomes softcap * tanh(s / softcap), before any bias.
#include "common.h"
#include "kv_layout.h"
#include "lane_moves.h"

constexpr int MAX_HEAD_DIM = 640;        // NV = 4 covers values up to 256 dims, NV = 10 up to 640

constexpr int AG_WAVES = 8, AG_KEYS = 16;      // waves a workgroup, keys a wave and step

// Eight neighbouring elements as floats (the array may start at any element).
typedef __attribute__((ext_vector_type(4), aligned(4))) float f32x4_any;
typedef __attribute__((ext_vector_type(4), aligned(2))) uint32_t u32x4_any;
__device__ __forceinline__ void load8(const float *p, float (&v)[8]) {
    const f32x4_any a = *(const f32x4_any *)p, b = *(const f32x4_any *)(p + 4);
#pragma unroll
    for (int e = 0; e < 4; ++e) { v[e] = a[e]; v[4 + e] = b[e]; }
}
__device__ __forceinline__ void load8(const bf16_t *p, float (&v)[8]) {
    const u32x4_any a = *(const u32x4_any *)p;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        v[2 * e] = __uint_as_float(a[e] << 16);
        v[2 * e + 1] = __uint_as_float(a[e] & 0xffff0000u);
    }
}

// NV: values of a lane, NV * 64 >= dv.  ONE: dh is at most 128, a lane keeps its part of the query in registers.
template <class T, int NV, bool ONE>
__global__ void __launch_bounds__(AG_WAVES *WAVE)
paged_attention_generic_kernel(const T *__restrict__ q, int q_stride, T *__restrict__ out, int out_stride,
                               const T *__restrict__ cache, const int *__restrict__ block_table, int max_pages,
                               const int *__restrict__ q_start, const int *__restrict__ ctx_len,
                               const int *__restrict__ req_of_token, int nh, int nkvh, int dh, int dv, int page,
                               float scale, int window, int chunk, const float *__restrict__ head_slopes,
                               const float *__restrict__ sinks, float softcap) {
    __shared__ float outs[AG_WAVES][NV * WAVE];
    __shared__ float tops[AG_WAVES], sums[AG_WAVES];
    const int t = blockIdx.x, h = blockIdx.y, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int key = lane >> 2, part = lane & 3;
    const int r = req_of_token[t];
    const int p = ctx_len[r] - (q_start[r + 1] - t);
    const int lo = chunk > 0 ? p - p % chunk : window > 0 ? (p - window + 1 > 0 ? p - window + 1 : 0) : 0;
    const int kvh = h / (nh / nkvh);
    const int dh8 = dh / 8;
    const float slope = head_slopes ? head_slopes[h] : 0.f;
    const T *qh = q + (size_t)t * q_stride + (size_t)h * dh;
    float qr[4][8];
    if constexpr (ONE) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int c8 = part + 4 * i;
            load8(qh + 8 * (c8 < dh8 ? c8 : 0), qr[i]);
            if (c8 >= dh8)
#pragma unroll
                for (int e = 0; e < 8; ++e) qr[i][e] = 0.f;
        }
    }

    const int *bt = block_table + (size_t)r * max_pages;
    const size_t page_elems = kv_page_elems(nkvh, dh, dv, page);
    const size_t v_base = kv_value_offset(nkvh, kvh, 0, 0, dh, dv, page);
    float m = -INFINITY, l = 0.f;
    float o[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) o[i] = 0.f;

    constexpr int STEP = AG_WAVES * AG_KEYS;
    for (int base = (lo / STEP) * STEP + wave * AG_KEYS; base <= p; base += STEP) {
        if (base + AG_KEYS <= lo) continue;
        const int j = base + key;
        const bool valid = j >= lo && j <= p;
        const int jr = min(max(j, lo), p);                       // (a key that is not the wave's is read in place of one that is not the query's)
        const T *kp = cache + (size_t)bt[jr / page] * page_elems + ((size_t)kvh * dh8 * page + jr % page) * 8;
        // the values' pieces of eight tokens, which lie in a page: read if any of their keys is the query's
        const T *vp[2];
        bool any[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int j0 = base + 8 * u;
            any[u] = j0 <= p && j0 + 8 > lo;
            vp[u] = cache + (size_t)(any[u] ? bt[j0 / page] : 0) * page_elems + v_base + j0 % page;
        }
        float v[ONE ? NV : 1][2][8];
        auto fetch = [&](int i, float (&x)[2][8]) {
            const int d = min(lane + WAVE * i, dv - 1);
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                if (any[u]) {
                    load8(vp[u] + (size_t)d * page, x[u]);
                } else {
#pragma unroll
                    for (int e = 0; e < 8; ++e) x[u][e] = 0.f;
                }
            }
        };
        float acc = 0.f;
        if constexpr (ONE) {
            float k[4][8];
#pragma unroll
            for (int i = 0; i < 4; ++i) load8(kp + (size_t)min(part + 4 * i, dh8 - 1) * page * 8, k[i]);
#pragma unroll
            for (int i = 0; i < NV; ++i) fetch(i, v[i]);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (part + 4 * i < dh8)
#pragma unroll
                    for (int e = 0; e < 8; ++e) acc += qr[i][e] * k[i][e];
            }
        } else {
#pragma unroll 4
            for (int c8 = part; c8 < dh8; c8 += 4) {
                float k[8], x[8];
                load8(kp + (size_t)c8 * page * 8, k);
                load8(qh + 8 * c8, x);
#pragma unroll
                for (int e = 0; e < 8; ++e) acc += x[e] * k[e];
            }
        }
        acc += lane_xor1(acc);
        acc += lane_xor2(acc);
        acc *= scale;
        if (softcap > 0.f) acc = softcap * tanhf(acc / softcap);
        const float s = valid ? acc + slope * (float)(j - p) : -INFINITY;
        const float m_new = fmaxf(m, wave_max_in_place(s));
        const float at = m_new == -INFINITY ? 0.f : m_new;      // (every score minus infinity so far: terms of zero)
        const float pj = valid ? expf(s - at) : 0.f;
        const float alpha = expf(m - at);                       // 0 in the first chunk (m = -inf)
        l = l * alpha + wave_sum_in_place(part == 0 ? pj : 0.f);
        m = m_new;
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            float x[2][8];
            if constexpr (!ONE) fetch(i, x);
            o[i] *= alpha;
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const int j2 = base + 8 * u + e;
                    const float pp = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(pj), 4 * (8 * u + e)));
                    const float val = ONE ? v[ONE ? i : 0][u][e] : x[u][e];
                    o[i] += (j2 >= lo && j2 <= p) ? pp * val : 0.f;          // (what lies beyond the query's keys may be any number)
                }
        }
    }
#pragma unroll
    for (int i = 0; i < NV; ++i) outs[wave][lane + WAVE * i] = o[i];
    if (lane == 0) {
        tops[wave] = m;
        sums[wave] = l;
    }
    __syncthreads();
    float top = -INFINITY;
#pragma unroll
    for (int w = 0; w < AG_WAVES; ++w) top = fmaxf(top, tops[w]);
    if (sinks) top = fmaxf(top, sinks[h]);                      // the sink's term stands in the denominator beside the keys'
    float keep[AG_WAVES], total = 0.f;
#pragma unroll
    for (int w = 0; w < AG_WAVES; ++w) {
        keep[w] = tops[w] == -INFINITY ? 0.f : expf(tops[w] - top);
        total += sums[w] * keep[w];
    }
    if (sinks) total += expf(sinks[h] - top);
    const float inv = 1.f / total;
    for (int d = threadIdx.x; d < dv; d += AG_WAVES * WAVE) {
        float x = 0.f;
#pragma unroll
        for (int w = 0; w < AG_WAVES; ++w) x += outs[w][d] * keep[w];
        out[(size_t)t * out_stride + (size_t)h * dv + d] = from_f32<T>(x * inv);
    }
}

// q: [n, q_stride] (head h of token t at t*q_stride + h*dh), out: [n, out_stride].
// cache: one layer's pages.  block_table: [n_req, max_pages] page ids (an entry that a
// window has passed may hold anything: it is not read).  q_start: [n_req + 1] offsets of
// the requests' tokens in the batch, ctx_len: [n_req] tokens each request holds after
// this step, req_of_token: [n].  head_slopes: null or [nh] 32-bit.
LCU_API int lcu_paged_attention_generic(const void *q, int q_stride, void *out, int out_stride, int type,
                                        const void *cache, const int *block_table, int max_pages,
                                        const int *q_start, const int *ctx_len, const int *req_of_token, int n,
                                        int nh, int nkvh, int dh, int dv, int page, float scale, int window,
                                        int chunk, const float *head_slopes, const float *sinks, float softcap, hipStream_t stream) {
    if (n <= 0) return LCU_OK;
    if (nh <= 0 || nkvh <= 0 || nh % nkvh || dh <= 0 || dh % 8 || dh > MAX_HEAD_DIM || dv <= 0 || dv > MAX_HEAD_DIM || page <= 0 || page % 8 ||
        max_pages <= 0 || window < 0 || chunk < 0 || (window > 0 && chunk > 0) || nh > 65535 || softcap < 0.f)
        return LCU_BAD_ARGUMENT;
    dim3 grid(n, nh), block(AG_WAVES * WAVE);
#define GO(T, NV, ONE) paged_attention_generic_kernel<T, NV, ONE><<<grid, block, 0, stream>>>((const T *)q, q_stride, (T *)out, out_stride, (const T *)cache, block_table, max_pages, q_start, ctx_len, req_of_token, nh, nkvh, dh, dv, page, scale, window, chunk, head_slopes, sinks, softcap)
#define SIZES(T) do { if (dh <= 128 && dv <= 128) GO(T, 2, true); else if (dv <= 256) GO(T, 4, false); else GO(T, 10, false); } while (0)
    if (type == LCU_F32) SIZES(float);
    else if (type == LCU_BF16) SIZES(bf16_t);
    else return LCU_BAD_ARGUMENT;
#undef GO
#undef SIZES
    LCU_LAUNCH_CHECK();
    return LCU_OK;
}
