// Causal attention over the paged key/value cache: the kernel that takes every
// shape (any head counts and groups, head sizes in steps of 8 up to 256, any page
// size that is a multiple of 8, a window or none), for 32-bit and bfloat16 storage.
//
// A workgroup per (token, head), which eight waves, or two or four in their places, share out.  A token's request, its absolute position p and the
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
// (token, head) that walked 64 keys at a time, a lane a key, and then the values key by key).  Prompts are bound by the loads of keys and
// values, each (token, head) its own: 2,048 tokens, 8 heads of 128 over 2, 32-bit 1.43 ms (4.42 before), 16 heads over a latent of 576 and 512,
// bfloat16, 10.0 (30.8).
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

constexpr int AG_WAVES = 8, AG_KEYS = 16;      // waves a workgroup (a power of two), keys a wave and step

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

// NV: values of a lane, NV * 64 >= dv.  KP > 0: dh is at most 32 * KP, a lane keeps its KP pieces of the query in registers.
// WAVES: waves of the workgroup, each of which does the work of AG_WAVES / WAVES, one after the other (the same bits).
template <class T, int NV, int KP, int WAVES>
__global__ void __launch_bounds__(WAVES *WAVE)
paged_attention_generic_kernel(const T *__restrict__ q, int q_stride, T *__restrict__ out, int out_stride,
                               const T *__restrict__ cache, const int *__restrict__ block_table, int max_pages,
                               const int *__restrict__ q_start, const int *__restrict__ ctx_len,
                               const int *__restrict__ req_of_token, int nh, int nkvh, int dh, int dv, int page,
                               float scale, int window, int chunk, const float *__restrict__ head_slopes,
                               const float *__restrict__ sinks, float softcap) {
    constexpr bool ONE = KP > 0;
    __shared__ float outs[AG_WAVES][NV * WAVE];
    __shared__ float tops[AG_WAVES], sums[AG_WAVES];
    const int t = blockIdx.x, h = blockIdx.y, lane = threadIdx.x & 63, wave0 = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int key = lane >> 2, part = lane & 3;
    const int r = req_of_token[t];
    const int p = ctx_len[r] - (q_start[r + 1] - t);
    const int lo = chunk > 0 ? p - p % chunk : window > 0 ? (p - window + 1 > 0 ? p - window + 1 : 0) : 0;
    const int kvh = h / (nh / nkvh);
    const int dh8 = dh / 8;
    const float slope = head_slopes ? head_slopes[h] : 0.f;
    const T *qh = q + (size_t)t * q_stride + (size_t)h * dh;
    // sixteen keys from 16 b on are those of wave b % AG_WAVES.  A wave without keys reads nothing and is not looked at in the end
    const int b0 = lo / AG_KEYS, blocks = p / AG_KEYS - b0;
    auto has_keys = [&](int w) { return ((w - b0) & (AG_WAVES - 1)) <= blocks; };
    float qr[KP ? KP : 1][8];
    if constexpr (ONE) if (WAVES < AG_WAVES || has_keys(wave0)) {
#pragma unroll
        for (int i = 0; i < KP; ++i) {
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
    constexpr int STEP = AG_WAVES * AG_KEYS;
    for (int wave = wave0; wave < AG_WAVES; wave += WAVES) {
        if (!has_keys(wave)) continue;
        float m = -INFINITY, l = 0.f;
        float o[NV];
#pragma unroll
        for (int i = 0; i < NV; ++i) o[i] = 0.f;

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
                float k[KP ? KP : 1][8];
#pragma unroll
                for (int i = 0; i < KP; ++i) load8(kp + (size_t)min(part + 4 * i, dh8 - 1) * page * 8, k[i]);
#pragma unroll
                for (int i = 0; i < NV; ++i) fetch(i, v[i]);
#pragma unroll
                for (int i = 0; i < KP; ++i) {
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
    }
    __syncthreads();
    if ((int)threadIdx.x >= dv) return;
    // (what a wave without keys would have left is read with the others, all at once, and not used)
    float top = -INFINITY, keep[AG_WAVES], total = 0.f;
#pragma unroll
    for (int w = 0; w < AG_WAVES; ++w) {
        const float x = tops[w];
        keep[w] = has_keys(w) ? x : -INFINITY;
        top = fmaxf(top, keep[w]);
    }
    if (sinks) top = fmaxf(top, sinks[h]);                      // the sink's term stands in the denominator beside the keys'
#pragma unroll
    for (int w = 0; w < AG_WAVES; ++w) {
        const float x = sums[w];
        keep[w] = keep[w] == -INFINITY ? 0.f : expf(keep[w] - top);
        total = has_keys(w) ? fmaf(x, keep[w], total) : total;
    }
    if (sinks) total += expf(sinks[h] - top);
    const float inv = 1.f / total;
    for (int d = threadIdx.x; d < dv; d += WAVES * WAVE) {
        float x = 0.f;
#pragma unroll
        for (int w = 0; w < AG_WAVES; ++w) {
            const float y = outs[w][d];
            x = has_keys(w) ? fmaf(y, keep[w], x) : x;
        }
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
    // A workgroup of eight waves is for steps that would leave compute units idle.  Where there are (token, head) pairs enough, waves that find no keys
    // only take the places of others: us with 8 / 4 / 2 waves, 40 prompts of 20 tokens, 32-bit, 8 heads of 128: 47.7 / 29.9 / 21.6, 16 heads over a
    // latent of 576: 447 / 245 / 142; one of 2,048 tokens 1,424 / 1,407 / 1,434.  Over keys of 20 to 2,000, seven shapes of heads: from 1,024 pairs on 4
    // waves take 0.93 of the time of 8 (geometric mean; the worst 1.06), from 2,048 on 2 waves 0.85 (1.14); below 1,024 2 waves take 1.5.
    const long long pairs = (long long)n * nh;
    const int waves = pairs >= 2048 ? 2 : pairs >= 1024 ? 4 : AG_WAVES;
    dim3 grid(n, nh);
#define GO(T, NV, KP, W) paged_attention_generic_kernel<T, NV, KP, W><<<grid, dim3(W * WAVE), 0, stream>>>((const T *)q, q_stride, (T *)out, out_stride, (const T *)cache, block_table, max_pages, q_start, ctx_len, req_of_token, nh, nkvh, dh, dv, page, scale, window, chunk, head_slopes, sinks, softcap)
#define WIDTHS(T, NV, KP) do { if (waves == 2) GO(T, NV, KP, 2); else if (waves == 4) GO(T, NV, KP, 4); else GO(T, NV, KP, AG_WAVES); } while (0)
#define SIZES(T) do { if (dh <= 64 && dv <= 64) WIDTHS(T, 1, 2); else if (dh <= 128 && dv <= 64) WIDTHS(T, 1, 4); else if (dh <= 128 && dv <= 128) WIDTHS(T, 2, 4); else if (dv <= 256) WIDTHS(T, 4, 0); else WIDTHS(T, 10, 0); } while (0)
    if (type == LCU_F32) SIZES(float);
    else if (type == LCU_BF16) SIZES(bf16_t);
    else return LCU_BAD_ARGUMENT;
#undef GO
#undef WIDTHS
#undef SIZES
    LCU_LAUNCH_CHECK();
    return LCU_OK;
}
