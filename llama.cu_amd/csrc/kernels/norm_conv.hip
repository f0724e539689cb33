// Layer norm (mean and variance, weight and bias) fused with the residual sum that precedes
// it, for one or two norms of the same row; and the short causal convolution over time that
// a sublayer may put in front of what it reads, with its per-request state.
//
// Layer norm of a row x of width d, all in 32-bit:
//   m = mean(x), var = mean((x - m)^2) (the deviations are taken from the mean that was
//   computed first), y = (x - m) * rsqrt(var + eps) * w + b.
// Short convolution of taps T on every channel c of rows h that belong to requests:
//   out[t] = h[t] + sum_{j < T} cw[c][j] * h[t - (T - 1) + j]
// where rows before the request's first row of this step come from the request's state (the
// last T - 1 rows of earlier steps) and rows before position 0 are zeros.
#include "common.h"
#include "rows.h"
#include "conv_rows.h"
#include "pair_sum.h"

constexpr int NC_THREADS = 256;
constexpr int MAX_TAPS = 16;

// x (32-bit residual stream, [n, d]) takes in `planes` planes of delta (type TD, plane_stride
// apart), is written back, and is normed with (w1, b1) into out1 and, if w2 is not null, with
// (w2, b2) into out2.  One block per row.
template <class TD, class TO>
__global__ void __launch_bounds__(NC_THREADS)
layernorm_kernel(float *__restrict__ x, const TD *__restrict__ delta, int planes, size_t plane_stride,
                 const float *__restrict__ w1, const float *__restrict__ b1, TO *__restrict__ out1,
                 const float *__restrict__ w2, const float *__restrict__ b2, TO *__restrict__ out2, int d, float eps) {
    __shared__ float scratch[16];
    float *xr = x + (size_t)blockIdx.x * d;
    float sum = 0.f;
    for (int c = threadIdx.x; c < d; c += NC_THREADS) {
        float v = xr[c];
        if (delta) {
            for (int p = 0; p < planes; ++p) v += to_f32(delta[p * plane_stride + (size_t)blockIdx.x * d + c]);
            xr[c] = v;
        }
        sum += v;
    }
    const float mean = block_sum(sum, scratch) / (float)d;
    float sq = 0.f;
    for (int c = threadIdx.x; c < d; c += NC_THREADS) {     // each thread reads back what it wrote itself
        const float dev = xr[c] - mean;
        sq += dev * dev;
    }
    const float rstd = rsqrtf(block_sum(sq, scratch) / (float)d + eps);
    for (int c = threadIdx.x; c < d; c += NC_THREADS) {
        const float z = (xr[c] - mean) * rstd;
        out1[(size_t)blockIdx.x * d + c] = from_f32<TO>(z * w1[c] + b1[c]);
        if (w2) out2[(size_t)blockIdx.x * d + c] = from_f32<TO>(z * w2[c] + b2[c]);
    }
}

// A row's elements in one thread's registers: PT pieces of V neighbours, T pieces apart.  The row takes in the planes
// of delta, is written back, and its mean and the inverse of its deviation come out.  A step of few rows is a chain of dependent
// trips to memory and through the barriers: one trip, two barriers.
// V is 4 where d is a multiple of 4, else 1, and T, the number of threads, 256 where that makes one piece a thread, else 512: which elements a
// thread adds, and so a row's bits, depend on d alone.  (A 32-bit model gives a token the same bits in a portion, whose norm and
// convolution are kernels of their own, and alone.)  2,048 rows of 64 or 100: 4.9 and 5.6 us with 512 threads, 3.6 and 4.0 with 256; one odd row of
// 513: 2.7 us with 512, 3.4 with 256 (2,048 of them 7.5 and 6.3).  WIDE: every address lets four elements be read at once.
// D: where delta comes from: planes of rows, or a token's experts (beside another branch's rows).
template <class T> struct PlanesOf {
    const T *p;
    int planes;
    size_t stride;
    __device__ __forceinline__ bool any() const { return p != nullptr; }
    template <int V, bool WIDE> __device__ __forceinline__ void first(size_t row, int c, int d, float *out) const { load_some<T, V, WIDE>(p + row * d + c, out); }
    template <int V, bool WIDE> __device__ __forceinline__ void add_rest(size_t row, int c, int d, float *out) const {
        for (int k = 1; k < planes; ++k) {
            float more[V];
            load_some<T, V, WIDE>(p + k * stride + row * d + c, more);
#pragma unroll
            for (int e = 0; e < V; ++e) out[e] += more[e];
        }
    }
};
template <class T> struct PairsOf {
    PairSum p;
    __device__ __forceinline__ bool any() const { return true; }
    template <int V, bool WIDE> __device__ __forceinline__ void first(size_t row, int c, int d, float *out) const {
        static_assert(V == 4 && WIDE, "");
        const pair_f32x4 v = pair_sum4<T>(p, row, c, d);
#pragma unroll
        for (int e = 0; e < 4; ++e) out[e] = v[e];
    }
    template <int V, bool WIDE> __device__ __forceinline__ void add_rest(size_t, int, int, float *) const {}
};
template <class D, int T, int V, int PT, bool WIDE>
__device__ __forceinline__ void take_row(float *xr, const D &delta, size_t row, int d, float eps,
                                         float (&v)[PT][V], float &mean, float &rstd, float (*scratch)[16]) {
    float sum = 0.f, first[PT][V];                   // (the row and the first plane are on their way before anything is added or written)
#pragma unroll
    for (int i = 0; i < PT; ++i) {
        const int c = (threadIdx.x + T * i) * V;
#pragma unroll
        for (int e = 0; e < V; ++e) v[i][e] = first[i][e] = 0.f;
        if (c < d) {
            load_some<float, V, WIDE>(xr + c, v[i]);
            if (delta.any()) delta.template first<V, WIDE>(row, c, d, first[i]);
        }
    }
#pragma unroll
    for (int i = 0; i < PT; ++i) {
        const int c = (threadIdx.x + T * i) * V;
        if (delta.any() && c < d) {
#pragma unroll
            for (int e = 0; e < V; ++e) v[i][e] += first[i][e];
            delta.template add_rest<V, WIDE>(row, c, d, v[i]);
            store_some<float, V, WIDE>(xr + c, v[i]);
        }
#pragma unroll
        for (int e = 0; e < V; ++e) sum += v[i][e];
    }
    mean = row_sum(sum, scratch[0]) / (float)d;
    float sq = 0.f;
#pragma unroll
    for (int i = 0; i < PT; ++i)
#pragma unroll
        for (int e = 0; e < V; ++e) {
            const float dev = v[i][e] - mean;
            if ((threadIdx.x + T * i) * V < d) sq += dev * dev;
        }
    rstd = rsqrtf(row_sum(sq, scratch[1]) / (float)d + eps);
}

// The same for rows of up to T * V * PT elements: the row stays in registers between its one read and its writes.  With 256
// threads and single elements 2,048 rows of 2,048 with two 32-bit outputs took 21.8 us, now 14.2, one row 5.5, now 2.3.
template <class D, class TO, int T, int V, int PT, bool WIDE>
__global__ void __launch_bounds__(T)
layernorm_row_kernel(float *__restrict__ x, const D delta,
                     const float *__restrict__ w1, const float *__restrict__ b1, TO *__restrict__ out1,
                     const float *__restrict__ w2, const float *__restrict__ b2, TO *__restrict__ out2, int d, float eps) {
    __shared__ float scratch[2][16];
    const size_t row_at = (size_t)blockIdx.x * d;
    float v[PT][V], w[2][PT][V], b[2][PT][V], mean, rstd;
    // (the weights are on their way while the sums are made)
#pragma unroll
    for (int i = 0; i < PT; ++i) {
        const int c = (threadIdx.x + T * i) * V;
        if (c < d) {
            load_some<float, V, WIDE>(w1 + c, w[0][i]);
            load_some<float, V, WIDE>(b1 + c, b[0][i]);
            if (w2) {
                load_some<float, V, WIDE>(w2 + c, w[1][i]);
                load_some<float, V, WIDE>(b2 + c, b[1][i]);
            }
        }
    }
    take_row<D, T, V, PT, WIDE>(x + row_at, delta, blockIdx.x, d, eps, v, mean, rstd, scratch);
#pragma unroll
    for (int i = 0; i < PT; ++i) {
        const int c = (threadIdx.x + T * i) * V;
        if (c >= d) continue;
        float y[V];
#pragma unroll
        for (int e = 0; e < V; ++e) y[e] = (v[i][e] - mean) * rstd * w[0][i][e] + b[0][i][e];
        store_some<TO, V, WIDE>(out1 + row_at + c, y);
        if (w2) {
#pragma unroll
            for (int e = 0; e < V; ++e) y[e] = (v[i][e] - mean) * rstd * w[1][i][e] + b[1][i][e];
            store_some<TO, V, WIDE>(out2 + row_at + c, y);
        }
    }
}

// delta_type: -1 none, LCU_F32 or LCU_BF16.  out_type: LCU_F32 or LCU_BF16.
LCU_API int lcu_layernorm(float *x, const void *delta, int delta_type, int planes, const float *w1, const float *b1,
                          void *out1, const float *w2, const float *b2, void *out2, int out_type, int n, int d,
                          float eps, hipStream_t stream) {
    if (n <= 0) return LCU_OK;
    if (d <= 0 || !w1 || !b1 || !out1 || (w2 && (!b2 || !out2)) || (delta && planes <= 0)) return LCU_BAD_ARGUMENT;
    const size_t stride = (size_t)n * d;
    dim3 grid(n), block(NC_THREADS);
    const int dt = delta ? delta_type : LCU_F32;
    const bool four = d % 4 == 0;
    const bool wide = four_ok(x, LCU_F32) && four_ok(delta, dt) && four_ok(w1, LCU_F32) && four_ok(b1, LCU_F32) && four_ok(out1, out_type) &&
                      four_ok(w2, LCU_F32) && four_ok(b2, LCU_F32) && four_ok(out2, out_type);
#define ROW(TD, TO, T, V, PT, WIDE) layernorm_row_kernel<PlanesOf<TD>, TO, T, V, PT, WIDE><<<grid, dim3(T), 0, stream>>>(x, PlanesOf<TD>{(const TD *)delta, planes, stride}, w1, b1, (TO *)out1, w2, b2, (TO *)out2, d, eps)
#define GO(TD, TO)                                                                                                           \
    do {                                                                                                                     \
        if (four && d <= 1024) { if (wide) ROW(TD, TO, 256, 4, 1, true); else ROW(TD, TO, 256, 4, 1, false); }               \
        else if (four && d <= 2048) { if (wide) ROW(TD, TO, 512, 4, 1, true); else ROW(TD, TO, 512, 4, 1, false); }          \
        else if (four && d <= 4096) { if (wide) ROW(TD, TO, 512, 4, 2, true); else ROW(TD, TO, 512, 4, 2, false); }          \
        else if (d <= 256) ROW(TD, TO, 256, 1, 1, false);                                                                    \
        else if (d <= 1024) ROW(TD, TO, 512, 1, 2, false);                                                                   \
        else if (d <= 4096) ROW(TD, TO, 512, 1, 8, false);                                                                   \
        else layernorm_kernel<TD, TO><<<grid, block, 0, stream>>>(x, (const TD *)delta, planes, stride, w1, b1, (TO *)out1,  \
                                                                  w2, b2, (TO *)out2, d, eps);                               \
    } while (0)
    if (dt == LCU_F32 && out_type == LCU_F32) GO(float, float);
    else if (dt == LCU_F32 && out_type == LCU_BF16) GO(float, bf16_t);
    else if (dt == LCU_BF16 && out_type == LCU_F32) GO(bf16_t, float);
    else if (dt == LCU_BF16 && out_type == LCU_BF16) GO(bf16_t, bf16_t);
    else return LCU_BAD_ARGUMENT;
#undef ROW
#undef GO
    LCU_LAUNCH_CHECK();
    return LCU_OK;
}

// The same with a token's experts' sum (in host memory; type: of the model) as delta.  d a multiple of 4, at most 4096, everything aligned for four.
LCU_API int lcu_layernorm_pairs(float *x, const PairSum *pairs, int type, const float *w1, const float *b1, void *out1, const float *w2, const float *b2,
                                void *out2, int out_type, int n, int d, float eps, hipStream_t stream) {
    if (n <= 0) return LCU_OK;
    if (!x || !pairs || !w1 || !b1 || !out1 || (w2 && (!b2 || !out2)) || !pair_sum_ok(*pairs, d) || d > 4096 || !four_ok(x, LCU_F32) ||
        !four_ok(w1, LCU_F32) || !four_ok(b1, LCU_F32) || !four_ok(out1, out_type) || !four_ok(w2, LCU_F32) || !four_ok(b2, LCU_F32) || !four_ok(out2, out_type))
        return LCU_BAD_ARGUMENT;
#define ROW(T_, TO, T, PT) layernorm_row_kernel<PairsOf<T_>, TO, T, 4, PT, true><<<dim3(n), dim3(T), 0, stream>>>(x, PairsOf<T_>{*pairs}, w1, b1, (TO *)out1, w2, b2, (TO *)out2, d, eps)
#define GO(T_, TO) do { if (d <= 1024) ROW(T_, TO, 256, 1); else if (d <= 2048) ROW(T_, TO, 512, 1); else ROW(T_, TO, 512, 2); } while (0)
    if (type == LCU_F32 && out_type == LCU_F32) GO(float, float);
    else if (type == LCU_BF16 && out_type == LCU_F32) GO(bf16_t, float);
    else if (type == LCU_BF16 && out_type == LCU_BF16) GO(bf16_t, bf16_t);
    else return LCU_BAD_ARGUMENT;
#undef GO
#undef ROW
    LCU_LAUNCH_CHECK();
    return LCU_OK;
}

// ---------------------------------------------------------------- short convolution
// `sets` independent convolutions at once (blockIdx.y): set s reads h + s * set_stride_h, the
// weights cw + s * d * taps ([d, taps]), its part of the state and writes
// out + s * set_stride_out.  state: [slots, sets, taps - 1, d] 32-bit, row i of a request's state is
// the row at position P0 - (taps - 1) + i, P0 the position of the request's first row of this
// step.  The state is only read here.
template <class TI, class TW, class TO>
__global__ void __launch_bounds__(NC_THREADS)
short_conv_kernel(const TI *__restrict__ h, size_t set_stride_h, const TW *__restrict__ cw, const float *__restrict__ st, TO *__restrict__ out, size_t set_stride_out, const int *__restrict__ q_start,
                  const int *__restrict__ ctx_len, const int *__restrict__ req_of_token,
                  const int *__restrict__ state_slot, int d, int taps) {
    const int t = blockIdx.x, s = blockIdx.y;
    const int r = req_of_token[t];
    const int first = q_start[r];
    const int pos = ctx_len[r] - (q_start[r + 1] - t);          // this row's position
    const TI *hs = h + s * set_stride_h;
    const TW *w = cw + (size_t)s * d * taps;
    const float *state = st + ((size_t)state_slot[r] * gridDim.y + s) * (taps - 1) * d;
    for (int c = threadIdx.x; c < d; c += NC_THREADS) {
        float acc = to_f32(hs[(size_t)t * d + c]);
        for (int j = 0; j < taps; ++j) {
            const int back = taps - 1 - j;                      // the row `back` positions earlier
            if (pos - back < 0) continue;                       // no such row: the request starts later
            float v;
            if (t - back >= first) v = to_f32(hs[(size_t)(t - back) * d + c]);
            else v = state[(size_t)(taps - 1 - (first - (t - back))) * d + c];
            acc = fmaf(to_f32(w[(size_t)c * taps + j]), v, acc);
        }
        out[s * set_stride_out + (size_t)t * d + c] = from_f32<TO>(acc);
    }
}

// Many tokens (conv_rows.h): the same sums in the same order.
template <class TI, class TW, class TO, int TAPS>
__global__ void __launch_bounds__(CONV_RUN_THREADS)
short_conv_rows_kernel(const TI *__restrict__ h, size_t set_stride_h, const TW *__restrict__ cw, const float *__restrict__ st, TO *__restrict__ out, size_t set_stride_out, const int *__restrict__ q_start,
                       const int *__restrict__ ctx_len, const int *__restrict__ req_of_token,
                       const int *__restrict__ state_slot, int n, int d) {
    const int t0 = blockIdx.x * CONV_RUN, count = min(CONV_RUN, n - t0), s = blockIdx.y, c = (blockIdx.z * CONV_RUN_THREADS + threadIdx.x) * 4;
    if (c >= d) return;
    const TI *hs = h + s * set_stride_h;
    const TW *w = cw + (size_t)s * d * TAPS;
    TO *o = out + s * set_stride_out + (size_t)t0 * d + c;
    float k[4 * TAPS];
#pragma unroll
    for (int q = 0; q < TAPS; ++q) load_as_f32<TW, 4>(w + (size_t)c * TAPS + 4 * q, k + 4 * q);
    conv_run<TAPS>(hs + c, d, t0, count, req_of_token, q_start, ctx_len, state_slot, d,
                   [&](int slot) { return st + ((size_t)slot * gridDim.y + s) * (TAPS - 1) * d + c; },
                   [&](int i, float (*row)[4], int pos, bool) {
        float acc[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[e] = row[TAPS - 1][e];
#pragma unroll
        for (int j = 0; j < TAPS; ++j)
            if (pos >= TAPS - 1 - j)                             // (else there is no such row)
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[e] = fmaf(k[e * TAPS + j], row[j][e], acc[e]);
        store_f32<TO, 4>(o + (size_t)i * d, acc);
    });
}

// After the convolution has run: every request's state becomes the last taps - 1 rows up to
// the end of this step (rows of this step, or of the old state, or zeros before position 0).
// A thread owns a channel: it reads all it needs, then writes.
template <class TI>
__global__ void __launch_bounds__(NC_THREADS)
short_conv_update_kernel(const TI *__restrict__ h, size_t set_stride_h, float *__restrict__ st,
                         const int *__restrict__ q_start, const int *__restrict__ ctx_len,
                         const int *__restrict__ state_slot, int d, int taps) {
    const int r = blockIdx.x, s = blockIdx.y;
    const int first = q_start[r], n_new = q_start[r + 1] - first;
    const int p0 = ctx_len[r] - n_new;                          // position of the first row of this step
    const TI *hs = h + s * set_stride_h;
    float *state = st + ((size_t)state_slot[r] * gridDim.y + s) * (taps - 1) * d;
    for (int c = blockIdx.z * NC_THREADS + threadIdx.x; c < d; c += gridDim.z * NC_THREADS) {
        float keep[MAX_TAPS];
#pragma unroll
        for (int i = 0; i < MAX_TAPS; ++i) {
            if (i < taps - 1) {
                const int back = taps - 1 - i;                  // the new row i lies `back` rows before the step's end
                const int row = n_new - back;                   // among this step's rows, if >= 0
                float v = 0.f;
                if (row >= 0) v = to_f32(hs[(size_t)(first + row) * d + c]);
                else if (p0 + row >= 0) v = state[(size_t)(taps - 1 + row) * d + c];
                keep[i] = v;
            }
        }
#pragma unroll
        for (int i = 0; i < MAX_TAPS; ++i)
            if (i < taps - 1) state[(size_t)i * d + c] = keep[i];
    }
}

// h: [sets][n, d] (sets set_stride_h elements apart), cw: [sets][d, taps], state: [slots, sets, taps - 1, d],
// out: [sets][n, d] (set_stride_out apart).  update: 0 only the convolution,
// 1 the convolution and then the state.
LCU_API int lcu_short_conv(const void *h, int h_type, long long set_stride_h, const void *cw, int w_type, float *state,
                           void *out, int out_type, long long set_stride_out, const int *q_start,
                           const int *ctx_len, const int *req_of_token, const int *state_slot, int n, int n_req, int d,
                           int taps, int sets, int update, hipStream_t stream) {
    if (n <= 0 || n_req <= 0) return LCU_OK;
    if (d <= 0 || taps < 1 || taps > MAX_TAPS || sets < 1 || sets > 8 || h_type != LCU_F32 && h_type != LCU_BF16) return LCU_BAD_ARGUMENT;
    if (w_type != h_type && !(w_type == LCU_F32) && !(h_type == LCU_F32 && w_type == LCU_BF16)) return LCU_BAD_ARGUMENT;
    dim3 grid(n, sets), block(NC_THREADS);
    const bool rows = n >= CONV_RUN_TOKENS && n / CONV_RUN_A_REQUEST >= n_req && (d > 2 * NC_THREADS || (long long)n * sets * d >= CONV_RUN_NARROW) && d % 4 == 0 && taps > 1 && taps <= CONV_RUN_TAPS && set_stride_h % 4 == 0 && set_stride_out % 4 == 0 && four_ok(h, h_type) &&
                      four_ok(cw, w_type) && four_ok(state, LCU_F32) && four_ok(out, out_type);
    const dim3 rgrid((n + CONV_RUN - 1) / CONV_RUN, sets, (d / 4 + CONV_RUN_THREADS - 1) / CONV_RUN_THREADS);
#define ROWS(TI, TW, TO, TAPS) short_conv_rows_kernel<TI, TW, TO, TAPS><<<rgrid, dim3(CONV_RUN_THREADS), 0, stream>>>((const TI *)h, (size_t)set_stride_h, (const TW *)cw, state, (TO *)out, (size_t)set_stride_out, q_start, ctx_len, req_of_token, state_slot, n, d)
#define GO(TI, TW, TO)                                                                                                                                          \
    do {                                                                                                                                                        \
        if (rows && taps == 4) ROWS(TI, TW, TO, 4);                                                                                                             \
        else if (rows && taps == 3) ROWS(TI, TW, TO, 3);                                                                                                        \
        else if (rows) ROWS(TI, TW, TO, 2);                                                                                                                     \
        else short_conv_kernel<TI, TW, TO><<<grid, block, 0, stream>>>((const TI *)h, (size_t)set_stride_h, (const TW *)cw, state, (TO *)out, (size_t)set_stride_out, q_start, ctx_len, req_of_token, state_slot, d, taps); \
    } while (0)
    if (h_type == LCU_F32 && w_type == LCU_F32 && out_type == LCU_F32) GO(float, float, float);
    else if (h_type == LCU_F32 && w_type == LCU_F32 && out_type == LCU_BF16) GO(float, float, bf16_t);
    else if (h_type == LCU_F32 && w_type == LCU_BF16 && out_type == LCU_BF16) GO(float, bf16_t, bf16_t);
    else if (h_type == LCU_F32 && w_type == LCU_BF16 && out_type == LCU_F32) GO(float, bf16_t, float);
    else if (h_type == LCU_BF16 && w_type == LCU_BF16 && out_type == LCU_BF16) GO(bf16_t, bf16_t, bf16_t);
    else if (h_type == LCU_BF16 && w_type == LCU_F32 && out_type == LCU_BF16) GO(bf16_t, float, bf16_t);
    else return LCU_BAD_ARGUMENT;
#undef GO
#undef ROWS
    LCU_LAUNCH_CHECK();
    if (update && taps > 1) {
        dim3 ugrid(n_req, sets, (d + NC_THREADS - 1) / NC_THREADS);
        if (h_type == LCU_F32)
            short_conv_update_kernel<float><<<ugrid, block, 0, stream>>>((const float *)h, (size_t)set_stride_h, state, q_start, ctx_len, state_slot, d, taps);
        else
            short_conv_update_kernel<bf16_t><<<ugrid, block, 0, stream>>>((const bf16_t *)h, (size_t)set_stride_h, state, q_start, ctx_len, state_slot, d, taps);
        LCU_LAUNCH_CHECK();
    }
    return LCU_OK;
}

// ---------------------------------------------------------------- a step of single tokens: all of the above in one kernel
// Every request feeds one token (row r is request r's): the residual sum, one or two layer norms, their short
// convolutions from the requests' states, and the states' update, with the row in registers throughout.  A block
// is the only reader and writer of its request's state, and a thread of its channels'.
// out: [sets][n, d] of TO; state: [slots, sets, taps - 1, d]; cw: [sets][d, taps] 32-bit.
// Everything that is read is read before the row's sums are made: one trip to memory.  V and WIDE as above; TAPS: the number
// of taps where a thread reads its 4 TAPS weights in pieces of four, or 0 (one by one, up to FUSED_TAPS).  With 256 threads,
// single numbers and the two sets one after the other four rows of 2,048 with four taps took 13.8 us, now 5.0.
constexpr int FUSED_TAPS = 8;
template <class D, class TO, int T, int V, int PT, bool WIDE, int TAPS>
__global__ void __launch_bounds__(T)
norm_conv_single_kernel(float *__restrict__ x, const D delta,
                        const float *__restrict__ w1, const float *__restrict__ b1, const float *__restrict__ w2,
                        const float *__restrict__ b2, const float *__restrict__ cw, float *__restrict__ st,
                        TO *__restrict__ out, size_t set_stride_out, const int *__restrict__ ctx_len,
                        const int *__restrict__ state_slot, int d, int taps_rt, int sets, float eps) {
    __shared__ float scratch[2][16];
    const int taps = TAPS ? TAPS : taps_rt;
    constexpr int MOST = TAPS ? TAPS : FUSED_TAPS;
    const int r = blockIdx.x;
    const int pos = ctx_len[r] - 1;                  // the token's position
    float *slot = st + (size_t)state_slot[r] * sets * (taps - 1) * d;
    float v[PT][V], mean, rstd;
    float old[2][PT][MOST > 1 ? MOST - 1 : 1][V], k[2][PT][V][MOST], wv[2][PT][V], bv[2][PT][V];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        if (s >= sets) break;
        const float *w = s ? w2 : w1, *b = s ? b2 : b1, *state = slot + (size_t)s * (taps - 1) * d;
#pragma unroll
        for (int i = 0; i < PT; ++i) {
            const int c = (threadIdx.x + T * i) * V;
            if (c >= d) continue;
            load_some<float, V, WIDE>(w + c, wv[s][i]);
            load_some<float, V, WIDE>(b + c, bv[s][i]);
            const float *kc = cw + ((size_t)s * d + c) * taps;
            if constexpr (WIDE && TAPS > 0) {                              // V * TAPS numbers in a row: TAPS pieces of four
#pragma unroll
                for (int q = 0; q < TAPS; ++q) {
                    float piece[4];
                    load_as_f32<float, 4>(kc + 4 * q, piece);
#pragma unroll
                    for (int u = 0; u < 4; ++u) k[s][i][(4 * q + u) / TAPS][(4 * q + u) % TAPS] = piece[u];
                }
            } else {
#pragma unroll
                for (int e = 0; e < V; ++e)
#pragma unroll
                    for (int j = 0; j < MOST; ++j)
                        if (j < taps) k[s][i][e][j] = kc[e * taps + j];
            }
#pragma unroll
            for (int j = 0; j < MOST - 1; ++j) {                     // row j of the state lies taps - 1 - j positions before the token
#pragma unroll
                for (int e = 0; e < V; ++e) old[s][i][j][e] = 0.f;
                if (j < taps - 1 && pos - (taps - 1 - j) >= 0) load_some<float, V, WIDE>(state + (size_t)j * d + c, old[s][i][j]);
            }
        }
    }
    take_row<D, T, V, PT, WIDE>(x + (size_t)r * d, delta, r, d, eps, v, mean, rstd, scratch);
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        if (s >= sets) break;
        float *state = slot + (size_t)s * (taps - 1) * d;
#pragma unroll
        for (int i = 0; i < PT; ++i) {
            const int c = (threadIdx.x + T * i) * V;
            if (c >= d) continue;
            float h[V], acc[V];
#pragma unroll
            for (int e = 0; e < V; ++e) acc[e] = h[e] = (v[i][e] - mean) * rstd * wv[s][i][e] + bv[s][i][e];
            // (the order of short_conv_kernel's additions)
#pragma unroll
            for (int j = 0; j < MOST; ++j) {
                if (j >= taps) break;
#pragma unroll
                for (int e = 0; e < V; ++e) acc[e] += k[s][i][e][j] * (j == taps - 1 ? h[e] : old[s][i][j < MOST - 1 ? j : 0][e]);
                if (j > 0 && j < taps - 1) store_some<float, V, WIDE>(state + (size_t)(j - 1) * d + c, old[s][i][j < MOST - 1 ? j : 0]);     // row j becomes row j - 1
            }
            if (taps > 1) store_some<float, V, WIDE>(state + (size_t)(taps - 2) * d + c, h);
            store_some<TO, V, WIDE>(out + s * set_stride_out + (size_t)r * d + c, acc);
        }
    }
}

LCU_API int lcu_norm_conv_single(float *x, const void *delta, int delta_type, int planes, const float *w1, const float *b1,
                                 const float *w2, const float *b2, const float *cw, float *state, void *out, int out_type,
                                 const int *ctx_len, const int *state_slot, int n, int d, int taps, int sets, float eps,
                                 hipStream_t stream) {
    if (n <= 0) return LCU_OK;
    if (d <= 0 || d > 2048 || taps < 1 || taps > 8 || sets < 1 || sets > 2 || !w1 || !b1 || (sets == 2 && (!w2 || !b2)) ||
        !cw || (taps > 1 && !state) || (delta && planes <= 0))
        return LCU_BAD_ARGUMENT;
    const size_t stride = (size_t)n * d;
    dim3 grid(n);
    const int dt = delta ? delta_type : LCU_F32;
    const bool wide = four_ok(x, LCU_F32) && four_ok(delta, dt) && four_ok(w1, LCU_F32) && four_ok(b1, LCU_F32) &&
                      four_ok(w2, LCU_F32) && four_ok(b2, LCU_F32) && four_ok(cw, LCU_F32) && four_ok(state, LCU_F32) && four_ok(out, out_type);
#define ROW(TD, TO, T, V, PT, WIDE, TAPS) norm_conv_single_kernel<PlanesOf<TD>, TO, T, V, PT, WIDE, TAPS><<<grid, dim3(T), 0, stream>>>(x, PlanesOf<TD>{(const TD *)delta, planes, stride}, w1, b1, w2, b2, cw, state, (TO *)out, stride, ctx_len, state_slot, d, taps, sets, eps)
#define SIZED(TD, TO, V, PT, WIDE, TAPS) do { if (d <= 1024) ROW(TD, TO, 256, V, PT, WIDE, TAPS); else ROW(TD, TO, 512, V, PT, WIDE, TAPS); } while (0)
#define GO(TD, TO)                                                      \
    do {                                                                \
        if (d % 4 && d <= 256) ROW(TD, TO, 256, 1, 1, false, 0);        \
        else if (d % 4 && d <= 1024) ROW(TD, TO, 512, 1, 2, false, 0);  \
        else if (d % 4) ROW(TD, TO, 512, 1, 4, false, 0);               \
        else if (!wide) SIZED(TD, TO, 4, 1, false, 0);                  \
        else if (taps == 1) SIZED(TD, TO, 4, 1, true, 1);               \
        else if (taps == 2) SIZED(TD, TO, 4, 1, true, 2);               \
        else if (taps == 3) SIZED(TD, TO, 4, 1, true, 3);               \
        else if (taps == 4) SIZED(TD, TO, 4, 1, true, 4);               \
        else if (taps == 5) SIZED(TD, TO, 4, 1, true, 5);               \
        else if (taps == 6) SIZED(TD, TO, 4, 1, true, 6);               \
        else if (taps == 7) SIZED(TD, TO, 4, 1, true, 7);               \
        else SIZED(TD, TO, 4, 1, true, 8);                              \
    } while (0)
    if (dt == LCU_F32 && out_type == LCU_F32) GO(float, float);
    else if (dt == LCU_F32 && out_type == LCU_BF16) GO(float, bf16_t);
    else if (dt == LCU_BF16 && out_type == LCU_F32) GO(bf16_t, float);
    else if (dt == LCU_BF16 && out_type == LCU_BF16) GO(bf16_t, bf16_t);
    else return LCU_BAD_ARGUMENT;
#undef SIZED
#undef ROW
#undef GO
    LCU_LAUNCH_CHECK();
    return LCU_OK;
}

// The same with a token's experts' sum (in host memory; type: of the model, and of out) as delta.  d a multiple of 4, everything aligned for four.
LCU_API int lcu_norm_conv_single_pairs(float *x, const PairSum *pairs, int type, const float *w1, const float *b1, const float *w2, const float *b2,
                                       const float *cw, float *state, void *out, const int *ctx_len, const int *state_slot, int n, int d, int taps, int sets,
                                       float eps, hipStream_t stream) {
    if (n <= 0) return LCU_OK;
    if (!x || !pairs || d > 2048 || taps < 1 || taps > 8 || sets < 1 || sets > 2 || !w1 || !b1 || (sets == 2 && (!w2 || !b2)) || !cw || (taps > 1 && !state) ||
        !pair_sum_ok(*pairs, d) || !four_ok(x, LCU_F32) || !four_ok(w1, LCU_F32) || !four_ok(b1, LCU_F32) || !four_ok(w2, LCU_F32) || !four_ok(b2, LCU_F32) ||
        !four_ok(cw, LCU_F32) || !four_ok(state, LCU_F32) || !four_ok(out, type))
        return LCU_BAD_ARGUMENT;
    const size_t stride = (size_t)n * d;
#define ROW(T_, T, TAPS) norm_conv_single_kernel<PairsOf<T_>, T_, T, 4, 1, true, TAPS><<<dim3(n), dim3(T), 0, stream>>>(x, PairsOf<T_>{*pairs}, w1, b1, w2, b2, cw, state, (T_ *)out, stride, ctx_len, state_slot, d, taps, sets, eps)
#define SIZED(T_, TAPS) do { if (d <= 1024) ROW(T_, 256, TAPS); else ROW(T_, 512, TAPS); } while (0)
#define GO(T_)                              \
    do {                                    \
        if (taps == 2) SIZED(T_, 2);        \
        else if (taps == 3) SIZED(T_, 3);   \
        else if (taps == 4) SIZED(T_, 4);   \
        else SIZED(T_, 0);                  \
    } while (0)
    if (type == LCU_BF16) GO(bf16_t);
    else if (type == LCU_F32) GO(float);
    else return LCU_BAD_ARGUMENT;
#undef GO
#undef SIZED
#undef ROW
    LCU_LAUNCH_CHECK();
    return LCU_OK;
}
