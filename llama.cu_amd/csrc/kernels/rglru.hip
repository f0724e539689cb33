// The recurrent block with a real-gated linear recurrent unit.  The mixer's product gives, per token, two branches
// of `width` channels, yin and xin (bias added here).  Then, per channel c and in 32-bit:
//
//   u   = conv_b + sum_j conv[c, j] * xin[t - taps + 1 + j]              (causal; rows before the request's start are zeros)
//   r   = sigmoid(Wa[b] u_b + ba),  i = sigmoid(Wi[b] u_b + bi)          (the channels in `blocks` equal parts, a square matrix each)
//   a   = exp(-c_exp * r * softplus(lam)),   S <- a * S + sqrt(1 - a^2) * i * u
//   out = S * gelu_tanh(yin)
//
// Per request the state is [taps, width] floats: rows 0 .. taps-2 the last taps-1 rows of xin (oldest first), row
// taps-1 the recurrence's S.  It is taken as zero where the request's first token of the step stands at position 0.
// In general two kernels: the convolution with the gates (a workgroup per tile of tokens, block of channels and tile of outputs; the
// block's two matrices are given transposed, [block][in][out], so that the lanes read neighbours), and the scan (a
// thread per request and channel walks the request's tokens in their order, then leaves the state; the state is read by
// the first kernel and written by the second alone).  Everything that does not depend on the token before (the gelu of
// the y branch too) is made in the first kernel, so that the chain carries one multiply-add and one product a token.  sqrt(1 - a^2) is
// taken as sqrt(-expm1(2 log a)): no cancellation where a is close to 1.
#include "common.h"

// Where (token t, channel c) stands in the scratch arrays a, gx and y: tiles of 64 channels, each tile's tokens one after
// the other, so that the scan's wave, which owns a tile, streams one contiguous run of memory (with rows of `width`
// floats all waves would walk the same few rows at the same time, and those rows lie in few memory channels).
__device__ __forceinline__ size_t tile_index(int t, int c, int n) {
    return ((size_t)(c >> 6) * n + t) * 64 + (c & 63);
}

__device__ __forceinline__ float gelu_tanh(float z) {
    return 0.5f * z * (1.0f + tanhf(0.7978845608028654f * (z + 0.044715f * z * z * z)));
}

// xin of channel c at token t (a row of the step), or what stood `m` tokens before the step's first token of the
// request (from the state: its row taps - 1 - m; zero before the request's start).
template <class TI>
__device__ __forceinline__ float conv_at(const TI *__restrict__ rows, int row_stride, int x_off, const float *__restrict__ bias,
                                         const float *__restrict__ conv_w, const float *__restrict__ conv_b,
                                         const float *__restrict__ st, int t, int t0, int first_pos, int c, int width, int taps) {
    float acc = conv_b ? conv_b[c] : 0.f;
    const float bx = bias ? bias[x_off + c] : 0.f;
    // no branch around a load: both places are read (at indices that exist) and one value is chosen, so that the loads of
    // all taps, and of the elements that a thread makes one after the other, are in flight together
    for (int j = 0; j < taps; ++j) {
        const int back = taps - 1 - j;                       // how many tokens before t
        const bool in_step = t - back >= t0;
        const int m = in_step ? 1 : t0 - (t - back);         // else: so many tokens before the step
        const bool in_state = !in_step && first_pos - m >= 0;
        const float here = to_f32(rows[(size_t)(in_step ? t - back : t) * row_stride + x_off + c]) + bx;
        const float before = st[(size_t)(in_state ? taps - 1 - m : 0) * width + c];
        acc += conv_w[(size_t)c * taps + j] * (in_step ? here : in_state ? before : 0.f);
    }
    return acc;
}

// The same for up to MOST taps, without a loop: the loads of all taps, and of the elements that a thread makes one after the other, are on
// their way together.
template <int MOST, class TI>
__device__ __forceinline__ float conv_few(const TI *__restrict__ rows, int row_stride, int x_off, const float *__restrict__ bias,
                                          const float *__restrict__ conv_w, const float *__restrict__ conv_b,
                                          const float *__restrict__ st, int t, int t0, int first_pos, int c, int width, int taps) {
    float here[MOST], before[MOST], w[MOST];
#pragma unroll
    for (int j = 0; j < MOST; ++j) {
        const int back = max(taps - 1 - j, 0), m = t0 - (t - back);
        here[j] = to_f32(rows[(size_t)(m <= 0 ? t - back : t) * row_stride + x_off + c]);
        before[j] = st[(size_t)(m > 0 && first_pos - m >= 0 ? taps - 1 - m : 0) * width + c];
        w[j] = conv_w[(size_t)c * taps + min(j, taps - 1)];
    }
    const float bx = bias ? bias[x_off + c] : 0.f;
    float acc = conv_b ? conv_b[c] : 0.f;
#pragma unroll
    for (int j = 0; j < MOST; ++j) {
        const int back = taps - 1 - j, m = t0 - (t - back);
        const float x = m <= 0 ? here[j] + bx : first_pos - m >= 0 ? before[j] : 0.f;
        acc = j < taps ? acc + w[j] * x : acc;
    }
    return acc;
}

constexpr int RG_TOK = 8;          // tokens a workgroup of the gates kernel takes
constexpr int RG_OUT = 32;         // output channels a workgroup takes
constexpr int RG_SLICES = 8;       // parts into which the sum over a block's input channels is cut (one per 32 threads)
constexpr int RG_AHEAD = 16;       // rows of the two matrices whose loads are on their way together
constexpr int RG_MAX_BS = 1024;    // channels of a block (LDS holds RG_TOK rows of them)

// The convolution and the gates.  A workgroup takes RG_TOK tokens, one block of channels and RG_OUT of its outputs: it
// makes u for all the block's channels of its tokens (in LDS; workgroups of the same block make the same u), then each
// of its eight groups of 32 threads sums over an eighth of the input channels, and the eight partial sums are added in
// a fixed order.  So a decoding step, with few tokens, still has blocks x (bs / 32) workgroups.  Latency bounds it: the
// matrices' rows are asked for before u is made, sixteen at a time, the next sixteen during the sums of these (one MI355X,
// 8 tokens, width 2048 in 16 blocks, 4 taps: 12.5 us with a loop over the taps and the gates' own vectors asked for at the
// end, 8.1 us now).
template <class TI>
__global__ void __launch_bounds__(RG_OUT * RG_SLICES)
rglru_gates_kernel(const TI *__restrict__ rows, int row_stride, int x_off, const float *__restrict__ bias,
                   const float *__restrict__ conv_w, const float *__restrict__ conv_b, const float *__restrict__ state,
                   const float *__restrict__ wa_t, const float *__restrict__ wi_t,
                   const float *__restrict__ ba, const float *__restrict__ bi, const float *__restrict__ lam, float c_exp,
                   float *__restrict__ a_out, float *__restrict__ gx_out, float *__restrict__ y_out, int y_off,
                   const int *__restrict__ q_start,
                   const int *__restrict__ ctx_len, const int *__restrict__ req_of_token, const int *__restrict__ state_slot,
                   int n, int width, int bs, int taps) {
    __shared__ __attribute__((aligned(16))) float us[RG_TOK][RG_MAX_BS];
    __shared__ float part[RG_SLICES][RG_TOK][2][RG_OUT];
    const int b = blockIdx.y, tok0 = blockIdx.x * RG_TOK, o0 = blockIdx.z * RG_OUT;
    const int nt = min(RG_TOK, n - tok0);
    const int og = threadIdx.x % RG_OUT, slice = threadIdx.x / RG_OUT, o = o0 + og;
    const int per = (bs + RG_SLICES - 1) / RG_SLICES;
    const int i0 = slice * per, i1 = min(bs, i0 + per);
    const float *wa = wa_t + (size_t)b * bs * bs + min(o, bs - 1), *wi = wi_t + (size_t)b * bs * bs + min(o, bs - 1);
    const bool fours = per % 4 == 0 && bs % 4 == 0;
    float a[2][RG_AHEAD], g[2][RG_AHEAD];
    auto fetch = [&](int u, int i) {                 // (a row beyond the end is the last one, and is not used)
#pragma unroll
        for (int e = 0; e < RG_AHEAD; ++e) {
            a[u][e] = wa[(size_t)min(i + e, bs - 1) * bs];
            g[u][e] = wi[(size_t)min(i + e, bs - 1) * bs];
        }
    };
    if (fours) fetch(0, i0);                         // on their way while u is made
    // what a thread needs in the end for its token (its slice's number) and channel
    const int c = b * bs + min(o, bs - 1);
    const size_t y_at = (size_t)(tok0 + min(slice, nt - 1)) * row_stride + y_off + c;
    const float l = lam[c], ba_c = ba[c], bi_c = bi[c], y_in = to_f32(rows[y_at]) + (bias ? bias[y_off + c] : 0.f);
    auto make = [&](int w, auto conv) {
        const int t = tok0 + w / bs, r = req_of_token[t], t0 = q_start[r];
        const int first_pos = ctx_len[r] - (q_start[r + 1] - t0);
        us[w / bs][w % bs] = conv(rows, row_stride, x_off, bias, conv_w, conv_b, state + (size_t)state_slot[r] * taps * width, t, t0,
                                  first_pos, b * bs + w % bs, width, taps);
    };
    // (the tokens that there are: the rows of us beyond them hold zeros, whose sums are not used)
    if (taps == 1) {
#pragma unroll 4
        for (int w = threadIdx.x; w < nt * bs; w += RG_OUT * RG_SLICES) make(w, conv_few<1, TI>);
    } else if (taps == 2) {
#pragma unroll 4
        for (int w = threadIdx.x; w < nt * bs; w += RG_OUT * RG_SLICES) make(w, conv_few<2, TI>);
    } else if (taps <= 4) {
#pragma unroll 4
        for (int w = threadIdx.x; w < nt * bs; w += RG_OUT * RG_SLICES) make(w, conv_few<4, TI>);
    } else {
        for (int w = threadIdx.x; w < nt * bs; w += RG_OUT * RG_SLICES) make(w, conv_at<TI>);
    }
    for (int w = nt * bs + threadIdx.x; w < RG_TOK * bs; w += RG_OUT * RG_SLICES) us[w / bs][w % bs] = 0.f;
    __syncthreads();
    float ra[RG_TOK], ri[RG_TOK];
#pragma unroll
    for (int tt = 0; tt < RG_TOK; ++tt) ra[tt] = ri[tt] = 0.f;
    if (fours) {
        for (int i = i0; i < i1; i += 2 * RG_AHEAD) {
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const int j = i + u * RG_AHEAD;
                if (j >= i1) break;
                if (j + RG_AHEAD < i1) fetch(u ^ 1, j + RG_AHEAD);
#pragma unroll
                for (int q = 0; q < RG_AHEAD; q += 4) {
                    if (j + q >= i1) break;
#pragma unroll
                    for (int tt = 0; tt < RG_TOK; ++tt) {
                        const float4 x = *(const float4 *)&us[tt][j + q];
                        ra[tt] += a[u][q] * x.x; ra[tt] += a[u][q + 1] * x.y; ra[tt] += a[u][q + 2] * x.z; ra[tt] += a[u][q + 3] * x.w;
                        ri[tt] += g[u][q] * x.x; ri[tt] += g[u][q + 1] * x.y; ri[tt] += g[u][q + 2] * x.z; ri[tt] += g[u][q + 3] * x.w;
                    }
                }
            }
        }
    } else {
        for (int i = i0; i < i1; ++i) {
            const float wa1 = wa[(size_t)i * bs], wi1 = wi[(size_t)i * bs];
#pragma unroll
            for (int tt = 0; tt < RG_TOK; ++tt) {
                ra[tt] += wa1 * us[tt][i];
                ri[tt] += wi1 * us[tt][i];
            }
        }
    }
#pragma unroll
    for (int tt = 0; tt < RG_TOK; ++tt) {
        part[slice][tt][0][og] = ra[tt];
        part[slice][tt][1][og] = ri[tt];
    }
    __syncthreads();
    const int tt = slice;                                     // eight slices, eight tokens: a thread finishes one token's channel
    if (o >= bs || tt >= nt) return;
    float sa = 0.f, si = 0.f;
#pragma unroll
    for (int k = 0; k < RG_SLICES; ++k) {
        sa += part[k][tt][0][og];
        si += part[k][tt][1][og];
    }
    const float sp = l > 20.f ? l : log1pf(expf(l));          // softplus
    const float r = 1.0f / (1.0f + expf(-(sa + ba_c)));
    const float gate = 1.0f / (1.0f + expf(-(si + bi_c)));
    const float log_a = -c_exp * r * sp;
    const float mult = sqrtf(-expm1f(2.0f * log_a));
    a_out[tile_index(tok0 + tt, c, n)] = expf(log_a);
    gx_out[tile_index(tok0 + tt, c, n)] = mult * gate * us[tt][o];
    y_out[tile_index(tok0 + tt, c, n)] = gelu_tanh(y_in);
}

constexpr int RG_BATCH = 16;       // tokens whose loads the scan has in flight at a time
constexpr int RG_RUNS = 16;        // runs into which the scan cuts a request that feeds many tokens
constexpr int RG_LONG = 512;       // from so many tokens on

// The same for many tokens: a workgroup takes RG_ROWS tokens and one block of channels, makes u once, and every thread
// sums over all input channels for its outputs, in one run (the sliced kernel adds eight partial sums: a token's gates
// differ between the two by rounding).
constexpr int RG_ROWS = 16;
constexpr int RG_FEW_ROWS = 64;    // up to so many tokens a step the sliced kernel runs (more workgroups), beyond it this one

template <class TI>
__global__ void __launch_bounds__(256)
rglru_gates_rows_kernel(const TI *__restrict__ rows, int row_stride, int x_off, const float *__restrict__ bias,
                        const float *__restrict__ conv_w, const float *__restrict__ conv_b, const float *__restrict__ state,
                        const float *__restrict__ wa_t, const float *__restrict__ wi_t,
                        const float *__restrict__ ba, const float *__restrict__ bi, const float *__restrict__ lam, float c_exp,
                        float *__restrict__ a_out, float *__restrict__ gx_out, float *__restrict__ y_out, int y_off,
                        const int *__restrict__ q_start,
                        const int *__restrict__ ctx_len, const int *__restrict__ req_of_token, const int *__restrict__ state_slot,
                        int n, int width, int bs, int taps) {
    extern __shared__ __attribute__((aligned(16))) float us_rows[];       // [RG_ROWS][bs4], bs4 = bs rounded up to 4
    const int bs4 = (bs + 3) / 4 * 4;
    const int b = blockIdx.y, tok0 = blockIdx.x * RG_ROWS;
    const int nt = min(RG_ROWS, n - tok0);
#pragma unroll 4
    for (int w = threadIdx.x; w < RG_ROWS * bs4; w += blockDim.x) {
        const int tt = w / bs4, i = w % bs4;
        float u = 0.f;
        if (tt < nt && i < bs) {
            const int t = tok0 + tt, r = req_of_token[t], t0 = q_start[r];
            const int first_pos = ctx_len[r] - (q_start[r + 1] - t0);
            u = conv_at(rows, row_stride, x_off, bias, conv_w, conv_b, state + (size_t)state_slot[r] * taps * width, t, t0,
                        first_pos, b * bs + i, width, taps);
        }
        us_rows[w] = u;
    }
    __syncthreads();
    for (int o = threadIdx.x; o < bs; o += blockDim.x) {
        const float *wa = wa_t + (size_t)b * bs * bs + o, *wi = wi_t + (size_t)b * bs * bs + o;
        float ra[RG_ROWS], ri[RG_ROWS];
#pragma unroll
        for (int tt = 0; tt < RG_ROWS; ++tt) ra[tt] = ri[tt] = 0.f;
        int i = 0;
        for (; i + 4 <= bs; i += 4) {
            float a[4], g[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) { a[e] = wa[(size_t)(i + e) * bs]; g[e] = wi[(size_t)(i + e) * bs]; }
#pragma unroll
            for (int tt = 0; tt < RG_ROWS; ++tt) {
                const float4 u = *(const float4 *)&us_rows[tt * bs4 + i];
                ra[tt] += a[0] * u.x; ra[tt] += a[1] * u.y; ra[tt] += a[2] * u.z; ra[tt] += a[3] * u.w;
                ri[tt] += g[0] * u.x; ri[tt] += g[1] * u.y; ri[tt] += g[2] * u.z; ri[tt] += g[3] * u.w;
            }
        }
        for (; i < bs; ++i) {
            const float a = wa[(size_t)i * bs], g = wi[(size_t)i * bs];
#pragma unroll
            for (int tt = 0; tt < RG_ROWS; ++tt) {
                ra[tt] += a * us_rows[tt * bs4 + i];
                ri[tt] += g * us_rows[tt * bs4 + i];
            }
        }
        const int c = b * bs + o;
        const float l = lam[c];
        const float sp = l > 20.f ? l : log1pf(expf(l));          // softplus
        const float bias_a = ba[c], bias_i = bi[c];
#pragma unroll
        for (int tt = 0; tt < RG_ROWS; ++tt) {
            if (tt < nt) {
                const float r = 1.0f / (1.0f + expf(-(ra[tt] + bias_a)));
                const float gate = 1.0f / (1.0f + expf(-(ri[tt] + bias_i)));
                const float log_a = -c_exp * r * sp;
                const float mult = sqrtf(-expm1f(2.0f * log_a));
                a_out[tile_index(tok0 + tt, c, n)] = expf(log_a);
                gx_out[tile_index(tok0 + tt, c, n)] = mult * gate * us_rows[tt * bs4 + o];
                y_out[tile_index(tok0 + tt, c, n)] = gelu_tanh(to_f32(rows[(size_t)(tok0 + tt) * row_stride + y_off + c]) + (bias ? bias[y_off + c] : 0.f));
            }
        }
    }
}

// Blocks of a multiple of sixteen channels, up to RG_MFMA_BS: the gates' products on the 32-bit matrix instruction.  It adds its four products one
// after the other, each multiplication and addition rounded once, as a chain of fmaf does (131,072 sums of each of several ranges compared, bit for
// bit); so its instructions take the input channels in their order, and the sums have the bits of the kernels above.  Lane (l, g) of 16 x 4 brings,
// of the sixteen k that four instructions take, those with k % 4 = g: the matrices stand in that order (lcu_rglru), so that a wave's load is 1 KB in
// one piece, and u lies in LDS so that a lane's four are side by side (rg_place).
//
// Many tokens: a workgroup takes 16 TT tokens and a block of channels, makes u for them (in LDS), and each of its waves takes 16 output
// channels of both gates at a time.  One MI355X, width 2048 in 16 blocks, 4 taps, with the scan behind it: 8 requests of 235 tokens 71 us (a thread
// an output channel and the sums on the vector unit: 108), 65 tokens 19 (47).  The matrix instructions are 14 us of the first, the functions (exp, expm1,
// tanh) 15, the scan 30.
constexpr int RG_MFMA_BS = 192, RG_MFMA_TAPS = 4, RG_MFMA_WIDE = 256, RG_MFMA_THREADS = 256;
typedef __attribute__((ext_vector_type(4))) float rg_f32x4;

// where input channel i of a block stands in LDS
__device__ __forceinline__ int rg_place(int i) { return (i & ~15) + 4 * (i & 3) + ((i >> 2) & 3); }

// the matrices' four pieces from input channel k0 on for 16 output channels (beyond the end: pieces that are not used)
__device__ __forceinline__ void rg_fetch(rg_f32x4 (&w)[2][4], const float *__restrict__ gates, int block, int tile, int tiles, int lane, int k0) {
    const float *at = gates + (size_t)(block * tiles + tile) * tiles * 512 + 4 * lane;
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int q = 0; q < 2; ++q) w[q][j] = *(const rg_f32x4 *)(at + 512 * (k0 / 16 + j < tiles ? k0 / 16 + j : 0) + 256 * q);
}

template <class TI, int TT>
__global__ void __launch_bounds__(RG_MFMA_THREADS, 3)
rglru_gates_mfma_kernel(const TI *__restrict__ rows, int row_stride, int x_off, const float *__restrict__ bias,
                        const float *__restrict__ conv_w, const float *__restrict__ conv_b, const float *__restrict__ state,
                        const float *__restrict__ gates,
                        const float *__restrict__ ba, const float *__restrict__ bi, const float *__restrict__ lam, float c_exp,
                        float *__restrict__ a_out, float *__restrict__ gx_out, float *__restrict__ y_out, int y_off,
                        const int *__restrict__ q_start, const int *__restrict__ ctx_len, const int *__restrict__ req_of_token,
                        const int *__restrict__ state_slot, int n, int width, int bs, int taps) {
    constexpr int TOK = 16 * TT, STEP = 64;                               // tokens; input channels whose columns are asked for together
    extern __shared__ __attribute__((aligned(16))) float us_tile[];       // [TOK][ld]
    const int ld = bs + 4;
    const int b = blockIdx.y, tok0 = blockIdx.x * TOK, nt = min(TOK, n - tok0);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l16 = lane & 15, g = lane >> 4;
    const int tiles = bs / 16, waves = RG_MFMA_THREADS / WAVE;
    rg_f32x4 w[2][4];
    rg_fetch(w, gates, b, min(wave, tiles - 1), tiles, lane, 0);
    // ---- u
    if (TT > 1 || taps <= RG_MFMA_TAPS) {
        // a thread walks a run of the tokens for one channel, with the tokens before it at hand, sixteen at a time
        __shared__ int first_row[TOK], ahead[TOK], slot_of[TOK];          // of a token's request: its first row, the tokens before that, its slot
        if (threadIdx.x < TOK) {
            const int r = req_of_token[tok0 + min((int)threadIdx.x, nt - 1)], t0 = q_start[r];
            first_row[threadIdx.x] = t0;
            ahead[threadIdx.x] = ctx_len[r] - (q_start[r + 1] - t0);
            slot_of[threadIdx.x] = state_slot[r];
        }
        __syncthreads();
        constexpr int BATCH = 16;
        const int runs = max(1, min(TOK / BATCH, RG_MFMA_THREADS / bs)), per = (TOK + runs - 1) / runs;
        for (int x = threadIdx.x; x < runs * bs; x += RG_MFMA_THREADS) {
            const int i = x % bs, c = b * bs + i, s0 = x / bs * per, s1 = min(TOK, s0 + per);
            const float bx = bias ? bias[x_off + c] : 0.f, cb = conv_b ? conv_b[c] : 0.f;
            float cw[RG_MFMA_TAPS], v[RG_MFMA_TAPS];                      // v[j]: the token taps - 1 - j before the next one
#pragma unroll
            for (int j = 0; j < RG_MFMA_TAPS; ++j) cw[j] = conv_w[(size_t)c * taps + min(j, taps - 1)];
            const TI *col = rows + x_off + c;
            v[0] = 0.f;
#pragma unroll
            for (int j = 0; j < RG_MFMA_TAPS - 1; ++j)
                v[j + 1] = to_f32(col[(size_t)max(0, min(n - 1, tok0 + s0 - (taps - 1 - j))) * row_stride]) + bx;
            for (int tb = s0; tb < s1; tb += BATCH) {
                float xs[BATCH];
#pragma unroll
                for (int e = 0; e < BATCH; ++e) xs[e] = to_f32(col[(size_t)min(n - 1, tok0 + tb + e) * row_stride]) + bx;
#pragma unroll
                for (int e = 0; e < BATCH; ++e) {
                    const int tt = tb + e, t = tok0 + tt;
                    if (tt >= s1) break;
#pragma unroll
                    for (int j = 0; j < RG_MFMA_TAPS - 1; ++j) v[j] = v[j + 1];
#pragma unroll
                    for (int j = 0; j < RG_MFMA_TAPS; ++j)
                        if (j == taps - 1) v[j] = xs[e];
                    float use[RG_MFMA_TAPS];
#pragma unroll
                    for (int j = 0; j < RG_MFMA_TAPS; ++j) use[j] = v[j];
                    const int t0 = first_row[tt];
                    if (t - t0 < taps - 1) {                              // (the tokens before it are not all in the step)
                        const float *st = state + (size_t)slot_of[tt] * taps * width + c;
#pragma unroll
                        for (int j = 0; j < RG_MFMA_TAPS - 1; ++j) {
                            const int m = t0 - (t - (taps - 1 - j));      // so many tokens before the step's first
                            if (j < taps - 1 && m > 0) use[j] = ahead[tt] - m >= 0 ? st[(size_t)(taps - 1 - m) * width] : 0.f;
                        }
                    }
                    float acc = cb;
#pragma unroll
                    for (int j = 0; j < RG_MFMA_TAPS; ++j)
                        if (j < taps) acc = fmaf(cw[j], use[j], acc);
                    us_tile[tt * ld + rg_place(i)] = tt < nt ? acc : 0.f;
                }
            }
        }
    } else {
        for (int x = threadIdx.x; x < TOK * bs; x += RG_MFMA_THREADS) {
            const int tt = x / bs, i = x % bs;
            float acc = 0.f;
            if (tt < nt) {
                const int t = tok0 + tt, r = req_of_token[t], t0 = q_start[r];
                const int first_pos = ctx_len[r] - (q_start[r + 1] - t0);
                acc = conv_at(rows, row_stride, x_off, bias, conv_w, conv_b, state + (size_t)state_slot[r] * taps * width, t, t0, first_pos, b * bs + i, width, taps);
            }
            us_tile[tt * ld + rg_place(i)] = acc;
        }
    }
    __syncthreads();
    // ---- the gates, 16 output channels at a time
    for (int tile = wave; tile < tiles; tile += waves) {
        const int o = 16 * tile + l16, c = b * bs + o;
        int lane_tok = 4 * g;                                             // (opaque: else sixteen tokens' addresses are made in front of the loop)
        asm volatile("" : "+v"(lane_tok));
        const float l = lam[c], ba_c = ba[c], bi_c = bi[c], by = bias ? bias[y_off + c] : 0.f;
        rg_f32x4 acc[2][TT];
#pragma unroll
        for (int m = 0; m < TT; ++m) acc[0][m] = acc[1][m] = rg_f32x4{0.f, 0.f, 0.f, 0.f};
        if (tile != wave) rg_fetch(w, gates, b, tile, tiles, lane, 0);
        for (int k = 0; k < bs; k += STEP) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if (k + 16 * j >= bs) break;
#pragma unroll
                for (int m = 0; m < TT; ++m) {
                    const rg_f32x4 x = *(const rg_f32x4 *)(us_tile + (16 * m + l16) * ld + k + 16 * j + 4 * g);
#pragma unroll
                    for (int e = 0; e < 4; ++e)
#pragma unroll
                        for (int q = 0; q < 2; ++q) acc[q][m] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[e], w[q][j][e], acc[q][m], 0, 0, 0);
                }
            }
            if (k + STEP < bs) rg_fetch(w, gates, b, tile, tiles, lane, k + STEP);
        }
        asm volatile("" : "+v"(lane_tok));
        float y_in[TT][4];
#pragma unroll
        for (int m = 0; m < TT; ++m)
#pragma unroll
            for (int r = 0; r < 4; ++r) y_in[m][r] = to_f32(rows[(size_t)min(n - 1, tok0 + 16 * m + lane_tok + r) * row_stride + y_off + c]);
        const float sp = l > 20.f ? l : log1pf(expf(l));                  // softplus
#pragma unroll
        for (int m = 0; m < TT; ++m)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int tt = 16 * m + lane_tok + r, t = tok0 + tt;
                if (tt >= nt) continue;
                const float gr = 1.0f / (1.0f + expf(-(acc[0][m][r] + ba_c)));
                const float gate = 1.0f / (1.0f + expf(-(acc[1][m][r] + bi_c)));
                const float log_a = -c_exp * gr * sp;
                const float mult = sqrtf(-expm1f(2.0f * log_a));
                a_out[tile_index(t, c, n)] = expf(log_a);
                gx_out[tile_index(t, c, n)] = mult * gate * us_tile[tt * ld + rg_place(o)];
                y_out[tile_index(t, c, n)] = gelu_tanh(y_in[m][r] + by);
            }
    }
}

// A step in which every request feeds one token (token i is request i's): the gates as above, the recurrence's step and the state's update in one
// kernel.  A workgroup takes four tokens and a block of channels; whatever of a slot's state belongs to a channel is read and written by
// its threads alone.  A wave takes 16 output channels, whose matrices it asks for in front of everything; then a thread an element for the functions,
// which with the lanes that hold the sums were four one after the other, most of them of tokens that are not there.  The sums are
// those of `slices` equal parts of the input channels, added in their order: RG_SLICES up to RG_FEW_ROWS tokens, one beyond, as the kernels above have them, so
// that a token's bits do not depend on what else a step of so many tokens holds.  32-bit rows whose fours are aligned (the layer's), up to four taps, slices of whole matrix
// instructions.  Latency bounds it: two trips to memory (four while the states' numbers were asked for behind the matrices: 8.6 us of a launch in a model of width 2048 with 8 requests,
// now 8.0), 1.7 us of matrix instructions.  One MI355X, 4 taps, us alone beside the sliced kernel and the scan, with four trips: width 2048
// in 16 blocks 8.0 / 10.9 with 8 requests, 8.8 / 14.0 with 64; width 1024 in 16 blocks 5.8 / 8.5 with 8.  (Blocks of 192 channels, whose twelve sixteens do not fit the
// registers: 24 / 10.4.)
constexpr int RG_ONE_TOK = 4, RG_ONE_BS = 128;

// MOST: sixteens of channels at most.  Up to 64 channels a workgroup has a wave for each sixteen, and so a thread for each element of its four tokens (with eight waves always, those without a
// matrix, which ask for a neighbour's, made blocks of 32 channels slower than four trips: width 2048 in 64 blocks, 64 requests, 10.2 us and 9.2; now 5.9), beyond it eight (96 channels, 256 requests:
// 17.3 us, with six waves, of which two SIMDs hold two, 20.1).
constexpr int rg_one_threads(int bs) { return bs <= 64 ? RG_ONE_TOK * bs : RG_ONE_TOK * RG_ONE_BS; }
template <class T, int MOST>
__global__ void __launch_bounds__(rg_one_threads(16 * MOST))
rglru_single_kernel(const float *__restrict__ rows, int row_stride, int y_off, int x_off, const float *__restrict__ bias,
                    const float *__restrict__ conv_w, const float *__restrict__ conv_b, float *__restrict__ state,
                    const float *__restrict__ gates, const float *__restrict__ ba, const float *__restrict__ bi, const float *__restrict__ lam, float c_exp,
                    T *__restrict__ out, const int *__restrict__ ctx_len, const int *__restrict__ state_slot, int n, int width, int bs, int taps, int slices) {
    __shared__ __attribute__((aligned(16))) float us_tile[RG_ONE_TOK * (16 * MOST + 4)], sums[2][RG_ONE_TOK][16 * MOST];
    const int ld = bs + 4, b = blockIdx.y, tok0 = blockIdx.x * RG_ONE_TOK, nt = min(RG_ONE_TOK, n - tok0);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l16 = lane & 15, g = lane >> 4;
    const int tiles = bs / 16, each = bs / 4 / slices;                    // matrix instructions a slice
    // ---- what a thread asks for: under no condition (threads without work ask for a neighbour's), as loads come back in order: the numbers of the states first, what hangs on
    // nothing, the matrices, and behind them what lies in the states
    auto load = [](const float *q) { return *(const rg_f32x4 *)q; };
    static_assert(RG_ONE_TOK * 16 == WAVE, "an element a thread, sixteen output channels a wave");
    const int x = min((int)threadIdx.x, nt * (bs / 4) - 1), tt = x / (bs / 4), i = x % (bs / 4) * 4, c = b * bs + i, t = tok0 + tt;      // u: four neighbouring channels of a token
    const int e_tt = min((int)threadIdx.x / bs, nt - 1), e_o = threadIdx.x % bs, e_t = tok0 + e_tt, e_c = b * bs + e_o;                // the recurrence: an element
    const bool e_in = (int)threadIdx.x / bs < nt;
    const int ctx = ctx_len[t], slot = state_slot[t], e_ctx = ctx_len[e_t], e_slot = state_slot[e_t];
    rg_f32x4 here = load(rows + (size_t)t * row_stride + x_off + c), old[RG_MFMA_TAPS - 1], acc = {}, zero = {};
    float cw[4 * RG_MFMA_TAPS];
    if (taps == 4) {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const rg_f32x4 four = load(conv_w + (size_t)c * 4 + 4 * k);
#pragma unroll
            for (int j = 0; j < 4; ++j) cw[4 * k + j] = four[j];
        }
    } else {
#pragma unroll
        for (int k = 0; k < 4; ++k)
#pragma unroll
            for (int j = 0; j < RG_MFMA_TAPS; ++j) cw[4 * k + j] = conv_w[(size_t)(c + k) * taps + min(j, taps - 1)];
    }
    if (conv_b) acc = load(conv_b + c);
    float x_bias[4] = {}, y_bias = 0.f;
    if (bias) {
#pragma unroll
        for (int k = 0; k < 4; ++k) x_bias[k] = bias[x_off + c + k];
        y_bias = bias[y_off + e_c];
    }
    const float e_lam = lam[e_c], e_ba = ba[e_c], e_bi = bi[e_c], y_in = rows[(size_t)e_t * row_stride + y_off + e_c];
    __builtin_amdgcn_sched_barrier(0);
    rg_f32x4 w[2][MOST];
    {
        const float *at = gates + (size_t)(b * tiles + min(wave, tiles - 1)) * tiles * 512 + 4 * lane;
#pragma unroll
        for (int j = 0; j < MOST; ++j)
#pragma unroll
            for (int q = 0; q < 2; ++q) w[q][j] = *(const rg_f32x4 *)(at + 512 * min(j, tiles - 1) + 256 * q);
    }
    __builtin_amdgcn_sched_barrier(0);
    float *st = state + (size_t)slot * taps * width + c;
#pragma unroll
    for (int j = 0; j < RG_MFMA_TAPS - 1; ++j) old[j] = load(st + (size_t)min(j, taps - 1) * width);
    float *e_at = state + ((size_t)e_slot * taps + taps - 1) * width + e_c;
    const float e_old = *e_at, e_s = e_ctx > 1 ? e_old : 0.f, e_y = y_in + y_bias;
    // ---- u
    if ((int)threadIdx.x < nt * (bs / 4)) {
        const int before = ctx - 1;                                       // how many tokens the request has behind it
#pragma unroll
        for (int k = 0; k < 4; ++k) here[k] += x_bias[k];
#pragma unroll
        for (int j = 0; j < RG_MFMA_TAPS; ++j) {
            const int back = taps - 1 - j;
            if (j < taps) {
                const rg_f32x4 v = back == 0 ? here : before >= back ? old[j < RG_MFMA_TAPS - 1 ? j : 0] : zero;
#pragma unroll
                for (int k = 0; k < 4; ++k) acc[k] = fmaf(cw[4 * k + j], v[k], acc[k]);
                if (j > 0) *(rg_f32x4 *)(st + (size_t)(j - 1) * width) = v;      // a row up; the oldest goes
            }
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) us_tile[tt * ld + rg_place(i + k)] = acc[k];
    }
    __syncthreads();
    // ---- the gates (the instruction's other rows are the last token's again)
    if (wave < tiles) {
        const float *up = us_tile + min(l16, nt - 1) * ld + 4 * g;
        const rg_f32x4 none = {0.f, 0.f, 0.f, 0.f};
        rg_f32x4 acc[2] = {none, none}, sum[2] = {none, none};
        int left = each;                                                  // instructions until the slice's sums are whole
#pragma unroll
        for (int j = 0; j < MOST; ++j) {
            if (j >= tiles) break;
            const rg_f32x4 x = *(const rg_f32x4 *)(up + 16 * j);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
#pragma unroll
                for (int q = 0; q < 2; ++q) acc[q] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[e], w[q][j][e], acc[q], 0, 0, 0);
                if (--left == 0) {
#pragma unroll
                    for (int q = 0; q < 2; ++q) {
                        sum[q] += acc[q];
                        acc[q] = none;
                    }
                    left = each;
                }
            }
        }
        if (g < RG_ONE_TOK / 4) {
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
                for (int r = 0; r < 4; ++r) sums[q][4 * g + r][16 * wave + l16] = sum[q][r];
        }
    }
    __syncthreads();
    if (e_in) {
        const float gr = 1.0f / (1.0f + expf(-(sums[0][e_tt][e_o] + e_ba)));
        const float gate = 1.0f / (1.0f + expf(-(sums[1][e_tt][e_o] + e_bi)));
        const float log_a = -c_exp * gr * (e_lam > 20.f ? e_lam : log1pf(expf(e_lam)));
        const float mult = sqrtf(-expm1f(2.0f * log_a));
        const float S = fmaf(expf(log_a), e_s, mult * gate * us_tile[e_tt * ld + rg_place(e_o)]);
        *e_at = S;
        out[(size_t)e_t * width + e_c] = from_f32<T>(S * gelu_tanh(e_y));
    }
}

// The recurrence over [s0, s1) from S, in the tokens' order; with WRITE the outputs too.  RG_BATCH tokens at a time: their
// loads go out together.  prod (if not null) receives the product of the decays.
template <class T, bool WRITE>
__device__ __forceinline__ float scan_run(const float *__restrict__ a, const float *__restrict__ gx, const float *__restrict__ y,
                                          T *__restrict__ out, int s0, int s1, int c, int n, int width, float S, float *prod) {
    float P = 1.f;
    int t = s0;
    for (; t + RG_BATCH <= s1; t += RG_BATCH) {
        float av[RG_BATCH], gv[RG_BATCH], yv[RG_BATCH];
#pragma unroll
        for (int e = 0; e < RG_BATCH; ++e) {
            av[e] = a[tile_index(t + e, c, n)];
            gv[e] = gx[tile_index(t + e, c, n)];
            if (WRITE) yv[e] = y[tile_index(t + e, c, n)];
        }
#pragma unroll
        for (int e = 0; e < RG_BATCH; ++e) {
            S = av[e] * S + gv[e];
            if (WRITE) out[(size_t)(t + e) * width + c] = from_f32<T>(S * yv[e]);
            else P *= av[e];
        }
    }
    for (; t < s1; ++t) {
        const float av = a[tile_index(t, c, n)];
        S = av * S + gx[tile_index(t, c, n)];
        if (WRITE) out[(size_t)t * width + c] = from_f32<T>(S * y[tile_index(t, c, n)]);
        else P *= av;
    }
    if (prod) *prod = P;
    return S;
}

// NSEG 1: a wave per 64 channels walks the request's tokens in their order.  NSEG > 1, for a request that feeds many
// tokens: the tokens are cut into NSEG runs, a wave each; every wave first walks its run from zero, which gives the run's
// effect on whatever state it starts from (S_end = P * S_start + B); then the runs' effects are chained, in order; then
// every wave walks its run again from its true start and writes.  (The recurrence is the same; the sums are made in
// another order, so the results differ from NSEG = 1 by rounding.)
template <class TI, class T, int NSEG>
__global__ void __launch_bounds__(64 * NSEG)
rglru_scan_kernel(const TI *__restrict__ rows, int row_stride, int y_off, int x_off, const float *__restrict__ bias,
                  const float *__restrict__ a, const float *__restrict__ gx, const float *__restrict__ y, float *__restrict__ state,
                  T *__restrict__ out, const int *__restrict__ q_start, const int *__restrict__ ctx_len,
                  const int *__restrict__ state_slot, int n, int width, int taps, int min_tokens) {
    __shared__ float eff[NSEG][2][64];
    const int r = blockIdx.y, lane = threadIdx.x % 64, seg = threadIdx.x / 64;
    const int c = blockIdx.x * 64 + lane;
    const int t0 = q_start[r], t1 = q_start[r + 1];
    // (a kernel of several runs leaves requests with few tokens to the kernel of one, and the other way round)
    if (t1 <= t0 || (NSEG > 1) != (t1 - t0 >= min_tokens)) return;
    const bool live = c < width;
    const int first_pos = ctx_len[r] - (t1 - t0);
    float *st = state + (size_t)state_slot[r] * taps * width;
    float S = (live && first_pos > 0) ? st[(size_t)(taps - 1) * width + c] : 0.f;
    if (NSEG == 1) {
        if (!live) return;
        S = scan_run<T, true>(a, gx, y, out, t0, t1, c, n, width, S, nullptr);
    } else {
        const int len = (t1 - t0 + NSEG - 1) / NSEG;
        const int s0 = min(t1, t0 + seg * len), s1 = min(t1, s0 + len);
        float P = 1.f, B = 0.f;
        if (live) B = scan_run<T, false>(a, gx, y, out, s0, s1, c, n, width, 0.f, &P);
        eff[seg][0][lane] = P;
        eff[seg][1][lane] = B;
        __syncthreads();
        for (int k = 0; k < seg; ++k) S = eff[k][0][lane] * S + eff[k][1][lane];
        if (!live) return;
        S = scan_run<T, true>(a, gx, y, out, s0, s1, c, n, width, S, nullptr);
        if (seg != NSEG - 1) return;                          // the last run's end is the request's
    }
    st[(size_t)(taps - 1) * width + c] = S;
    // the convolution's state: the last taps - 1 rows of xin, oldest first; where the step brought fewer, older rows move up
    const int q = t1 - t0;
    const float bx = bias ? bias[x_off + c] : 0.f;
    float keep[16];
    for (int k = 0; k < taps - 1; ++k) {
        const int back = taps - 1 - k;                           // row k is the one `back` tokens before the request's end
        float x = 0.f;
        if (back <= q) x = to_f32(rows[(size_t)(t1 - back) * row_stride + x_off + c]) + bx;
        else if (first_pos > 0) {
            const int old = k + q;                               // where that row stands in the state as the step found it
            if (old < taps - 1 && first_pos - (back - q) >= 0) x = st[(size_t)old * width + c];
        }
        keep[k] = x;
    }
    for (int k = 0; k < taps - 1; ++k) st[(size_t)k * width + c] = keep[k];
}

// rows: [n, row_stride] of in_type, yin at y_off and xin at x_off (width each); bias: null or float32 over the row's
// columns.  conv_w [width, taps], conv_b [width] (may be null), wa_t / wi_t [blocks, bs, bs] transposed ([in][out]),
// ba / bi / lam [width], all float32; gates (may be null): both matrices in the order in which the matrix instruction takes them, [blocks][bs / 16 output
// tiles][bs / 16 input tiles][2][64 lanes (l, g)][4]: output 16 tile + l, input 16 tile + 4 e + g, for bs a multiple of 16 up to 192 (read in steps of
// more than 64 tokens and of single tokens).  single: every request feeds one token.  state: float32 [slots, taps, width].  a, gx, y: float32 scratch of n * (width rounded up to 64) floats each.
// out: [n, width] of out_type.
LCU_API int lcu_rglru(const void *rows, int in_type, int row_stride, int y_off, int x_off, const float *bias,
                      const float *conv_w, const float *conv_b, const float *wa_t, const float *wi_t, const float *gates, const float *ba,
                      const float *bi, const float *lam, float c_exp, float *state, float *a, float *gx, float *y, void *out,
                      int out_type, const int *q_start, const int *ctx_len, const int *req_of_token, const int *state_slot,
                      int n, int n_req, int width, int blocks, int taps, int single, hipStream_t stream) {
    if (n <= 0 || n_req <= 0) return LCU_OK;
    if (width <= 0 || blocks <= 0 || width % blocks || width / blocks > RG_MAX_BS || taps < 1 || taps > 16 || n_req > 65535 ||
        !rows || !conv_w || !wa_t || !wi_t || !ba || !bi || !lam || !state || !a || !gx || !y || !out)
        return LCU_BAD_ARGUMENT;
    const int bs = width / blocks;
    if ((in_type != LCU_F32 && in_type != LCU_BF16) || (out_type != LCU_F32 && out_type != LCU_BF16) || (in_type == LCU_BF16 && out_type == LCU_F32))
        return LCU_BAD_ARGUMENT;
    const bool matrix = gates != nullptr;
    if (matrix && (bs % 16 || bs > RG_MFMA_BS || (uintptr_t)gates % 16)) return LCU_BAD_ARGUMENT;
    const int slices = n > RG_FEW_ROWS ? 1 : RG_SLICES;
    // (a matrix instruction's four input channels lie in one slice)
    if (matrix && single && n == n_req && taps <= RG_MFMA_TAPS && bs <= RG_ONE_BS && in_type == LCU_F32 && bs % (4 * slices) == 0 && x_off % 4 == 0 && row_stride % 4 == 0 &&
        ((uintptr_t)rows | (uintptr_t)conv_w | (uintptr_t)conv_b | (uintptr_t)state) % 16 == 0) {
#define ONE(T, MOST)                                                                                                                                                      \
    rglru_single_kernel<T, MOST><<<dim3((n + RG_ONE_TOK - 1) / RG_ONE_TOK, blocks), dim3(rg_one_threads(bs)), 0, stream>>>((const float *)rows, row_stride, y_off, x_off, bias, conv_w, \
                                                                              conv_b, state, gates, ba, bi, lam, c_exp, (T *)out, ctx_len, state_slot, n, width, bs, taps, slices)
#define STEP(T) do { if (bs <= 32) ONE(T, 2); else if (bs <= 64) ONE(T, 4); else if (bs <= 96) ONE(T, 6); else ONE(T, RG_ONE_BS / 16); } while (0)
        if (out_type == LCU_BF16) STEP(bf16_t);
        else STEP(float);
#undef STEP
#undef ONE
        LCU_LAUNCH_CHECK();
        return LCU_OK;
    }
    if (matrix && n > RG_FEW_ROWS) {
        // 64 tokens a workgroup where those are RG_MFMA_WIDE at least (the matrices are read for each), else 16; 16 with more taps, whose convolution is a chain of loads a
        // tap (8 requests of 235 tokens, width 2048 in 16 blocks, 5 taps: 95 us, with 64 tokens a workgroup 122, on the vector unit 113)
        const bool wide = taps <= RG_MFMA_TAPS && (long long)((n + 63) / 64) * blocks >= RG_MFMA_WIDE;
#define GATES(TI, TT)                                                                                                                          \
    rglru_gates_mfma_kernel<TI, TT><<<dim3((n + 16 * TT - 1) / (16 * TT), blocks), dim3(RG_MFMA_THREADS), 16 * TT * (bs + 4) * sizeof(float), stream>>>( \
        (const TI *)rows, row_stride, x_off, bias, conv_w, conv_b, state, gates, ba, bi, lam, c_exp, a, gx, y, y_off, q_start, ctx_len, req_of_token,      \
        state_slot, n, width, bs, taps)
        if (in_type == LCU_F32) { if (wide) GATES(float, 4); else GATES(float, 1); }
        else { if (wide) GATES(bf16_t, 4); else GATES(bf16_t, 1); }
#undef GATES
        LCU_LAUNCH_CHECK();
    } else if (n > RG_FEW_ROWS) {
        const int bs4 = (bs + 3) / 4 * 4;
        dim3 grid((n + RG_ROWS - 1) / RG_ROWS, blocks), block(bs >= 256 ? 256 : (bs + 63) / 64 * 64);
        const size_t lds = (size_t)RG_ROWS * bs4 * sizeof(float);
        if (in_type == LCU_F32)
            rglru_gates_rows_kernel<float><<<grid, block, lds, stream>>>((const float *)rows, row_stride, x_off, bias, conv_w, conv_b, state, wa_t, wi_t, ba, bi, lam, c_exp, a, gx, y, y_off, q_start, ctx_len, req_of_token, state_slot, n, width, bs, taps);
        else if (in_type == LCU_BF16)
            rglru_gates_rows_kernel<bf16_t><<<grid, block, lds, stream>>>((const bf16_t *)rows, row_stride, x_off, bias, conv_w, conv_b, state, wa_t, wi_t, ba, bi, lam, c_exp, a, gx, y, y_off, q_start, ctx_len, req_of_token, state_slot, n, width, bs, taps);
        else
            return LCU_BAD_ARGUMENT;
        LCU_LAUNCH_CHECK();
    } else {
        dim3 grid((n + RG_TOK - 1) / RG_TOK, blocks, (bs + RG_OUT - 1) / RG_OUT), block(RG_OUT * RG_SLICES);
        if (in_type == LCU_F32)
            rglru_gates_kernel<float><<<grid, block, 0, stream>>>((const float *)rows, row_stride, x_off, bias, conv_w, conv_b, state, wa_t, wi_t, ba, bi, lam, c_exp, a, gx, y, y_off, q_start, ctx_len, req_of_token, state_slot, n, width, bs, taps);
        else if (in_type == LCU_BF16)
            rglru_gates_kernel<bf16_t><<<grid, block, 0, stream>>>((const bf16_t *)rows, row_stride, x_off, bias, conv_w, conv_b, state, wa_t, wi_t, ba, bi, lam, c_exp, a, gx, y, y_off, q_start, ctx_len, req_of_token, state_slot, n, width, bs, taps);
        else
            return LCU_BAD_ARGUMENT;
        LCU_LAUNCH_CHECK();
    }
    {
        // two launches: requests that feed many tokens (if the step's size allows any) are cut into runs, the others not
        dim3 grid((width + 63) / 64, n_req);
#define GO(TI, T) do { rglru_scan_kernel<TI, T, 1><<<grid, dim3(64), 0, stream>>>((const TI *)rows, row_stride, y_off, x_off, bias, a, gx, y, state, (T *)out, q_start, ctx_len, state_slot, n, width, taps, RG_LONG); \
                       if (n >= RG_LONG) rglru_scan_kernel<TI, T, RG_RUNS><<<grid, dim3(64 * RG_RUNS), 0, stream>>>((const TI *)rows, row_stride, y_off, x_off, bias, a, gx, y, state, (T *)out, q_start, ctx_len, state_slot, n, width, taps, RG_LONG); } while (0)
        if (in_type == LCU_F32 && out_type == LCU_F32) GO(float, float);
        else if (in_type == LCU_F32 && out_type == LCU_BF16) GO(float, bf16_t);
        else if (in_type == LCU_BF16 && out_type == LCU_BF16) GO(bf16_t, bf16_t);
        else return LCU_BAD_ARGUMENT;
#undef GO
        LCU_LAUNCH_CHECK();
    }
    return LCU_OK;
}
