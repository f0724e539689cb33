// The generalised delta rule: a recurrent mixer whose state per head is a matrix S [dk, dv]
// (key channel, value channel) in 32-bit.  For every token, with per key channel a decay w, a
// removal rate a, the key k, its unit vector u = k / sqrt(sum(k^2) + 1e-6), the query r, and
// per value channel v:
//   S <- diag(w) S - (a * u) (u^T S) + k v^T        (decay and removal act on S as the token found it)
//   o  = S^T r
// Everything that enters the recurrence is 32-bit.  Three kernels:
//   prep  (parallel over tokens and heads): w, a * u, u, k, r as 32-bit vectors;
//           w = exp(-exp(-1/2) * sigmoid(w0 + W2 tanh(l))), l the row's low-rank projection,
//           a = sigmoid(a_lin + a_bias);
//   scan  (sequential over a request's tokens, parallel over requests, heads and value
//           channels: column j of S depends on column j alone, so a column stays in the registers
//           of its lanes from the request's first token of the step to its last);
//   out   (parallel): o of each head divided by its root mean square, times a weight, times
//           sigmoid(gate).
// A request that feeds many tokens in a step goes through chunks on the matrix cores instead of the scan (delta_chunks.h, which says when: from some
// 64 to 200 tokens on) if its outputs are rounded to bfloat16; 32-bit models keep the scan, whose bits do not depend on the cut of a prompt.
// A token's result depends on the tokens before it in its request only; portions that are scanned are folded in in an
// order of operations that does not depend on how the request was cut into them, chunks change roundings.  Where every request feeds one token
// the three are one kernel (the gated rule, with its convolution: two), with the same bits.
#include <limits.h>
#include "common.h"
#include "lane_moves.h"
#include "delta_chunks.h"

constexpr int MAX_RANK = 512;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;
constexpr float DECAY_SCALE = 0.6065306597126334f;      // exp(-1/2)

__device__ __forceinline__ float sigmoidf_(float z) { return 1.0f / (1.0f + expf(-z)); }

// proj: [n, row_stride] rows that hold r, k, a_lin (dk per head each) and the low-rank
// projection l (rank) at the given column offsets.  w2t: [rank, heads * dk], the decay's second matrix
// transposed.  prep: [n, heads, 5, dk] 32-bit.
// A workgroup per (TB tokens, head, 64 key channels), a wave per quarter of the rank: a value of w2t serves TB tokens.  (A workgroup
// per token and head read 4 dk rank bytes of w2t for it: 57 us for 2,048 tokens of 16 heads of 128 with a rank of 64.)  The
// sum over the rank is made of the quarters' four, whatever TB is.
template <class T, int TB>
__global__ void __launch_bounds__(256)
delta_prep_kernel(const T *__restrict__ proj, int row_stride, int off_r, int off_k, int off_a, int off_l,
                  const float *__restrict__ w2t, const float *__restrict__ w0,
                  const float *__restrict__ a_bias, float *__restrict__ prep, int n, int heads, int dk, int rank) {
    extern __shared__ __attribute__((aligned(16))) float th[];         // [rank][TB]
    __shared__ float part[4][TB][WAVE], inv[TB];
    const int t0 = blockIdx.x * TB, h = blockIdx.y, lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nt = min(TB, n - t0), i = blockIdx.z * WAVE + lane, c = h * dk + min(i, dk - 1);
    // EARLY: what does not wait for the others is asked for first, the wave's own tokens' values and the first of its quarter of w2t (one MI355X, 2,014 tokens of 16
    // heads of 128, rank 64: 40 us, 48 with every load where its value is used).  One token's four waves would ask for the same rows (16 tokens of 16 heads of 128, the whole rule: 10.9 us, 10.7 so)
    constexpr bool EARLY = TB > 1;
    constexpr int OWN = (TB + 3) / 4, FIRST = 16, SIDE = TB > 1 ? 4 : 1;
    const int quarter = (rank + 3) / 4, j0 = wave * quarter, j1 = min(rank, j0 + quarter);
    const float *w = w2t + c;                                 // (neighbouring lanes, neighbouring addresses)
    float kv[OWN], av[OWN], rv[OWN], ka[OWN], kb[OWN], wv[FIRST];
    if constexpr (EARLY) {
#pragma unroll
        for (int o = 0; o < OWN; ++o) {
            const T *row = proj + (size_t)(t0 + min(wave + 4 * o, nt - 1)) * row_stride, *k = row + off_k + h * dk;
            ka[o] = to_f32(k[min(lane, dk - 1)]);
            kb[o] = to_f32(k[min(lane + WAVE, dk - 1)]);
            kv[o] = to_f32(row[off_k + c]);
            av[o] = to_f32(row[off_a + c]);
            rv[o] = to_f32(row[off_r + c]);
        }
#pragma unroll
        for (int x = 0; x < FIRST; ++x) wv[x] = w[(size_t)max(min(j0 + x, j1 - 1), 0) * heads * dk];
    }
    // (the projection's values by fours: one after the other a rank of 256 is eight trips to memory.  With w2t by sixteens, the next behind them, the whole rule of 2,000 tokens and 16 heads
    // of 64 with 16 value columns, bfloat16, rank 64, 256 and 400: 124, 145 and 166 us; the compiler's eight at a time 124, 166 and 202)
    for (int x0 = threadIdx.x; x0 < rank * TB; x0 += 256 * SIDE) {
        float l[SIDE];
#pragma unroll
        for (int b = 0; b < SIDE; ++b) {
            const int x = min(x0 + 256 * b, rank * TB - 1);
            l[b] = to_f32(proj[(size_t)(t0 + min(x / rank, nt - 1)) * row_stride + off_l + x % rank]);
        }
#pragma unroll
        for (int b = 0; b < SIDE; ++b) {
            const int x = x0 + 256 * b, t = x / rank;
            if (x < rank * TB) th[x % rank * TB + t] = t < nt ? tanhf(l[b]) : 0.f;
        }
    }
#pragma unroll
    for (int o = 0; o < OWN; ++o) {
        const int t = wave + 4 * o;
        if (t >= nt) break;
        const T *row = proj + (size_t)(t0 + t) * row_stride + off_k + h * dk;
        float ss = 0.f;
        if constexpr (EARLY) {
            ss = lane < dk ? ka[o] * ka[o] : 0.f;
            if (lane + WAVE < dk) ss = fmaf(kb[o], kb[o], ss);
        }
        for (int x = lane + (EARLY ? 2 * WAVE : 0); x < dk; x += WAVE) {
            const float kk = to_f32(row[x]);
            ss = fmaf(kk, kk, ss);
        }
        ss = wave_sum_in_place(ss);
        if (lane == 0) inv[t] = 1.0f / sqrtf(ss + 1e-6f);
    }
    __syncthreads();
    float z[TB];
#pragma unroll
    for (int t = 0; t < TB; ++t) z[t] = 0.f;
    if constexpr (EARLY) {
        // sixteen at a time, the next on their way meanwhile
        for (int j = j0; j < j1; j += FIRST) {
            float next[FIRST];
            if (j + FIRST < j1) {
#pragma unroll
                for (int x = 0; x < FIRST; ++x) next[x] = w[(size_t)min(j + FIRST + x, j1 - 1) * heads * dk];
            }
            auto add = [&](int x) {
#pragma unroll
                for (int t = 0; t < TB; ++t) z[t] = fmaf(wv[x], th[(j + x) * TB + t], z[t]);
            };
            if (j + FIRST <= j1) {
#pragma unroll
                for (int x = 0; x < FIRST; ++x) add(x);
            } else {
#pragma unroll
                for (int x = 0; x < FIRST; ++x)
                    if (j + x < j1) add(x);
            }
#pragma unroll
            for (int x = 0; x < FIRST; ++x) wv[x] = next[x];
        }
    } else {
#pragma unroll 8
        for (int j = j0; j < j1; ++j) {
            const float v = w[(size_t)j * heads * dk];
#pragma unroll
            for (int t = 0; t < TB; ++t) z[t] = fmaf(v, th[j * TB + t], z[t]);
        }
    }
#pragma unroll
    for (int t = 0; t < TB; ++t) part[wave][t][lane] = z[t];
    __syncthreads();
    if (i >= dk) return;
#pragma unroll
    for (int o = 0; o < OWN; ++o) {
        const int t = wave + 4 * o;
        if (t >= nt) break;
        const float sum = (part[0][t][lane] + part[1][t][lane]) + (part[2][t][lane] + part[3][t][lane]);
        if constexpr (!EARLY) {
            const T *row = proj + (size_t)(t0 + t) * row_stride;
            kv[o] = to_f32(row[off_k + c]);
            av[o] = to_f32(row[off_a + c]);
            rv[o] = to_f32(row[off_r + c]);
        }
        const float u = kv[o] * inv[t];
        float *out = prep + ((size_t)(t0 + t) * heads + h) * 5 * dk;
        out[i] = expf(-DECAY_SCALE * sigmoidf_(w0[c] + sum));
        out[dk + i] = sigmoidf_(av[o] + a_bias[c]) * u;
        out[2 * dk + i] = u;
        out[3 * dk + i] = kv[o];
        out[4 * dk + i] = rv[o];
    }
}

// DK > 0 (a multiple of 16): one wave per (request, head, 16 or 8 value channels).  The wave's lanes are four groups of
// 16 (eight of 8 where DK is a multiple of 32): lane (g, j) keeps the part g of column j of S (key channels
// g * DK/groups .. + DK/groups - 1) in registers, so a token costs a lane DK/groups of each pass, and the two sums over
// key channels (u^T S and S^T r) cross the groups in the vector unit.  A request's tokens are one chain, so what a
// token costs a wave is what counts: more lanes a column make it shorter.  The tokens' five vectors go through LDS, eight tokens at a time (all lanes copy, each reads its
// quarter), the next eight tokens' are on their way meanwhile.
// DK == 0: any dk, one wave per (request, head, 64 value channels), the column stays in the state's memory.
// state: [slots, heads, dk, dv]; o: [n, heads * dv] 32-bit.

// The sum of the values that the lanes l, l + 16, l + 32 and l + 48 hold (and l + 8 of each, with eight groups), in all
// of them, always added in the same order.  The rows of 16 lanes are swapped in the vector unit (v_permlane16_swap,
// v_permlane32_swap): a shuffle through LDS takes far longer, and the recurrence waits for this value twice a token.
template <int GROUPS>
__device__ __forceinline__ float sum_over_groups(float x) {
    if (GROUPS == 8)            // eight groups of 8 lanes: first the two groups of a row of 16 (the row rotated by 8, in the vector unit too)
        x += __uint_as_float((unsigned)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(x), 0x128, 0xf, 0xf, false));
    const unsigned u = __float_as_uint(x);
    const auto a = __builtin_amdgcn_permlane16_swap(u, u, false, false);     // (rows 0 0 2 2, rows 1 1 3 3)
    const unsigned v = __float_as_uint(__uint_as_float(a[0]) + __uint_as_float(a[1]));
    const auto b = __builtin_amdgcn_permlane32_swap(v, v, false, false);     // (lower half twice, upper half twice)
    return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

template <class T, int DK>
constexpr int scan_groups() { return DK > 0 && DK % 32 == 0 ? 8 : 4; }

// GATED: the gated rule, whose decay g and rate beta are one number each per token and head and whose key is its unit
// key: S <- g S + u (v - (beta g) (u^T S)) with v the value times beta already.  A token then brings two vectors (u, r) and
// two numbers (g, beta g) instead of five vectors: prep rows are [u | r | g, beta g, log g, 0], 2 dk + 4 floats.
template <class T, int DK, bool GATED>
__global__ void __launch_bounds__(64)
delta_scan_kernel(const T *__restrict__ proj, int row_stride, int off_v, const float *__restrict__ vf, const float *__restrict__ prep,
                  float *__restrict__ state, size_t slot_stride, float *__restrict__ o, const int *__restrict__ q_start,
                  const int *__restrict__ ctx_len, const int *__restrict__ state_slot, int heads, int dk_rt, int dv, const int *__restrict__ done) {
    const int r = blockIdx.x, h = blockIdx.y;
    const int t0 = q_start[r], t1 = q_start[r + 1];
    if (done && done[r]) return;                             // it went through chunks
    const bool fresh = ctx_len[r] - (t1 - t0) == 0;          // the request's first token: the state starts at zero
    if constexpr (DK > 0) {
        constexpr int SCAN_GROUPS = scan_groups<T, DK>(), SCAN_COLS = WAVE / SCAN_GROUPS;
        constexpr int SL = DK / SCAN_GROUPS;                  // key channels of a lane
        constexpr int NV = GATED ? 2 : 5;                     // vectors of a token
        constexpr int ROW = NV * DK + (GATED ? 4 : 0);        // floats of a token's prep row
        constexpr int PER_LANE = (ROW + 63) / 64;
        constexpr int TB = DK <= 128 ? 8 : 4;                 // tokens whose vectors are brought in together
        const int g = threadIdx.x / SCAN_COLS, j = blockIdx.z * SCAN_COLS + threadIdx.x % SCAN_COLS;
        const bool live = j < dv;
        const int jj = live ? j : dv - 1;                     // lanes beyond dv compute along and store nothing
        float *col = state + (size_t)state_slot[r] * slot_stride + ((size_t)h * DK + g * SL) * dv + jj;   // S[g * SL + i][j] at col[i * dv]
        // a vector in LDS: the four groups' quarters, each followed by four floats of padding, so that the groups' reads of
        // their quarters (the same offset in each) fall into different banks
        constexpr int SLP = SL + 4, VEC = SCAN_GROUPS * SLP;
        __shared__ __attribute__((aligned(16))) float vec[2][TB][NV * VEC + (GATED ? 4 : 0)];
        float S[SL];
#pragma unroll
        for (int i = 0; i < SL; ++i) S[i] = fresh ? 0.f : col[(size_t)i * dv];
        // the vectors and values of the next TB tokens, on their way while the TB before them are folded in: a
        // token's own arithmetic is far shorter than a trip to memory
        float next[TB][PER_LANE], v_next[TB];
        const T *vp = proj + off_v + h * dv + jj;
        const float *vfp = vf ? vf + h * dv + jj : nullptr;         // the values as 32-bit rows [n, heads * dv] of their own
        auto fetch = [&](int t) {
#pragma unroll
            for (int b = 0; b < TB; ++b) {
                if (t + b >= t1) break;                       // (a step of one token brings in one token)
                const float *p = prep + ((size_t)(t + b) * heads + h) * ROW;
#pragma unroll
                for (int e = 0; e < PER_LANE; ++e) {
                    const int idx = e * 64 + threadIdx.x;
                    next[b][e] = idx < ROW ? p[idx] : 0.f;
                }
                v_next[b] = vfp ? vfp[(size_t)(t + b) * heads * dv] : to_f32(vp[(size_t)(t + b) * row_stride]);
            }
        };
        if (t0 < t1) fetch(t0);
        int turn = 0;
        for (int t = t0; t < t1; t += TB, turn ^= 1) {
            float v[TB];
#pragma unroll
            for (int b = 0; b < TB; ++b) {
                if (t + b >= t1) break;
                v[b] = v_next[b];
#pragma unroll
                for (int e = 0; e < PER_LANE; ++e) {
                    const int idx = e * 64 + threadIdx.x;
                    if (idx < NV * DK) vec[turn][b][idx / DK * VEC + idx % DK / SL * SLP + idx % SL] = next[b][e];
                    else if (GATED && idx < ROW) vec[turn][b][NV * VEC + idx - NV * DK] = next[b][e];
                }
            }
            __syncthreads();                                  // (the buffer of two turns ago was last read before the barrier of the turn between)
            if (t + TB < t1) fetch(t + TB);
#pragma unroll
            for (int b = 0; b < TB; ++b) {
                if (t + b >= t1) break;
                const float *W = vec[turn][b] + g * SLP, *AU = W + VEC, *U = GATED ? W : W + 2 * VEC, *K = W + 3 * VEC,
                            *R = GATED ? W + VEC : W + 4 * VEC;
                // four sums side by side in each pass (added in a fixed order): one chain of SL dependent additions
                // would be most of a token's time
                float us4[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int i = 0; i < SL; ++i) us4[i & 3] += U[i] * S[i];
                const float us = sum_over_groups<SCAN_GROUPS>((us4[0] + us4[1]) + (us4[2] + us4[3]));
                float acc4[4] = {0.f, 0.f, 0.f, 0.f};
                if constexpr (GATED) {
                    const float gd = vec[turn][b][NV * VEC], c = v[b] - vec[turn][b][NV * VEC + 1] * us;
#pragma unroll
                    for (int i = 0; i < SL; ++i) {
                        S[i] = __builtin_fmaf(gd, S[i], U[i] * c);       // (written out: the kernel for one token rounds alike)
                        acc4[i & 3] += S[i] * R[i];
                    }
                } else {
#pragma unroll
                    for (int i = 0; i < SL; ++i) {
                        S[i] = W[i] * S[i] - AU[i] * us + K[i] * v[b];
                        acc4[i & 3] += S[i] * R[i];
                    }
                }
                const float acc = sum_over_groups<SCAN_GROUPS>((acc4[0] + acc4[1]) + (acc4[2] + acc4[3]));
                if (live && g == 0) o[(size_t)(t + b) * heads * dv + h * dv + j] = acc;
            }
        }
        if (live) {
#pragma unroll
            for (int i = 0; i < SL; ++i) col[(size_t)i * dv] = S[i];
        }
    } else {
        const int dk = dk_rt, j = blockIdx.z * 64 + threadIdx.x;
        const bool live = j < dv;
        const int jj = live ? j : dv - 1;
        float *col = state + (size_t)state_slot[r] * slot_stride + ((size_t)h * dk) * dv + jj;     // S[i][j] at col[i * dv]
        if (fresh && live)
            for (int i = 0; i < dk; ++i) col[(size_t)i * dv] = 0.f;
        for (int t = t0; t < t1; ++t) {
            const float v = vf ? vf[(size_t)t * heads * dv + h * dv + jj] : to_f32(proj[(size_t)t * row_stride + off_v + h * dv + jj]);
            const float *p = prep + ((size_t)t * heads + h) * (GATED ? 2 * dk + 4 : 5 * dk);
            float us = 0.f, acc = 0.f;
            if constexpr (GATED) {
                for (int i = 0; i < dk; ++i) us += p[i] * col[(size_t)i * dv];
                const float gd = p[2 * dk], c = v - p[2 * dk + 1] * us;
                for (int i = 0; i < dk; ++i) {
                    const float s = gd * col[(size_t)i * dv] + p[i] * c;
                    if (live) col[(size_t)i * dv] = s;
                    acc += s * p[dk + i];
                }
            } else {
                for (int i = 0; i < dk; ++i) us += p[2 * dk + i] * col[(size_t)i * dv];
                for (int i = 0; i < dk; ++i) {
                    const float s = p[i] * col[(size_t)i * dv] - p[dk + i] * us + p[3 * dk + i] * v;
                    if (live) col[(size_t)i * dv] = s;
                    acc += s * p[4 * dk + i];
                }
            }
            if (live) o[(size_t)t * heads * dv + h * dv + j] = acc;
        }
    }
}

// One wave per (token, head), four a workgroup: out = o / rms(o) * weight * sigmoid(gate).  A lane's first two values and gates are asked for at once.  One MI355X, 2,000
// tokens of 16 heads of 128, us: 12.3 (14.4 with a workgroup a wave, the gates behind the sum).
template <class T>
__global__ void __launch_bounds__(256)
delta_out_kernel(const float *__restrict__ o, const T *__restrict__ proj, int row_stride, int off_g,
                 const float *__restrict__ weight, T *__restrict__ out, int n, int heads, int dv, float eps) {
    const long long item = blockIdx.x * 4ll + (threadIdx.x >> 6);
    if (item >= (long long)n * heads) return;
    const int t = (int)(item / heads), h = (int)(item % heads), lane = threadIdx.x & 63;
    const float *oh = o + (size_t)t * heads * dv + h * dv, *wh = weight + (size_t)h * dv;
    const T *gate = proj + (size_t)t * row_stride + off_g + h * dv;
    const int j0 = min(lane, dv - 1), j1 = min(lane + WAVE, dv - 1);
    const float o0 = oh[j0], o1 = oh[j1], g0 = to_f32(gate[j0]), g1 = to_f32(gate[j1]), w0 = wh[j0], w1 = wh[j1];
    float ss = lane < dv ? o0 * o0 : 0.f;
    if (lane + WAVE < dv) ss = fmaf(o1, o1, ss);
    for (int j = lane + 2 * WAVE; j < dv; j += WAVE) ss = fmaf(oh[j], oh[j], ss);
    const float f = rsqrtf(wave_sum(ss) / (float)dv + eps);
    auto put = [&](int j, float ov, float gv, float wv) { out[(size_t)t * heads * dv + h * dv + j] = from_f32<T>(ov * f * wv * sigmoidf_(gv)); };
    if (lane < dv) put(lane, o0, g0, w0);
    if (lane + WAVE < dv) put(lane + WAVE, o1, g1, w1);
    for (int j = lane + 2 * WAVE; j < dv; j += WAVE) put(j, oh[j], to_f32(gate[j]), wh[j]);
}

// The recurrence over the step's tokens: the scan for every head size it is compiled for, and the chunks where a request may feed
// enough tokens (`work`: delta_chunk_floats floats; null: everything is scanned).  vf: null, or the values as 32-bit rows.
template <class T, bool GATED = false>
static int delta_scan_launch(const T *proj, int row_stride, int off_v, const float *vf, const float *prep, float *work, float *state,
                             size_t slot_stride, float *o, const int *q_start, const int *ctx_len, const int *state_slot,
                             int n, int n_req, int heads, int dk, int dv, hipStream_t stream) {
    const int *done = nullptr;
    const DeltaLine chunks = delta_line(heads, dk, dv, GATED);
    if (work && delta_chunks_possible(n, n_req, dk, chunks.line)) {
        DeltaChunkArgs c = {};
        c.prep = prep; c.proj = proj; c.row_stride = row_stride; c.off_v = off_v; c.vf = vf;
        c.state = state; c.slot_stride = slot_stride; c.o = o;
        c.q_start = q_start; c.ctx_len = ctx_len; c.state_slot = state_slot;
        c.n_req = n_req; c.heads = heads; c.dk = dk; c.dv = dv; c.line = chunks;
        const int rc = delta_chunks_launch<T, GATED>(c, work, n, stream);
        if (rc != LCU_OK) return rc;
        if (n_req == 1 && chunks.chunks_pay(n, n, (n + DELTA_CHUNK - 1) / DELTA_CHUNK)) return LCU_OK;
        done = delta_done(work, n, n_req, heads, dk, dv, GATED);
    }
#define SCAN(DK) delta_scan_kernel<T, DK, GATED><<<dim3(n_req, heads, (dv + (DK ? 64 / scan_groups<T, DK>() : 64) - 1) / (DK ? 64 / scan_groups<T, DK>() : 64)), dim3(64), 0, stream>>>(proj, row_stride, off_v, vf, prep, state, slot_stride, o, q_start, ctx_len, state_slot, heads, dk, dv, done)
    switch (dk) {
    case 16: SCAN(16); break;
    case 32: SCAN(32); break;
    case 48: SCAN(48); break;
    case 64: SCAN(64); break;
    case 80: SCAN(80); break;
    case 96: SCAN(96); break;
    case 112: SCAN(112); break;
    case 128: SCAN(128); break;
    case 192: SCAN(192); break;
    case 256: SCAN(256); break;
    default: SCAN(0); break;
    }
#undef SCAN
    LCU_LAUNCH_CHECK();
    return LCU_OK;
}

template <class T>
static int delta_rule_t(const T *proj, int row_stride, int off_r, int off_k, int off_v, int off_g, int off_a, int off_l,
                        const float *w2, const float *w0, const float *a_bias, const float *weight, float *prep, float *work,
                        float *o, float *state, T *out, const int *q_start, const int *ctx_len, const int *state_slot,
                        int n, int n_req, int heads, int dk, int dv, int rank, float eps, hipStream_t stream) {
    // eight tokens a workgroup where that still gives every compute unit some
#define PREP(TB) delta_prep_kernel<T, TB><<<dim3((n + TB - 1) / TB, heads, (dk + WAVE - 1) / WAVE), dim3(256), rank * TB * sizeof(float), stream>>>(proj, row_stride, off_r, off_k, off_a, off_l, w2, w0, a_bias, prep, n, heads, dk, rank)
    if ((long long)n * heads >= 8 * 512) PREP(8);
    else PREP(1);
#undef PREP
    LCU_LAUNCH_CHECK();
    const int rc = delta_scan_launch<T>(proj, row_stride, off_v, nullptr, prep, work, state, (size_t)heads * dk * dv, o, q_start, ctx_len,
                                        state_slot, n, n_req, heads, dk, dv, stream);
    if (rc != LCU_OK) return rc;
    delta_out_kernel<T><<<dim3((unsigned)(((long long)n * heads + 3) / 4)), dim3(256), 0, stream>>>(o, proj, row_stride, off_g, weight, out, n, heads, dv, eps);
    LCU_LAUNCH_CHECK();
    return LCU_OK;
}

// proj: [n, row_stride] of `type`; the offsets are columns.  w2: [rank, heads * dk] (transposed), w0, a_bias: [heads * dk],
// weight: [heads * dv], all 32-bit.  prep: scratch [n, heads, 5, dk], o: scratch [n, heads * dv], work: scratch of
// lcu_delta_work_floats floats (null: every request is scanned token by token), all 32-bit.
// state: [slots, heads, dk, dv] 32-bit.  out: [n, heads * dv] of `type`.
// Whether requests of a step that feeds q_lens (host memory) tokens go through chunks, if it has the memory for them.
LCU_API int lcu_delta_chunked(const int *q_lens, int n_req, int heads, int dk, int dv, int gated) {
    if (heads <= 0 || dk <= 0 || dk > 128 || dv <= 0) return 0;
    const DeltaLine line = delta_line(heads, dk, dv, gated);
    int longest = 0, tokens = 0, chunks = 0;
    for (int r = 0; r < n_req; ++r) {
        if (q_lens[r] < line.line) continue;
        longest = longest > q_lens[r] ? longest : q_lens[r];
        tokens += q_lens[r];
        chunks += (q_lens[r] + DELTA_CHUNK - 1) / DELTA_CHUNK;
    }
    return line.chunks_pay(longest, tokens, chunks);
}

LCU_API long long lcu_delta_work_floats(int n, int n_req, int heads, int dk, int dv, int gated) {
    return n > 0 && n_req > 0 && heads > 0 && dk > 0 && dv > 0 ? (long long)delta_chunk_floats(n, n_req, heads, dk, dv, gated) : 0;
}

LCU_API int lcu_delta_rule(const void *proj, int type, int row_stride, int off_r, int off_k, int off_v, int off_g,
                           int off_a, int off_l, const float *w2, const float *w0, const float *a_bias,
                           const float *weight, float *prep, float *work, float *o, float *state, void *out, const int *q_start,
                           const int *ctx_len, const int *state_slot, int n, int n_req, int heads, int dk, int dv,
                           int rank, float eps, hipStream_t stream) {
    if (n <= 0 || n_req <= 0) return LCU_OK;
    if (heads <= 0 || heads > 65535 || dk <= 0 || dv <= 0 || rank <= 0 || rank > MAX_RANK || dv > 8 * 65535) return LCU_BAD_ARGUMENT;
    if (type == LCU_F32)
        return delta_rule_t<float>((const float *)proj, row_stride, off_r, off_k, off_v, off_g, off_a, off_l, w2, w0, a_bias, weight, prep, work, o, state, (float *)out, q_start, ctx_len, state_slot, n, n_req, heads, dk, dv, rank, eps, stream);
    if (type == LCU_BF16)
        return delta_rule_t<bf16_t>((const bf16_t *)proj, row_stride, off_r, off_k, off_v, off_g, off_a, off_l, w2, w0, a_bias, weight, prep, work, o, state, (bf16_t *)out, q_start, ctx_len, state_slot, n, n_req, heads, dk, dv, rank, eps, stream);
    return LCU_BAD_ARGUMENT;
}

// ---------------------------------------------------------------- one token a request
// A step in which every request feeds one token (decoding).  What the kernels above take a launch each for, 2 to 5 us of which most is the way of their
// inputs from another kernel's stores, is one workgroup's work here: a workgroup per (request, head), whose four waves take 32 columns of S at
// a time.  A lane holds four neighbouring columns (16-byte loads) of SL = DK / 8 key channels, the groups of lanes as in the scan; every sum is made in
// the scan's order, so a token has the same bits either way.  The matrices are on their way while the token's vectors are made.
// Few requests wait for memory's latency, many for the matrices, read and written once.  16 heads of 128 x 128, rank 64, a chain of such steps: 1 request 9.1 ->
// 6.3 us, 16 requests 23.9 -> 9.0, 200 requests 246 -> 68; the gated rule with its convolution and products 18.7 -> 15.5, 27.4 -> 19.9, 224 -> 91.  (Where it is
// longer: lcu_delta_single_pays.)
// STREAM: the state's loads and stores are non-temporal.
template <int DK, bool STREAM = false> struct SingleColumns {
    static constexpr int SL = DK / 8, SLP = SL + 4, VEC = 8 * SLP;      // a vector in LDS: the groups' shares, four floats of padding behind each
    f32x4_t S[SL];
    __device__ __forceinline__ void load(const float *m, int g, int col, int dv, bool fresh) {
#pragma unroll
        for (int i = 0; i < SL; ++i) {
            const f32x4_t *from = (const f32x4_t *)(m + (size_t)(g * SL + i) * dv + col);
            S[i] = fresh ? f32x4_t{0.f, 0.f, 0.f, 0.f} : STREAM ? __builtin_nontemporal_load(from) : *from;
        }
    }
    __device__ __forceinline__ void store(float *m, int g, int col, int dv) const {
#pragma unroll
        for (int i = 0; i < SL; ++i) {
            f32x4_t *to = (f32x4_t *)(m + (size_t)(g * SL + i) * dv + col);
            if (STREAM) __builtin_nontemporal_store(S[i], to);
            else *to = S[i];
        }
    }
    // u^T S of the four columns: U, the unit key's share of the lane's group
    __device__ __forceinline__ f32x4_t times(const float *U) const {
        f32x4_t p[4] = {};
#pragma unroll
        for (int i = 0; i < SL; ++i) {
#pragma unroll
            for (int e = 0; e < 4; ++e) p[i & 3][e] += U[i] * S[i][e];
        }
        f32x4_t out;
#pragma unroll
        for (int e = 0; e < 4; ++e) out[e] = sum_over_groups<8>((p[0][e] + p[1][e]) + (p[2][e] + p[3][e]));
        return out;
    }
};
// where element i of a vector stands in LDS
template <int DK> __device__ __forceinline__ int single_at(int i) { return i / SingleColumns<DK>::SL * SingleColumns<DK>::SLP + i % SingleColumns<DK>::SL; }

constexpr int SINGLE_MAX_DV = 512;

// The general rule from its projections to what the output matrix reads.  The arithmetic is that of delta_prep_kernel, delta_scan_kernel and delta_out_kernel.
template <class T, int DK, bool STREAM>
__global__ void __launch_bounds__(256)
delta_single_kernel(const T *__restrict__ proj, int row_stride, int off_r, int off_k, int off_v, int off_g, int off_a, int off_l,
                    const float *__restrict__ w2t, const float *__restrict__ w0, const float *__restrict__ a_bias, const float *__restrict__ weight,
                    float *__restrict__ state, T *__restrict__ out, const int *__restrict__ ctx_len, const int *__restrict__ state_slot,
                    int heads, int dv, int rank, float eps) {
    typedef SingleColumns<DK, STREAM> C;
    constexpr int SL = C::SL, HALVES = (DK + WAVE - 1) / WAVE, AHEAD = 16;
    __shared__ __attribute__((aligned(16))) float th[MAX_RANK], vec[5][C::VEC], part[4][HALVES][WAVE], os[SINGLE_MAX_DV];
    const int r = blockIdx.x, h = blockIdx.y, lane = threadIdx.x & 63, wave = threadIdx.x >> 6, g = lane / 8;
    const bool fresh = ctx_len[r] == 1;
    const T *row = proj + (size_t)r * row_stride;
    float *m = state + ((size_t)state_slot[r] * heads + h) * DK * dv;
    C c;
    int col = 32 * wave + lane % 8 * 4;
    // every load whose place is known goes out first: with each where it is used six trips to memory stood behind one another (14.8 us, the three
    // kernels 16.2)
    const int quarter = (rank + 3) / 4, j0 = wave * quarter, j1 = min(rank, j0 + quarter);
    auto second = [&](int j, int b) { return w2t[(size_t)min(j, rank - 1) * heads * DK + h * DK + min(b * WAVE + lane, DK - 1)]; };
    float lo = 0.f, k2[HALVES], w2[AHEAD][HALVES], v[4], mine[5], out_w = 0.f, out_g = 0.f;
    if ((int)threadIdx.x < rank) lo = to_f32(row[off_l + threadIdx.x]);
#pragma unroll
    for (int b = 0; b < HALVES; ++b) k2[b] = b * WAVE + lane < DK ? to_f32(row[off_k + h * DK + b * WAVE + lane]) : 0.f;
    {
        const int ch = h * DK + min((int)threadIdx.x, DK - 1);
        mine[0] = w0[ch];
        mine[1] = to_f32(row[off_a + ch]);
        mine[2] = a_bias[ch];
        mine[3] = to_f32(row[off_k + ch]);
        mine[4] = to_f32(row[off_r + ch]);
    }
#pragma unroll
    for (int j = 0; j < AHEAD; ++j)
#pragma unroll
        for (int b = 0; b < HALVES; ++b) w2[j][b] = second(j0 + j, b);
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = to_f32(row[off_v + h * dv + min(col, dv - 4) + e]);
    if ((int)threadIdx.x < dv) {
        out_w = weight[h * dv + threadIdx.x];
        out_g = to_f32(row[off_g + h * dv + threadIdx.x]);
    }
    c.load(m, g, min(col, dv - 4), dv, fresh);
    __builtin_amdgcn_sched_barrier(0);
    // the token's vectors
    if ((int)threadIdx.x < rank) th[threadIdx.x] = tanhf(lo);
    for (int x = threadIdx.x + 256; x < rank; x += 256) th[x] = tanhf(to_f32(row[off_l + x]));
    float ss = 0.f;
#pragma unroll
    for (int b = 0; b < HALVES; ++b) ss = __builtin_fmaf(k2[b], k2[b], ss);      // (as the other kernel's loop does it; of two products the compiler may round either)
    const float inv = 1.0f / sqrtf(wave_sum_in_place(ss) + 1e-6f);
    lds_barrier();
    float z[HALVES] = {};
#pragma unroll
    for (int j = 0; j < AHEAD; ++j) {
        if (j0 + j >= j1) break;
#pragma unroll
        for (int b = 0; b < HALVES; ++b) z[b] = __builtin_fmaf(w2[j][b], th[j0 + j], z[b]);
    }
#pragma unroll 8
    for (int j = j0 + AHEAD; j < j1; ++j) {
#pragma unroll
        for (int b = 0; b < HALVES; ++b) z[b] = __builtin_fmaf(second(j, b), th[j], z[b]);
    }
#pragma unroll
    for (int b = 0; b < HALVES; ++b) part[wave][b][lane] = z[b];
    lds_barrier();
    if (threadIdx.x < DK) {
        const int i = threadIdx.x, b = i / WAVE, l = i % WAVE, at = single_at<DK>(i);
        const float sum = (part[0][b][l] + part[1][b][l]) + (part[2][b][l] + part[3][b][l]);
        const float u = mine[3] * inv;
        vec[0][at] = expf(-DECAY_SCALE * sigmoidf_(mine[0] + sum));
        vec[1][at] = sigmoidf_(mine[1] + mine[2]) * u;
        vec[2][at] = u;
        vec[3][at] = mine[3];
        vec[4][at] = mine[4];
    }
    lds_barrier();
    const float *W = vec[0] + g * C::SLP, *AU = W + C::VEC, *U = W + 2 * C::VEC, *K = W + 3 * C::VEC, *R = W + 4 * C::VEC;
    for (;;) {
        const bool live = col < dv;
        const f32x4_t us = c.times(U);
#pragma unroll
        for (int i = 0; i < SL; ++i) {
#pragma unroll
            for (int e = 0; e < 4; ++e) c.S[i][e] = W[i] * c.S[i][e] - AU[i] * us[e] + K[i] * v[e];
        }
        const f32x4_t o = c.times(R);
        if (live) {
            c.store(m, g, col, dv);
            if (g == 0) *(f32x4_t *)(os + col) = o;
        }
        col += 128;
        if (col - lane % 8 * 4 >= dv) break;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = to_f32(row[off_v + h * dv + min(col, dv - 4) + e]);
        c.load(m, g, min(col, dv - 4), dv, fresh);
    }
    lds_barrier();
    ss = 0.f;
    for (int j = lane; j < dv; j += 64) ss += os[j] * os[j];
    const float f = rsqrtf(wave_sum(ss) / (float)dv + eps);
    for (int j = threadIdx.x; j < dv; j += 256) {
        const int ch = h * dv + j;
        const bool first = j == (int)threadIdx.x;
        const float gate = sigmoidf_(first ? out_g : to_f32(row[off_g + ch]));
        out[(size_t)r * heads * dv + ch] = from_f32<T>(os[j] * f * (first ? out_w : weight[ch]) * gate);
    }
}

// Sizes for which the kernels for one token a request are there: whole groups of key channels, four columns an access.
static bool single_sizes(int heads, int dk, int dv) {
    return heads > 0 && heads <= 65535 && (dk == 32 || dk == 64 || dk == 96 || dk == 128) && dv > 0 && dv % 4 == 0 && dv <= SINGLE_MAX_DV;
}
// A step's states of this size are in no cache when their layer's turn comes again, and what they leave there would push out what is.  16 heads of 128 x 128 over eight
// layers, us a layer: 48 MB 26.8, past the caches 21.8, 64 MB 34.4 and 26.9 (the gated rule with its convolution 41.4 and 35.1; with 40 MB of something else read between the layers 55.9
// and 49.0); 8 heads of 64 x 256, 48 MB 24.6 and 23.0.  Below it goes either way: 32 MB 15.1 and 12.8, but 15.6 and 17.2; four layers alone, all of whose states the
// last-level cache holds, lose at 48 MB too (18.7 and 23.6).
static bool past_caches(int n_req, int heads, int dk, int dv) { return (long long)n_req * heads * dk * dv * 4 >= (48ll << 20); }
LCU_API int lcu_delta_single_takes(int heads, int dk, int dv) { return single_sizes(heads, dk, dv); }

// Whether the one kernel takes less time than the three.  Where heads have few columns its workgroups, eight on a compute unit at a time, have little to do behind what each makes
// anew, the decay's product over the rank above all, and from some thousands of them on the kernels that share that win.  64 heads of 64 x 4, rank 8: 256 requests
// 78 us, with three kernels 46, 64 requests 23 and 19, 16 requests 8.3 and 9.5; 32 heads of 32 x 16, rank 64: 96 requests 16 and 18, 256 requests 35 and 33; 32 of 32 x 32,
// rank 512, 256 requests: 79 and 70, rank 64 36 and 54.  And where a few workgroups walk the most columns behind the longest ranks: 4 heads of
// 128 x 512, rank 512, one request 19.7 and 16.2, rank 64 12.0 and 13.3, 32 workgroups 21.3 and 26.6.
LCU_API int lcu_delta_single_pays(int n_req, int heads, int dk, int dv, int rank) {
    const long long items = (long long)n_req * heads;
    const bool long_rank = rank > 256;
    if (dv <= 16) return long_rank ? items * dk < 65536 : dv >= 12 ? items <= 4096 : items * dk <= 65536;
    if (dv < 32 || (dv == 32 && dk < 64)) return !long_rank || items <= 3072;
    return !(long_rank && dk * dv > 128 * 384 && items <= 8);
}

// lcu_delta_rule for a step in which every request feeds one token (row r is request r's), where lcu_delta_single_takes says so; state 16-byte aligned.
LCU_API int lcu_delta_single(const void *proj, int type, int row_stride, int off_r, int off_k, int off_v, int off_g, int off_a, int off_l,
                             const float *w2, const float *w0, const float *a_bias, const float *weight, float *state, void *out, const int *ctx_len,
                             const int *state_slot, int n_req, int heads, int dk, int dv, int rank, float eps, hipStream_t stream) {
    if (n_req <= 0) return LCU_OK;
    if (rank <= 0 || rank > MAX_RANK || (type != LCU_F32 && type != LCU_BF16) || (uintptr_t)state % 16) return LCU_BAD_ARGUMENT;
    if (!single_sizes(heads, dk, dv)) return LCU_UNSUPPORTED;
    const bool past = past_caches(n_req, heads, dk, dv);
#define GO(T, DK) (past ? delta_single_kernel<T, DK, true> : delta_single_kernel<T, DK, false>)<<<dim3(n_req, heads), dim3(256), 0, stream>>>((const T *)proj, row_stride, off_r, off_k, off_v, off_g, off_a, off_l, w2, w0, a_bias, weight, state, (T *)out, ctx_len, state_slot, heads, dv, rank, eps)
#define SIZES(T) do { if (dk == 32) GO(T, 32); else if (dk == 64) GO(T, 64); else if (dk == 96) GO(T, 96); else GO(T, 128); } while (0)
    if (type == LCU_F32) SIZES(float);
    else SIZES(bf16_t);
#undef SIZES
#undef GO
    LCU_LAUNCH_CHECK();
    return LCU_OK;
}

// ---------------------------------------------------------------- the gated delta rule
// One decay and one rate per head and token:  S <- g S;  u = beta (v - S^T k);  S <- S + k u^T;  o = S^T q,  with q and k
// unit vectors per head (q also times dk^-1/2).  Written out, S <- g S - (beta g k)(k^T S) + k (beta v)^T with S as the
// token found it, or S <- g S + k (beta v - (beta g)(k^T S)): the scan above in its gated form, which takes per token
// the unit key, the query, the two numbers g and beta g, and the values beta v.  Several value heads may share one
// query/key head (`group` of them).
//   prep (parallel over tokens and value heads): the scan's two vectors and two numbers, and the values times beta;
//   out  (parallel): o of each head divided by its root mean square, times a weight, times silu(gate).
// qkv: [n, qk_heads * dk (q) | qk_heads * dk (k) | heads * dv (v)] 32-bit, the projections behind their convolutions
// and activations.  rows: [n, row_stride] 32-bit holding per head the decay's and the rate's projections at columns
// off_a and off_b, and the gate's heads * dv columns at off_g.
__device__ __forceinline__ float softplus_(float z) { return z > 20.f ? z : log1pf(expf(z)); }

// One wave per (token, value head), four a workgroup.
__global__ void __launch_bounds__(256)
gated_delta_prep_kernel(const float *__restrict__ qkv, const float *__restrict__ rows, int row_stride, int off_a,
                        int off_b, const float *__restrict__ a_log, const float *__restrict__ dt_bias,
                        float *__restrict__ prep, float *__restrict__ vb, int n, int heads, int group, int dk, int dv) {
    const int item = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (item >= n * heads) return;
    const int t = item / heads, h = item % heads, qh = h / group, qk_heads = heads / group;
    const int width = 2 * qk_heads * dk + heads * dv;
    const float *q = qkv + (size_t)t * width + qh * dk, *k = q + qk_heads * dk;
    const float *v = qkv + (size_t)t * width + 2 * qk_heads * dk + h * dv;
    const float *row = rows + (size_t)t * row_stride;
    // (a lane's first two of each are asked for at once, before anything is made of them: 2,000 tokens of 16 heads of 128 22.5 us, 26.3 otherwise)
    const int i0 = min(lane, dk - 1), i1 = min(lane + WAVE, dk - 1), v0 = min(lane, dv - 1), v1 = min(lane + WAVE, dv - 1);
    const float qa = q[i0], qb = q[i1], ka = k[i0], kb = k[i1], va = v[v0], vc = v[v1];
    const float beta = sigmoidf_(row[off_b + h]);
    const float lg = -expf(a_log[h]) * softplus_(row[off_a + h] + dt_bias[h]), g = expf(lg);
    float sq = lane < dk ? qa * qa : 0.f, sk = lane < dk ? ka * ka : 0.f;
    if (lane + WAVE < dk) {
        sq = fmaf(qb, qb, sq);
        sk = fmaf(kb, kb, sk);
    }
#pragma unroll 4
    for (int i = lane + 2 * WAVE; i < dk; i += WAVE) {
        sq = fmaf(q[i], q[i], sq);
        sk = fmaf(k[i], k[i], sk);
    }
    sq = wave_sum_in_place(sq);
    sk = wave_sum_in_place(sk);
    const float qf = 1.0f / sqrtf(sq + 1e-6f) / sqrtf((float)dk), kf = 1.0f / sqrtf(sk + 1e-6f);
    float *out = prep + (size_t)item * (2 * dk + 4);
    auto put = [&](int i, float qv, float kv) {
        out[i] = kv * kf;
        out[dk + i] = qv * qf;
    };
    if (lane < dk) put(lane, qa, ka);
    if (lane + WAVE < dk) put(lane + WAVE, qb, kb);
#pragma unroll 4
    for (int i = lane + 2 * WAVE; i < dk; i += WAVE) put(i, q[i], k[i]);
    if (lane < 4) out[2 * dk + lane] = lane == 0 ? g : lane == 1 ? beta * g : lane == 2 ? lg : 0.f;
    float *vo = vb + (size_t)item * dv;
    if (lane < dv) vo[lane] = beta * va;
    if (lane + WAVE < dv) vo[lane + WAVE] = beta * vc;
#pragma unroll 4
    for (int j = lane + 2 * WAVE; j < dv; j += WAVE) vo[j] = beta * v[j];
}

// One wave per (token, head), four a workgroup: out = o / rms(o) * weight * silu(gate); weight: [dv], shared by the heads.  One MI355X, 2,000 tokens of 16 heads of 128, us:
// 13.3 (15.8 with a workgroup a wave, the gates behind the sum).
template <class T>
__global__ void __launch_bounds__(256)
gated_delta_out_kernel(const float *__restrict__ o, const float *__restrict__ rows, int row_stride, int off_g,
                       const float *__restrict__ weight, T *__restrict__ out, int n, int heads, int dv, float eps) {
    const int item = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (item >= n * heads) return;
    const int t = item / heads, h = item % heads;
    const float *oh = o + (size_t)t * heads * dv + h * dv, *gate = rows + (size_t)t * row_stride + off_g + h * dv;
    const int j0 = min(lane, dv - 1), j1 = min(lane + WAVE, dv - 1);
    const float o0 = oh[j0], o1 = oh[j1], z0 = gate[j0], z1 = gate[j1], w0 = weight[j0], w1 = weight[j1];
    float ss = lane < dv ? o0 * o0 : 0.f;
    if (lane + WAVE < dv) ss = fmaf(o1, o1, ss);
    for (int j = lane + 2 * WAVE; j < dv; j += WAVE) ss = fmaf(oh[j], oh[j], ss);
    const float f = 1.0f / sqrtf(wave_sum(ss) / (float)dv + eps);
    auto put = [&](int j, float ov, float z, float wv) { out[(size_t)t * heads * dv + h * dv + j] = from_f32<T>(ov * f * wv * (z / (1.0f + expf(-z)))); };
    if (lane < dv) put(lane, o0, z0, w0);
    if (lane + WAVE < dv) put(lane + WAVE, o1, z1, w1);
    for (int j = lane + 2 * WAVE; j < dv; j += WAVE) put(j, oh[j], gate[j], weight[j]);
}

// a_log, dt_bias: [heads]; weight: [dv], 32-bit.  prep: scratch [n, heads, 2 * dk + 4]; vb, o: scratch [n, heads * dv], work: as above, 32-bit.
// state: slot s at state + s * slot_stride, [heads, dk, dv] 32-bit.  out: [n, heads * dv] of out_type.
LCU_API int lcu_gated_delta_rule(const float *qkv, const float *rows, int row_stride, int off_a, int off_b, int off_g,
                                 const float *a_log, const float *dt_bias, const float *weight, float *prep, float *vb, float *work, float *o,
                                 float *state, long long slot_stride, void *out, int out_type, const int *q_start,
                                 const int *ctx_len, const int *state_slot, int n, int n_req, int heads, int qk_heads, int dk,
                                 int dv, float eps, hipStream_t stream) {
    if (n <= 0 || n_req <= 0) return LCU_OK;
    if (heads <= 0 || heads > 65535 || qk_heads <= 0 || heads % qk_heads || dk <= 0 || dv <= 0 || dv > 8 * 65535 ||
        (out_type != LCU_F32 && out_type != LCU_BF16))
        return LCU_BAD_ARGUMENT;
    if ((long long)n * heads > INT_MAX - 4) return LCU_BAD_ARGUMENT;
    gated_delta_prep_kernel<<<dim3((n * heads + 3) / 4), dim3(256), 0, stream>>>(qkv, rows, row_stride, off_a, off_b, a_log, dt_bias, prep, vb,
                                                                                n, heads, heads / qk_heads, dk, dv);
    LCU_LAUNCH_CHECK();
    const int rc = delta_scan_launch<float, true>(nullptr, 0, 0, vb, prep, work, state, (size_t)slot_stride, o, q_start, ctx_len, state_slot, n, n_req,
                                            heads, dk, dv, stream);
    if (rc != LCU_OK) return rc;
    if (out_type == LCU_F32)
        gated_delta_out_kernel<float><<<dim3((n * heads + 3) / 4), dim3(256), 0, stream>>>(o, rows, row_stride, off_g, weight, (float *)out, n, heads, dv, eps);
    else
        gated_delta_out_kernel<bf16_t><<<dim3((n * heads + 3) / 4), dim3(256), 0, stream>>>(o, rows, row_stride, off_g, weight, (bf16_t *)out, n, heads, dv, eps);
    LCU_LAUNCH_CHECK();
    return LCU_OK;
}

// One token a request, in two kernels: the convolution and the vectors, then the recurrence and the output.  (One kernel for both would have a workgroup
// per query/key head, whose channels several value heads read and one must move on: four of them for a request with four such heads.)
// The convolution of causal_conv.hip (taps oldest first, silu behind it) and gated_delta_prep_kernel: a workgroup per (request, query/key head).
constexpr int SINGLE_MAX_TAPS = 8, SINGLE_MAX_GROUP = 64;
__global__ void __launch_bounds__(1024)
gated_delta_single_prep_kernel(const float *__restrict__ rows, int row_stride, int off_a, int off_b, const float *__restrict__ conv_w, int taps,
                               float *__restrict__ inputs, size_t slot_stride, const float *__restrict__ a_log, const float *__restrict__ dt_bias,
                               float *__restrict__ prep, float *__restrict__ vb, const int *__restrict__ ctx_len, const int *__restrict__ state_slot,
                               int heads, int qk_heads, int dk, int dv) {
    __shared__ float q[128], k[128], numbers[SINGLE_MAX_GROUP][4];
    const int r = blockIdx.x, qh = blockIdx.y, threads = blockDim.x, lane = threadIdx.x & 63, group = heads / qk_heads;
    const int channels = 2 * qk_heads * dk + heads * dv;
    const bool fresh = ctx_len[r] == 1;
    const float *row = rows + (size_t)r * row_stride;
    float *st = inputs + (size_t)state_slot[r] * slot_stride;
    float beta = 0.f, a = 0.f, al = 0.f, db = 0.f;
    if ((int)threadIdx.x < group) {
        const int h = qh * group + threadIdx.x;
        beta = row[off_b + h];
        a = row[off_a + h];
        al = a_log[h];
        db = dt_bias[h];
    }
    for (int x = threadIdx.x; x < 2 * dk + group * dv; x += threads) {
        const int c = x < dk ? qh * dk + x : x < 2 * dk ? (qk_heads + qh) * dk + x - dk : 2 * qk_heads * dk + qh * group * dv + x - 2 * dk;
        const float cur = row[c], last = conv_w[(size_t)c * taps + taps - 1], rate = x < 2 * dk ? 0.f : row[off_b + qh * group + (x - 2 * dk) / dv];
        float v[SINGLE_MAX_TAPS - 1], w[SINGLE_MAX_TAPS - 1];
#pragma unroll
        for (int i = 0; i < SINGLE_MAX_TAPS - 1; ++i) {      // (all loads before the first store)
            const bool in = i < taps - 1;
            v[i] = in && !fresh ? st[(size_t)i * channels + c] : 0.f;
            w[i] = in ? conv_w[(size_t)c * taps + i] : 0.f;
        }
        float acc = 0.f;
#pragma unroll
        for (int i = 0; i < SINGLE_MAX_TAPS - 1; ++i)
            if (i < taps - 1) acc = __builtin_fmaf(w[i], v[i], acc);
        acc = __builtin_fmaf(last, cur, acc);
#pragma unroll
        for (int i = 0; i < SINGLE_MAX_TAPS - 1; ++i)
            if (i > 0 && i < taps - 1) st[(size_t)(i - 1) * channels + c] = v[i];
        if (taps > 1) st[(size_t)(taps - 2) * channels + c] = cur;
        const float y = acc / (1.0f + expf(-acc));
        if (x < dk) q[x] = y;
        else if (x < 2 * dk) k[x - dk] = y;
        else {
            const int h = qh * group + (x - 2 * dk) / dv, j = (x - 2 * dk) % dv;
            vb[((size_t)r * heads + h) * dv + j] = sigmoidf_(rate) * y;
        }
    }
    if ((int)threadIdx.x < group) {
        const float lg = -expf(al) * softplus_(a + db), gd = expf(lg);
        float *to = numbers[threadIdx.x];
        to[0] = gd;
        to[1] = sigmoidf_(beta) * gd;
        to[2] = lg;
        to[3] = 0.f;
    }
    lds_barrier();
    float sq = 0.f, sk = 0.f;
    for (int i = lane; i < dk; i += 64) {
        sq = __builtin_fmaf(q[i], q[i], sq);
        sk = __builtin_fmaf(k[i], k[i], sk);
    }
    sq = wave_sum_in_place(sq);
    sk = wave_sum_in_place(sk);
    const float qf = 1.0f / sqrtf(sq + 1e-6f) / sqrtf((float)dk), kf = 1.0f / sqrtf(sk + 1e-6f);
    const int per = 2 * dk + 4;
    for (int x = threadIdx.x; x < group * per; x += threads) {
        const int i = x % per;
        prep[((size_t)r * heads + qh * group) * per + x] = i < dk ? k[i] * kf : i < 2 * dk ? q[i - dk] * qf : numbers[x / per][i - 2 * dk];
    }
}

// The recurrence and gated_delta_out_kernel: a workgroup per (request, value head).
template <class T, int DK, bool STREAM>
__global__ void __launch_bounds__(256)
gated_delta_single_kernel(const float *__restrict__ prep, const float *__restrict__ vb, const float *__restrict__ rows, int row_stride, int off_g,
                          const float *__restrict__ weight, float *__restrict__ state, size_t slot_stride, T *__restrict__ out,
                          const int *__restrict__ ctx_len, const int *__restrict__ state_slot, int heads, int dv, float eps) {
    typedef SingleColumns<DK, STREAM> C;
    constexpr int SL = C::SL;
    __shared__ __attribute__((aligned(16))) float os[SINGLE_MAX_DV];
    const int r = blockIdx.x, h = blockIdx.y, lane = threadIdx.x & 63, wave = threadIdx.x >> 6, g = lane / 8;
    const bool fresh = ctx_len[r] == 1;
    const size_t item = (size_t)r * heads + h;
    float *m = state + (size_t)state_slot[r] * slot_stride + (size_t)h * DK * dv;
    const float *p = prep + item * (2 * DK + 4);
    C c;
    int col = 32 * wave + lane % 8 * 4;
    c.load(m, g, min(col, dv - 4), dv, fresh);
    float U[SL], R[SL];
#pragma unroll
    for (int i = 0; i < SL; i += 4) {
        *(f32x4_t *)(U + i) = *(const f32x4_t *)(p + g * SL + i);
        *(f32x4_t *)(R + i) = *(const f32x4_t *)(p + DK + g * SL + i);
    }
    const float gd = p[2 * DK], bg = p[2 * DK + 1];
    f32x4_t v = *(const f32x4_t *)(vb + item * dv + min(col, dv - 4));
    float out_w = 0.f, out_g = 0.f;
    if ((int)threadIdx.x < dv) {
        out_w = weight[threadIdx.x];
        out_g = rows[(size_t)r * row_stride + off_g + h * dv + threadIdx.x];
    }
    __builtin_amdgcn_sched_barrier(0);
    for (;;) {
        const bool live = col < dv;
        const f32x4_t us = c.times(U);
        f32x4_t e4;
#pragma unroll
        for (int e = 0; e < 4; ++e) e4[e] = v[e] - bg * us[e];
#pragma unroll
        for (int i = 0; i < SL; ++i) {
#pragma unroll
            for (int e = 0; e < 4; ++e) c.S[i][e] = __builtin_fmaf(gd, c.S[i][e], U[i] * e4[e]);
        }
        const f32x4_t o = c.times(R);
        if (live) {
            c.store(m, g, col, dv);
            if (g == 0) *(f32x4_t *)(os + col) = o;
        }
        col += 128;
        if (col - lane % 8 * 4 >= dv) break;
        v = *(const f32x4_t *)(vb + item * dv + min(col, dv - 4));
        c.load(m, g, min(col, dv - 4), dv, fresh);
    }
    lds_barrier();
    float ss = 0.f;
    for (int j = lane; j < dv; j += 64) ss += os[j] * os[j];
    const float f = 1.0f / sqrtf(wave_sum(ss) / (float)dv + eps);
    for (int j = threadIdx.x; j < dv; j += 256) {
        const bool first = j == (int)threadIdx.x;
        const float z = first ? out_g : rows[(size_t)r * row_stride + off_g + h * dv + j];
        out[item * dv + j] = from_f32<T>(os[j] * f * (first ? out_w : weight[j]) * (z / (1.0f + expf(-z))));
    }
}

LCU_API int lcu_gated_delta_single_takes(int heads, int qk_heads, int dk, int dv, int taps, long long slot_stride) {
    return single_sizes(heads, dk, dv) && qk_heads > 0 && heads % qk_heads == 0 && heads / qk_heads <= SINGLE_MAX_GROUP && taps >= 1 && taps <= SINGLE_MAX_TAPS && slot_stride % 4 == 0;
}

// Whether they take less time than the convolution's two kernels and the rule's three.  Not, as above, with few columns and many workgroups (16 heads of 128 x 4 with 4 for
// queries and keys, with the products: 128 requests 28 us and 26, 32 of 128 x 16, 96 requests 41 and 41, 16 of 64 x 12, 128 requests 23 and 26), nor where a few workgroups have
// the convolution of many channels each (8 heads of 128 x 512 with one for queries and keys: one request 30 and 24, 8 requests 35 and 34; with two 27 and 24, four requests 29 and 30).
LCU_API int lcu_gated_delta_single_pays(int n_req, int heads, int qk_heads, int dk, int dv) {
    const long long items = (long long)n_req * heads, channels = (long long)(heads / qk_heads) * dv + 2 * dk;
    if (dv <= 16 && !(dv >= 12 ? dk <= 64 || items <= 2048 : items * dk <= 131072)) return 0;
    return channels < 2304 || items * 64 >= channels;
}

// lcu_causal_conv (silu, no bias, over the rows' first 2 * qk_heads * dk + heads * dv columns) and lcu_gated_delta_rule for a step in which every request
// feeds one token, where lcu_gated_delta_single_takes says so.  inputs: the convolution's [taps - 1, channels] of slot 0; both states' slots lie
// slot_stride apart, the matrices 16-byte aligned.  prep, vb: as above.
LCU_API int lcu_gated_delta_single(const float *rows, int row_stride, int off_a, int off_b, int off_g, const float *conv_w, int taps, float *inputs,
                                   const float *a_log, const float *dt_bias, const float *weight, float *prep, float *vb, float *state,
                                   long long slot_stride, void *out, int out_type, const int *ctx_len, const int *state_slot, int n_req, int heads,
                                   int qk_heads, int dk, int dv, float eps, hipStream_t stream) {
    if (n_req <= 0) return LCU_OK;
    if ((out_type != LCU_F32 && out_type != LCU_BF16) || ((uintptr_t)state | (uintptr_t)prep | (uintptr_t)vb) % 16 || (taps > 1 && !inputs)) return LCU_BAD_ARGUMENT;
    if (!lcu_gated_delta_single_takes(heads, qk_heads, dk, dv, taps, slot_stride)) return LCU_UNSUPPORTED;
    const int wide = 2 * dk + heads / qk_heads * dv;          // a thread a channel, if there are so many
    gated_delta_single_prep_kernel<<<dim3(n_req, qk_heads), dim3(wide >= 1024 ? 1024 : (wide + 63) / 64 * 64), 0, stream>>>(rows, row_stride, off_a, off_b, conv_w, taps, inputs, (size_t)slot_stride, a_log,
                                                                                   dt_bias, prep, vb, ctx_len, state_slot, heads, qk_heads, dk, dv);
    LCU_LAUNCH_CHECK();
    const bool past = past_caches(n_req, heads, dk, dv);
#define GO(T, DK) (past ? gated_delta_single_kernel<T, DK, true> : gated_delta_single_kernel<T, DK, false>)<<<dim3(n_req, heads), dim3(256), 0, stream>>>(prep, vb, rows, row_stride, off_g, weight, state, (size_t)slot_stride, (T *)out, ctx_len, state_slot, heads, dv, eps)
#define SIZES(T) do { if (dk == 32) GO(T, 32); else if (dk == 64) GO(T, 64); else if (dk == 96) GO(T, 96); else GO(T, 128); } while (0)
    if (out_type == LCU_F32) SIZES(float);
    else SIZES(bf16_t);
#undef SIZES
#undef GO
    LCU_LAUNCH_CHECK();
    return LCU_OK;
}
