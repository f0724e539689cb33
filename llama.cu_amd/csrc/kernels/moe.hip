// A feed-forward of many small experts of which each token uses a few.
//
//   route:   z = W_router h (+ bias) (32-bit), the `top` experts with the largest z (ties: the lower
//            index), each with the weight sigmoid(z) (a token's weights are not made to add up to one) or,
//            in the other mode, with the softmax over the chosen logits alone; or, in a third, with scores s = softmax(z)
//            over all experts, the choice by s + a correction per expert, and the chosen scores divided by their sum (or as
//            they are) times a factor as weights; the choice may be limited to the experts of the best groups; rows of the router's matrix behind the experts' are gates: sigmoid of their logit goes out per
//            token; the last experts may be identity experts, which have no matrices and return their input;
//   group:   the (token, choice) pairs sorted by expert and cut into tiles of up to 128 rows of one expert, on the
//            device (nothing comes back to the host); where experts have few pairs a product's workgroups look for theirs
//            themselves instead;
//   up:      act = gelu(W_up[e] (weight * h))    the weight scales what goes INTO the expert; or, gated:
//            act = silu(W_gate[e] h) * (W_up[e] h) (or the limited form, gate_act.h), and the weight scales what comes OUT of the expert
//   down:    y = W_down[e] act, added to the token's output row (32-bit), in the gated form times the weight
//            and beside a shared expert's row times its gate.
// The products run on the matrix cores: bfloat16 operands with v_mfma_f32_16x16x32_bf16, or
// true 32-bit with v_mfma_f32_16x16x4_f32; sums are 32-bit.  A row's result depends on that
// row and its expert alone (never on which rows share its tile), so it does not depend on
// the batch.
#include "common.h"
#include "gate_act.h"
#include "lane_moves.h"
#include "pair_sum.h"
#include "rows.h"

constexpr int MOE_MAX_EXPERTS = 1024;
constexpr int MOE_TILE_ROWS = 128;       // rows of a tile of the kernel for many rows at most

typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;

// ---------------------------------------------------------------- route
// One block per token (256 threads; 1024 where a step has few tokens, so that more of a token's experts are
// multiplied side by side).  h: [n, d] of T; router: [experts, d] 32-bit.  ids, wts: [n, top].  A wave takes
// the experts e = wave, wave + waves, ...; with d a multiple of 8 a lane keeps its share of the row (eight
// neighbouring elements of every 512) in registers for all of them.
template <class T> struct alignas(8 * sizeof(T)) Row8 { T v[8]; };
constexpr int ROUTE_CHUNKS = 8;                  // rows of up to 8 * 512 elements stay in registers

// bias: null or [experts], added to the logits.  mode 0: the weight of a chosen expert is sigmoid(z); 1: the softmax over
// the chosen logits; 2: s = softmax(z) over all experts, the choice goes by s + bias (the bias is not added to the
// logits), the weights are the chosen s divided by their sum + 1e-20 (renorm 0: as they are), times `scale`.  groups > 1 (mode 2):
// the experts are so many groups of neighbours, a group counts as its best expert's s + bias, and only experts of the `keep` best
// groups (ties: the lower index) can be chosen.  extra: rows of `router` behind the experts' (at most MOE_MAX_EXTRA); gates [n, extra] takes sigmoid
// of their logits (they are no experts and are never chosen).
constexpr int MOE_MAX_EXTRA = 8;
// The choice and its weights from a token's logits z, by one wave.  zc, sc: LDS, a number an expert each.
__device__ __forceinline__ void route_choose(float *z, float *zc, float *sc, int t, int lane, const float *__restrict__ bias, int *__restrict__ ids,
                                             float *__restrict__ wts, float *__restrict__ gates, int n_experts, int top, int mode, int extra, int groups,
                                             int keep, int renorm, float scale) {
    for (int e = lane; e < extra; e += WAVE) gates[(size_t)t * extra + e] = 1.0f / (1.0f + expf(-z[n_experts + e]));
    const bool one_each = n_experts <= WAVE;         // an expert a lane: the choice stays in registers
    if (mode == 2) {                                 // scores over all experts; z becomes what the choice goes by
        float m = -INFINITY;
        for (int e = lane; e < n_experts; e += WAVE) m = fmaxf(m, z[e]);
        m = wave_max_in_place(m);
        float part = 0.f;
        for (int e = lane; e < n_experts; e += WAVE) part += expf(z[e] - m);
        const float sum = wave_sum_in_place(part);
        for (int e = lane; e < n_experts; e += WAVE) {
            const float s = expf(z[e] - m) / sum;
            sc[e] = s;
            z[e] = s + (bias ? bias[e] : 0.f);
        }
        __threadfence_block();
        if (groups > 1) {
            // every group's best (in zc), then every group's place among them; the experts of a group behind the kept ones are out
            const int per = n_experts / groups;
            for (int g = lane; g < groups; g += WAVE) {
                float best = z[g * per];
                for (int e = 1; e < per; ++e) best = fmaxf(best, z[g * per + e]);
                zc[g] = best;
            }
            __threadfence_block();
            for (int g = lane; g < groups; g += WAVE) {
                int before = 0;
                for (int o = 0; o < groups; ++o) before += zc[o] > zc[g] || (zc[o] == zc[g] && o < g);
                if (before >= keep)
                    for (int e = 0; e < per; ++e) z[g * per + e] = -INFINITY;
            }
            __threadfence_block();
        }
    }
    float mine = lane < n_experts ? z[lane] : -INFINITY;
    for (int k = 0; k < top; ++k) {
        int arg;
        float value;                                 // what the weight is made of
        if (one_each) {
            const float best = wave_max_in_place(mine);
            const unsigned long long who = __ballot(lane < n_experts && mine == best);
            arg = who ? __ffsll((long long)who) - 1 : 0;     // the lowest of equals; every logit NaN: any expert
            // where fewer logits are finite than experts are chosen, what is left may be an expert that was chosen already: it comes with
            // the -inf that stands in its place now, and so with no weight
            value = mode == 2 ? sc[arg] : who ? best : z[arg];
            if (lane == arg) mine = -INFINITY;
        } else {
            float best = -INFINITY;
            arg = 0x7fffffff;
            for (int e = lane; e < n_experts; e += WAVE) {
                const float v = z[e];
                if (v > best || (v == best && e < arg)) { best = v; arg = e; }
            }
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) {
                const float ob = __shfl_xor(best, off, WAVE);
                const int oa = __shfl_xor(arg, off, WAVE);
                if (ob > best || (ob == best && oa < arg)) { best = ob; arg = oa; }
            }
            if (arg >= n_experts) arg = 0;
            value = mode == 2 ? sc[arg] : z[arg];
            __threadfence_block();
            if (lane == 0) z[arg] = -INFINITY;
            __threadfence_block();
        }
        if (lane == 0) {
            ids[(size_t)t * top + k] = arg;
            zc[k] = value;
            if (mode == 0) wts[(size_t)t * top + k] = 1.0f / (1.0f + expf(-value));
        }
    }
    __threadfence_block();
    if (mode == 2) {                                 // the chosen scores, made to add up to one
        float part = 0.f;
        for (int k = lane; k < top; k += WAVE) part += zc[k];
        const float sum = renorm ? wave_sum_in_place(part) + 1e-20f : 1.f;
        for (int k = lane; k < top; k += WAVE) wts[(size_t)t * top + k] = zc[k] / sum * scale;
    }
    if (mode == 1) {                                 // the softmax over the chosen logits (the first is the largest)
        const float z0 = zc[0];
        float part = 0.f;
        for (int k = lane; k < top; k += WAVE) part += expf(zc[k] - z0);
        const float sum = wave_sum_in_place(part);
        for (int k = lane; k < top; k += WAVE) wts[(size_t)t * top + k] = expf(zc[k] - z0) / sum;
    }
}

template <class T, int THREADS>
__global__ void __launch_bounds__(THREADS)
moe_route_kernel(const T *__restrict__ h, const float *__restrict__ router, const float *__restrict__ bias, int *__restrict__ ids,
                 float *__restrict__ wts, float *__restrict__ gates, int d, int n_experts, int top, int mode, int extra, int groups, int keep,
                 int renorm, float scale) {
    __shared__ float z[MOE_MAX_EXPERTS + MOE_MAX_EXTRA];
    __shared__ float zc[MOE_MAX_EXPERTS];
    __shared__ float sc[MOE_MAX_EXPERTS];
    const float *logit_bias = mode == 2 ? nullptr : bias;
    const int experts = n_experts + extra;          // rows of the router's matrix
    const int t = blockIdx.x, wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
    const T *row = h + (size_t)t * d;
    if (d % 8 == 0 && d <= ROUTE_CHUNKS * 512) {
        float x[ROUTE_CHUNKS][8];
#pragma unroll
        for (int k = 0; k < ROUTE_CHUNKS; ++k) {
            const int c = k * 512 + lane * 8;
            if (c < d) {
                const Row8<T> in = *(const Row8<T> *)(row + c);
#pragma unroll
                for (int e = 0; e < 8; ++e) x[k][e] = to_f32(in.v[e]);
            }
        }
        // two rows of the router at a time, so that 17 rows on 16 waves (16 experts and a gate) are not two trips to memory; but one where a wave has
        // many long rows, which are trips enough and twice of which leave no room for the next ones' loads (1,024 rows of 4,096, one token: 183 us, two at a
        // time 222)
        const bool two = experts <= 64 + MOE_MAX_EXTRA || d <= ROUTE_CHUNKS * 256;
        for (int e = wave; e < experts; e += (two ? 2 : 1) * (THREADS / WAVE)) {
            const int e2 = two ? e + THREADS / WAVE : experts;
            const float *w = router + (size_t)e * d, *v = router + (size_t)(e2 < experts ? e2 : e) * d;
            float acc = 0.f, acc2 = 0.f;
            if (e2 < experts) {
#pragma unroll
                for (int k = 0; k < ROUTE_CHUNKS; ++k) {
                    const int c = k * 512 + lane * 8;
                    if (c < d) {
                        const f32x4 w0 = *(const f32x4 *)(w + c), w1 = *(const f32x4 *)(w + c + 4), v0 = *(const f32x4 *)(v + c), v1 = *(const f32x4 *)(v + c + 4);
#pragma unroll
                        for (int i = 0; i < 4; ++i) { acc += x[k][i] * w0[i]; acc2 += x[k][i] * v0[i]; }
#pragma unroll
                        for (int i = 0; i < 4; ++i) { acc += x[k][4 + i] * w1[i]; acc2 += x[k][4 + i] * v1[i]; }
                    }
                }
                acc2 = wave_sum_in_place(acc2);
                if (lane == 0) z[e2] = acc2 + (logit_bias && e2 < n_experts ? logit_bias[e2] : 0.f);
            } else {
#pragma unroll
                for (int k = 0; k < ROUTE_CHUNKS; ++k) {
                    const int c = k * 512 + lane * 8;
                    if (c < d) {
                        const f32x4 w0 = *(const f32x4 *)(w + c), w1 = *(const f32x4 *)(w + c + 4);
#pragma unroll
                        for (int i = 0; i < 4; ++i) acc += x[k][i] * w0[i];
#pragma unroll
                        for (int i = 0; i < 4; ++i) acc += x[k][4 + i] * w1[i];
                    }
                }
            }
            acc = wave_sum_in_place(acc);
            if (lane == 0) z[e] = acc + (logit_bias && e < n_experts ? logit_bias[e] : 0.f);
        }
    } else {
        for (int e = wave; e < experts; e += THREADS / WAVE) {
            const float *w = router + (size_t)e * d;
            float acc = 0.f;
            for (int c = lane; c < d; c += WAVE) acc += to_f32(row[c]) * w[c];
            acc = wave_sum_in_place(acc);
            if (lane == 0) z[e] = acc + (logit_bias && e < n_experts ? logit_bias[e] : 0.f);
        }
    }
    __syncthreads();
    // the first wave does the rest alone
    if (wave != 0) return;
    route_choose(z, zc, sc, t, lane, bias, ids, wts, gates, n_experts, top, mode, extra, groups, keep, renorm, scale);
}

// Rows of CHUNKS * 512 elements: no load hangs on a comparison, so a wave asks for its tokens' rows and its first two rows of the router at once, and
// from then on for the next row while it works on one (the loop above waits for every 512 elements in turn).  TOKENS tokens a workgroup: the router's
// matrix comes out of the second-level cache once for all of them, which bounds long steps, and a wave each makes their choices.  The same sums in the
// same order.  One MI355X, 2,000 tokens, us: 16 experts and a gate, rows of 1024 6.5 (9.9), 2048 8.5 (16.3), 4096 20.4 (29.2); 256 experts 42 (72), 54 (142), 151 (309).  Small steps, which
// share the rows out over the waves of 1,024 threads, gain nothing: 16 tokens and experts 5.1 (4.8).
constexpr int ROUTE_THREADS = 256;
template <class T, int CHUNKS, int TOKENS>
__global__ void __launch_bounds__(ROUTE_THREADS)
moe_route_rows_kernel(const T *__restrict__ h, const float *__restrict__ router, const float *__restrict__ bias, int *__restrict__ ids,
                      float *__restrict__ wts, float *__restrict__ gates, int n, int n_experts, int top, int mode, int extra, int groups, int keep,
                      int renorm, float scale) {
    extern __shared__ float lds[];
    constexpr int WAVES = ROUTE_THREADS / WAVE, D = CHUNKS * 512;
    static_assert(TOKENS <= WAVES, "a wave a token");
    const int experts = n_experts + extra, t0 = blockIdx.x * TOKENS, wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
    float x[TOKENS][CHUNKS][8];
    f32x4 w[2 * CHUNKS], next[2 * CHUNKS];
    auto fetch = [&](int e, f32x4 *to) {
        const float *from = router + (size_t)min(e, experts - 1) * D + lane * 8;
#pragma unroll
        for (int k = 0; k < CHUNKS; ++k) { to[2 * k] = *(const f32x4 *)(from + k * 512); to[2 * k + 1] = *(const f32x4 *)(from + k * 512 + 4); }
    };
    fetch(wave, w);
#pragma unroll
    for (int b = 0; b < TOKENS; ++b)
#pragma unroll
        for (int k = 0; k < CHUNKS; ++k) load_as_f32<T, 8>(h + (size_t)min(t0 + b, n - 1) * D + k * 512 + lane * 8, x[b][k]);
    for (int e = wave; e < experts; e += WAVES) {
        fetch(e + WAVES, next);
#pragma unroll
        for (int b = 0; b < TOKENS; ++b) {
            float acc = 0.f;
#pragma unroll
            for (int k = 0; k < CHUNKS; ++k)
#pragma unroll
                for (int i = 0; i < 8; ++i) acc = fmaf(x[b][k][i], w[2 * k + i / 4][i % 4], acc);
            acc = wave_sum_in_place(acc);
            if (lane == 0) lds[b * 3 * experts + e] = acc;
        }
#pragma unroll
        for (int k = 0; k < 2 * CHUNKS; ++k) w[k] = next[k];
    }
    __syncthreads();
    if (wave >= TOKENS || t0 + wave >= n) return;
    float *z = lds + wave * 3 * experts;
    if (mode != 2 && bias) {                                     // (here, all at once: in the loop every row would wait for its number)
        for (int e = lane; e < n_experts; e += WAVE) z[e] += bias[e];
        __threadfence_block();
    }
    route_choose(z, z + experts, z + 2 * experts, t0 + wave, lane, bias, ids, wts, gates, n_experts, top, mode, extra, groups, keep, renorm, scale);
}

// Tokens a workgroup of it for `chunks` * 512 elements and so many rows of the router, 0: the general kernel.  The line lies where a workgroup more on every compute unit costs as
// much as its tokens share.  Measured from 512 to 4,096 elements, 4 to 256 rows and 64 to 2,000 tokens, bfloat16, 64 rows, us with the general kernel, 1, 2 and 4 tokens: 400 tokens
// of 1024 9.2, 6.8, 7.6, 10.6, of 3072 17.0, 16.7, 11.7, 17.0; 520 of 2048 15.5, 16.3, 11.5, 13.8, of 4096 26.8, 30.5, 24.6, 21.8; 1,000 of 1024 11.6, 11.9, 8.6, 10.8; 2,000 of 2048 41.2, 36.8, 23.8,
// 17.6, of 3072 60.9, 57.4, 31.8, 33.7 (four tokens of more than 2048 and two of 4096 leave a compute unit one workgroup).  Four rows, one a wave, leave nothing to
// ask for early, and in 32 bits the tokens' rows are most of what is read: 520 tokens of 2048 4.1, 4.7, 4.5, 4.5, 2,000 8.1, 8.9, 7.3, 6.8, of 3072 9.6, 12.2, 10.0, 11.2.  A form that masks the last
// 512, for the widths between, took up to a quarter longer: with 16 rows and 1,000 tokens of 1000 elements as long as the general kernel (6.8 us), of 1528 too (7.8).
static int route_tokens(int n, int chunks, int rows, int type) {
    const long long values = (long long)n * chunks * 512;
    if (type == LCU_F32 && rows <= ROUTE_THREADS / WAVE && chunks >= 4 && (chunks > 4 || values < 2000000)) return 0;
    if (chunks <= 4) return values < 750000 ? 1 : values < 3000000 ? 2 : 4;
    return chunks < 8 || n <= 512 ? 2 : 4;
}

// ---------------------------------------------------------------- group
// One block.  ids: [total] experts of the (token, choice) pairs in flat order.  Writes
// sorted_to_flat [total] (the pairs sorted by expert), and the tiles of up to rows_per_tile rows:
// tile_expert, tile_begin (first sorted row), tile_rows, each [max_tiles], and n_tiles [1].  Only the first `tiled`
// experts get tiles: the ones behind them have no matrices (identity experts), and their pairs are only sorted.  An expert's tiles are as few as
// can be and of nearly the same size, a multiple of 16 rows but for the last.
// A thread an expert: the pairs and tiles before its own by a sum over the threads (one thread that walked 1,024 experts took 40 us).
static_assert(MOE_MAX_EXPERTS <= 1024, "a thread an expert");
__global__ void __launch_bounds__(1024)
moe_group_kernel(const int *__restrict__ ids, int total, int experts, int *__restrict__ sorted_to_flat,
                 int *__restrict__ tile_expert, int *__restrict__ tile_begin, int *__restrict__ tile_rows,
                 int *__restrict__ n_tiles, int max_tiles, int rows_per_tile, int tiled) {
    __shared__ int count[MOE_MAX_EXPERTS];
    __shared__ int cursor[MOE_MAX_EXPERTS];
    __shared__ int ends[2][1024 / WAVE];
    const int e = threadIdx.x, lane = e % WAVE, wave = e / WAVE;
    if (e < experts) count[e] = 0;
    __syncthreads();
    for (int i = threadIdx.x; i < total; i += blockDim.x) atomicAdd(&count[ids[i]], 1);
    __syncthreads();
    const int pairs = e < experts ? count[e] : 0, tiles = e < tiled ? (pairs + rows_per_tile - 1) / rows_per_tile : 0;
    int at = pairs, tile = tiles;                   // up to and with this expert, first within the wave
#pragma unroll
    for (int off = 1; off < WAVE; off <<= 1) {
        const int a = __shfl_up(at, off, WAVE), b = __shfl_up(tile, off, WAVE);
        if (lane >= off) { at += a; tile += b; }
    }
    if (lane == WAVE - 1) { ends[0][wave] = at; ends[1][wave] = tile; }
    __syncthreads();
    for (int w = 0; w < wave; ++w) { at += ends[0][w]; tile += ends[1][w]; }
    if (e == 1023) n_tiles[0] = min(tile, max_tiles);
    at -= pairs;
    tile -= tiles;
    if (e < experts) cursor[e] = at;
    const int even = tiles ? ((pairs + tiles - 1) / tiles + 15) / 16 * 16 : 0;
    for (int k = 0; k < tiles && tile + k < max_tiles; ++k) {
        tile_expert[tile + k] = e;
        tile_begin[tile + k] = at + k * even;
        tile_rows[tile + k] = min(pairs - k * even, even);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < total; i += blockDim.x) sorted_to_flat[atomicAdd(&cursor[ids[i]], 1)] = i;
}

// ---------------------------------------------------------------- the experts' products
template <class T> struct Mma;
template <> struct Mma<bf16_t> {
    static constexpr int PER_LANE = 8, KSTEP = 32;       // elements of k a lane loads (16 bytes), and a step covers
    typedef u32x4 frag;
    static __device__ __forceinline__ frag zero() { return frag{0u, 0u, 0u, 0u}; }
    static __device__ __forceinline__ frag load(const bf16_t *p) { return *(const frag *)p; }
    static __device__ __forceinline__ frag scaled(frag v, float s) {
        frag o;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float lo = __uint_as_float(v[i] << 16) * s, hi = __uint_as_float(v[i] & 0xffff0000u) * s;
            o[i] = pack2_bf16(lo, hi);
        }
        return o;
    }
    static __device__ __forceinline__ f32x4 mma(frag a, frag b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
    }
};
template <> struct Mma<float> {
    static constexpr int PER_LANE = 4, KSTEP = 16;
    typedef f32x4 frag;
    static __device__ __forceinline__ frag zero() { return frag{0.f, 0.f, 0.f, 0.f}; }
    static __device__ __forceinline__ frag load(const float *p) { return *(const frag *)p; }
    static __device__ __forceinline__ frag scaled(frag v, float s) { return v * s; }
    // four instructions of k = 4: instruction e takes element e of every lane's four, so the sixteen k of a step are
    // shared out the same way on both operands
    static __device__ __forceinline__ f32x4 mma(frag a, frag b, f32x4 c) {
#pragma unroll
        for (int e = 0; e < 4; ++e) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], b[e], c, 0, 0, 0);
        return c;
    }
};

__device__ __forceinline__ float gelu_erf(float z) { return 0.5f * z * (1.0f + erff(z * 0.70710678118654752f)); }

template <class T> struct alignas(4 * sizeof(T)) Quad { T v[4]; };

enum { MOE_UP = 0, MOE_DOWN = 1, MOE_UP_GATED = 2 };

// Both kernels below multiply rows of one expert with that expert's matrix w[e] ([N, K], as it is or PACKED, see Unit) on the
// matrix cores.  The weight is the instruction's first operand (16
// features x k), the rows the second (k x 16 rows): a lane then holds four neighbouring features of
// one row.  Rows and features beyond the tile's or the matrix's end are computed from clamped
// addresses and never stored.  K is a multiple of the elements in 16 bytes.
//   MOE_UP:   x = h [n, K], a row is the token of its pair, scaled by the pair's weight; out_t = act
//             [total, N] at the pair's row (few rows: the flat pair's; many: the sorted one's), gelu applied.
//   MOE_DOWN: x = act [total, K] at the pair's row; out_f [total or n, N] 32-bit at the flat pair
//             (add == 0: stored) or at the pair's token (add == 1: added; only with top == 1).
//   MOE_UP_GATED: x = h [n, K], not scaled; w[e] holds N = 2 * features rows, in turns 16 rows of the gate matrix and the
//             16 rows of the up matrix that meet them; out_t = act [total, N / 2] at the pair's row,
//             silu(gate) * up, or with limit > 0 the limited form with alpha and limit.

// Where a lane's part of the matrix lies: lane (g, l16) of unit (16 rows, KSTEP of k) takes row l16, PER_LANE elements from k = g *
// PER_LANE on.  PACKED: w[e] is [ceil(N / 16)][ceil(K / KSTEP)][64 lanes][PER_LANE], zeros beyond N and K: a wave's load is one piece
// of 1 KB.  Otherwise it is [N][K], and a load takes half a line of each of 16 rows.
template <class T, bool PACKED> struct Unit {
    typedef Mma<T> M;
    const T *p;
    int k_left;                                      // elements of k from this lane's first one on (not PACKED)
    __device__ __forceinline__ Unit(const T *w, int tile, int N, int K, int steps, int lane) {
        if (PACKED) {
            const int tiles = (N + 15) / 16;
            p = w + ((size_t)(tile < tiles ? tile : tiles - 1) * steps * WAVE + lane) * M::PER_LANE;
        } else {
            const int row = tile * 16 + lane % 16;
            p = w + (size_t)(row < N ? row : N - 1) * K + lane / 16 * M::PER_LANE;
            k_left = K - lane / 16 * M::PER_LANE;
        }
    }
    // read once: past the caches' lines that other data lives in, where a load takes whole lines
    __device__ __forceinline__ typename M::frag load(int step) const {
        if (PACKED) return __builtin_nontemporal_load((const typename M::frag *)(p + (size_t)step * WAVE * M::PER_LANE));
        return step * M::KSTEP < k_left ? M::load(p + step * M::KSTEP) : M::zero();
    }
    // the same for a piece that several workgroups read; not PACKED and beyond K: a piece of the row that exists
    __device__ __forceinline__ typename M::frag cached(int step) const {
        return M::load(PACKED ? p + (size_t)step * WAVE * M::PER_LANE : p + min(step * M::KSTEP, k_left - M::PER_LANE));
    }
};

// Both kernels sum K in four parts of so many steps (an even number: 128 bytes a row), one after the other, and add the parts up in
// turn: the kernel for few rows gives each of its waves a part, and a row has the same bits whichever kernel its step goes to.
__device__ __forceinline__ int quarter_steps(int steps) { return (steps + 7) / 8 * 2; }

// Few rows an expert (decoding).  A workgroup takes 32 rows of an expert's matrix and the expert's rows, 16 at a time, or 48 where there are
// more of them; its four waves take a quarter of K each, steps of loads always on their way, and add up through LDS in a fixed order.
// Up to MOE_LIST pairs a step (MOE_LIST_F32 in 32 bits), a workgroup an expert looks through the step's pairs for the expert's (a list in LDS, in any order: a
// row's result does not depend on its place): no kernel in front.  Beyond, the pairs come sorted and in tiles of 16 rows (moe_group_kernel),
// a workgroup a tile: each looking through thousands of numbers took longer than the kernel in front (1,024 experts, 1,024 tokens of eight:
// 552 us, now 143), and an expert that most tokens name was one workgroup's, 16 rows at a time (64 experts, all of 512 tokens
// on one: 120 us, now 24; of 128 tokens 38, now 28).
// What bounds it is the experts' matrices out of memory, once.  One wave for 16 features and all of K left 3 to 4 waves a compute
// unit, which waited for eight loads and then issued the next eight: 2.8 (gated first product) and 3.2 TB/s (second) for 14 of 16
// experts of 2 x 1024 x 2048 and 2048 x 1024, 42 and 18 us; now 24 and 14 us, and 16 experts of 2 x 1408 x 2048 52 -> 34.5 us, 5.3 TB/s.
// A shared expert that every token uses rides along as one more expert (sw: its matrix, packed alike, of s_n rows and s_k columns; only
// while the tokens are few, as each 16 of them read it once): beside the others it costs its bytes, in kernels of its own it took
// 11 and 5 us.
// (Eight steps on their way and half as many waves: 25 and 37.5.)
constexpr int MOE_LIST = 128, MOE_LIST_F32 = 64;      // (in 32 bits the matrix instructions of a workgroup's rows take longer)
template <int N> struct Int { static constexpr int value = N; };
template <class T, int MODE, bool PACKED>
__global__ void __launch_bounds__(256, 4)
moe_gemm_few_kernel(const T *__restrict__ x, int x_stride, const T *__restrict__ w, size_t w_expert_stride, int N, int K,
                    const int *__restrict__ ids, int total, const float *__restrict__ wts, T *__restrict__ out_t,
                    float *__restrict__ out_f, int out_stride, int top, int add, float alpha, float limit, int experts,
                    const T *__restrict__ sx, const T *__restrict__ sw, int s_n, int s_k, T *__restrict__ s_out_t, float *__restrict__ s_out_f,
                    const int *__restrict__ sorted, const int *__restrict__ tile_expert, const int *__restrict__ tile_begin,
                    const int *__restrict__ tile_rows, const int *__restrict__ n_tiles, int max_tiles) {
    typedef Mma<T> M;
    typedef typename M::frag frag;
    constexpr bool GATED = MODE == MOE_UP_GATED, UP = MODE != MOE_DOWN;
    __shared__ int list[MOE_LIST], found;
    __shared__ f32x4 red[4][2][WAVE];
    const int tid = threadIdx.x, wave = tid / WAVE, lane = tid % WAVE, g = lane / 16, l16 = lane % 16;
    const bool shared = (int)blockIdx.y == (sorted ? max_tiles : experts);
    if (sorted && !shared && (int)blockIdx.y >= n_tiles[0]) return;
    const int e = sorted && !shared ? tile_expert[blockIdx.y] : (int)blockIdx.y;
    const T *we = w + (size_t)e * w_expert_stride;
    if (shared) {                                    // every token's rows [n, s_k] and a matrix of its own size
        total /= top;
        top = 1;
        x = sx;
        we = sw;
        N = s_n;
        K = s_k;
        x_stride = GATED ? x_stride : s_k;
        out_t = s_out_t;
        out_f = s_out_f;
        out_stride = GATED ? s_n / 2 : out_stride;
        alpha = 1.f;
        limit = 0.f;
    }
    if ((int)blockIdx.x * 32 >= N) return;
    const int tile0 = 2 * blockIdx.x, steps = (K + M::KSTEP - 1) / M::KSTEP, per = quarter_steps(steps);
    const int s0 = wave * per, s1 = min(steps, s0 + per);
    const Unit<T, PACKED> w0(we, tile0, N, K, steps, lane), w1(we, tile0 + 1, N, K, steps, lane);
    const int *rows = list;                          // the pairs of this workgroup's rows (null: row r is token r)
    int count = total;
    if (shared) {
        rows = nullptr;
    } else if (sorted) {
        rows = sorted + tile_begin[blockIdx.y];
        count = tile_rows[blockIdx.y];
    } else {
        if (tid == 0) found = 0;
        __syncthreads();
        if (tid < total && ids[tid] == e) list[atomicAdd(&found, 1)] = tid;      // (total is at most MOE_LIST, a thread a pair)
        __syncthreads();
        count = found;
    }
    // rows r0 .. of RT tiles of 16
    auto pass = [&](auto rt, auto ahead, int r0) {
        constexpr int RT = decltype(rt)::value, AHEAD = decltype(ahead)::value;
        int flat[RT];
        unsigned xat[RT];                            // (few rows: their elements are less than 2^32)
        float sc[RT];
#pragma unroll
        for (int m = 0; m < RT; ++m) {
            const int r = min(r0 + 16 * m + l16, count - 1);
            flat[m] = rows ? rows[r] : r;
            xat[m] = (unsigned)(UP ? flat[m] / top : flat[m]) * x_stride + g * M::PER_LANE;
            if (MODE == MOE_UP) sc[m] = wts[flat[m]];
        }
        const int x_left = K - g * M::PER_LANE;
        f32x4 acc[RT][2];
#pragma unroll
        for (int m = 0; m < RT; ++m) acc[m][0] = acc[m][1] = f32x4{0.f, 0.f, 0.f, 0.f};
        frag a0[AHEAD], a1[AHEAD], b[AHEAD][RT];
        auto fetch = [&](int u, int s) {
            a0[u] = w0.load(s);
            a1[u] = w1.load(s);
#pragma unroll
            for (int m = 0; m < RT; ++m) b[u][m] = s * M::KSTEP < x_left ? M::load(x + xat[m] + s * M::KSTEP) : M::zero();
        };
#pragma unroll
        for (int u = 0; u < AHEAD; ++u)
            if (s0 + u < s1) fetch(u, s0 + u);
        for (int s = s0; s < s1; s += AHEAD) {
#pragma unroll
            for (int u = 0; u < AHEAD; ++u) {
                if (s + u >= s1) break;
#pragma unroll
                for (int m = 0; m < RT; ++m) {
                    const frag bb = MODE == MOE_UP ? M::scaled(b[u][m], sc[m]) : b[u][m];
                    acc[m][0] = M::mma(a0[u], bb, acc[m][0]);
                    acc[m][1] = M::mma(a1[u], bb, acc[m][1]);
                }
                if (s + u + AHEAD < s1) fetch(u, s + u + AHEAD);
            }
        }
#pragma unroll
        for (int m = 0; m < RT; ++m) {
            if (m > 0 && r0 + 16 * m >= count) break;
            if (r0 + m) __syncthreads();             // the sums of the rows before have been read
            red[wave][0][lane] = acc[m][0];
            red[wave][1][lane] = acc[m][1];
            __syncthreads();
            // the first wave stores (with two products' sums the first two, one each): four neighbouring features of a row a lane
            if (wave < (GATED ? 1 : 2)) {
                const bool valid = r0 + 16 * m + l16 < count;
                const f32x4 v = ((red[0][wave][lane] + red[1][wave][lane]) + red[2][wave][lane]) + red[3][wave][lane];
                const int dst = !UP && add ? flat[m] / top : flat[m];
                if constexpr (GATED) {
                    const f32x4 up = ((red[0][1][lane] + red[1][1][lane]) + red[2][1][lane]) + red[3][1][lane];
                    Quad<T> q;
#pragma unroll
                    for (int i = 0; i < 4; ++i) q.v[i] = from_f32<T>(gate_up_of(v[i], up[i], alpha, limit));
                    if (valid && tile0 * 16 < N) *(Quad<T> *)(out_t + (size_t)dst * out_stride + tile0 * 8 + 4 * g) = q;
                } else {
                    const int col = (tile0 + wave) * 16 + 4 * g;         // (N is a multiple of 4)
                    if (valid && col < N) {
                        if constexpr (MODE == MOE_UP) {
                            Quad<T> q;
#pragma unroll
                            for (int i = 0; i < 4; ++i) q.v[i] = from_f32<T>(gelu_erf(v[i]));
                            *(Quad<T> *)(out_t + (size_t)dst * out_stride + col) = q;
                        } else {
                            f32x4 *o = (f32x4 *)(out_f + (size_t)dst * out_stride + col);
                            *o = add ? *o + v : v;
                        }
                    }
                }
            }
        }
    };
    if (count <= 16) {
        if (count > 0) pass(Int<1>(), Int<4>(), 0);
    } else {
        for (int r0 = 0; r0 < count; r0 += 48) pass(Int<3>(), Int<2>(), r0);
    }
}

// The least pairs (one to eight tokens of two, say): a workgroup looks for the blockIdx.y-th expert that any of them names, so the launch holds no
// workgroups of experts without a pair, and has eight waves, a quarter of K and one of the two tiles each, with eight steps on their way: few workgroups then
// ask for as much at a time as many would.  An expert's pairs go sixteen at a time; a token may name an expert more than once, so they may be more than the tokens, and what is beyond the
// first sixteen goes through a loop of its own (one loop for all takes more registers: 14.8 us in the place of 10.8 for a token of two).  The sums are added up as in the kernel for few rows: the same bits.  What bounds it is the way of the numbers of the experts
// and of their matrices' first lines through memory, one after the other, and what a workgroup does to find its pairs: a turn an expert, and one permutation of the lanes (a
// turn a pair and fifteen for the rows took 8 us of 64 pairs, 4 experts of 2 x 1024 x 1024: 20.5, now 12.7).  One MI355X, both products, us, with the kernel for few rows everywhere and now: a token of two experts of
// 2 x 1024 x 2048 with a shared one of 704 13.6 and 11.9, two tokens 19.5 and 17.5; a token of two of 2 x 1408 x 2048 14.4 and 11.9, of four of 2 x 512 x 2048 11.9 and 10.5, of one of
// 2 x 3584 x 1024 16.4 and 13.1; four tokens of two of 64 of 2 x 512 x 1024 13.8 and 10.2.
constexpr int MOE_SLOTS = 64, MOE_SLOT_ROWS = 16;      // pairs, a lane each; tokens
// Whether the kernel takes a product of `rows` features.  From some 400 workgroups on four waves with two tiles each read the rows half as often: four tokens of two of 2 x 1408 x 2048 23.7 and 25.4, eight of
// four of 2 x 512 x 2048 29.3 and 46.6.  From 256 on it is so where half of the experts or more are named, so that the other kernel holds few workgroups for nothing: 12 tokens of two of 32 of 2 x 256 x 512 9.0
// and 9.8, 3 of four of 16 of 2 x 512 x 2048 15.8 and 16.4; but 3 of four of 64 of 2 x 512 x 1024 15.0 and 11.9.  With more than a dozen pairs an expert the turns of the two kernels are equally full: 16 tokens of
// four, all of 4 experts of 2 x 1024 x 1024, 32 bits 19.0 and 20.0, 12 tokens 18.4 and 18.3.
static bool moe_slots_take(int n, int top, int experts, int rows) {
    const int total = n * top, slots = total < experts ? total : experts;
    return total <= MOE_SLOTS && n <= MOE_SLOT_ROWS && total <= 12 * slots && (rows + 31) / 32 * slots <= (experts >= 2 * slots ? 384 : 256);
}
// The same for whoever wants to know.
LCU_API int lcu_moe_slots_take(int n, int top, int experts, int rows) { return n > 0 && top > 0 && experts > 0 && rows > 0 && moe_slots_take(n, top, experts, rows); }

template <class T, int MODE, bool PACKED>
__global__ void __launch_bounds__(512)
moe_gemm_slots_kernel(const T *__restrict__ x, int x_stride, const T *__restrict__ w, size_t w_expert_stride, int N, int K,
                      const int *__restrict__ ids, int total, const float *__restrict__ wts, T *__restrict__ out_t,
                      float *__restrict__ out_f, int out_stride, int top, int add, float alpha, float limit, int experts, int slots,
                      const T *__restrict__ sx, const T *__restrict__ sw, int s_n, int s_k, T *__restrict__ s_out_t, float *__restrict__ s_out_f) {
    typedef Mma<T> M;
    typedef typename M::frag frag;
    constexpr bool GATED = MODE == MOE_UP_GATED, UP = MODE != MOE_DOWN;
    __shared__ f32x4 red[4][2][WAVE];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), lane = threadIdx.x % WAVE, g = lane / 16, l16 = lane % 16;
    const int part = wave & 3, side = wave >> 2;
    const bool shared = (int)blockIdx.y == slots;
    const T *we = sw;
    int count = total, sorted = lane;                // lane r: the expert's r-th pair
    if (shared) {                                    // every token's rows [n, s_k] and a matrix of its own size
        count /= top;                                // (at most MOE_SLOT_ROWS)
        top = 1;
        x = sx;
        N = s_n;
        K = s_k;
        x_stride = GATED ? x_stride : s_k;
        out_t = s_out_t;
        out_f = s_out_f;
        out_stride = GATED ? s_n / 2 : out_stride;
        alpha = 1.f;
        limit = 0.f;
    } else {
        const int mine = lane < total ? ids[lane] : -1;
        unsigned long long left = __ballot(mine >= 0 && mine < experts), pairs = 0;      // (identity experts have no matrices)
        int e = 0;
        for (int y = 0; y <= (int)blockIdx.y; ++y) { // an expert a turn, in the order of their first pairs
            left &= ~pairs;
            if (!left) return;
            e = __builtin_amdgcn_readlane(mine, __builtin_ctzll(left));
            pairs = __ballot(mine == e);
        }
        count = __popcll(pairs);
        const int before = __builtin_amdgcn_mbcnt_hi((uint32_t)(pairs >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)pairs, 0));
        sorted = __builtin_amdgcn_ds_permute(4 * (mine == e ? before : count + lane - before), lane);
        we = w + (size_t)e * w_expert_stride;
    }
    if ((int)blockIdx.x * 32 >= N) return;
    const int tile0 = 2 * blockIdx.x, steps = (K + M::KSTEP - 1) / M::KSTEP, per = quarter_steps(steps);
    const int s0 = min(steps, part * per), s1 = min(steps, s0 + per);
    // sixteen of the pairs, from the r0-th on
    auto pass = [&](auto ahead, int r0) {
        constexpr int AHEAD = decltype(ahead)::value;
        const Unit<T, PACKED> wu(we, tile0 + side, N, K, steps, lane);
        const int flat = __builtin_amdgcn_ds_bpermute(4 * min(r0 + l16, count - 1), sorted);      // of row l16
        const T *xr = x + (size_t)(UP ? flat / top : flat) * x_stride + g * M::PER_LANE;
        const float sc = MODE == MOE_UP ? wts[flat] : 1.f;
        const int x_left = K - g * M::PER_LANE;
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
        frag a[AHEAD], b[AHEAD];
        auto fetch = [&](int u, int s) {
            a[u] = wu.load(s);
            b[u] = s * M::KSTEP < x_left ? M::load(xr + s * M::KSTEP) : M::zero();
        };
#pragma unroll
        for (int u = 0; u < AHEAD; ++u)
            if (s0 + u < s1) fetch(u, s0 + u);
        for (int s = s0; s < s1; s += AHEAD) {
#pragma unroll
            for (int u = 0; u < AHEAD; ++u) {
                if (s + u >= s1) break;
                acc = M::mma(a[u], MODE == MOE_UP ? M::scaled(b[u], sc) : b[u], acc);
                if (s + u + AHEAD < s1) fetch(u, s + u + AHEAD);
            }
        }
        asm volatile("s_nop 3" : "+v"(acc));         // the last matrix instruction's wait, which the compiler leaves a state short behind the branches
        if (r0 > 0) __syncthreads();                 // the sums of the rows before have been read
        red[part][side][lane] = acc;
        __syncthreads();
        // the first wave stores (with two products' sums the first two, one each): four neighbouring features of a row a lane
        if (wave >= (GATED ? 1 : 2) || r0 + l16 >= count) return;
        const f32x4 v = ((red[0][wave][lane] + red[1][wave][lane]) + red[2][wave][lane]) + red[3][wave][lane];
        const int dst = !UP && add ? flat / top : flat;
        if constexpr (GATED) {
            const f32x4 up = ((red[0][1][lane] + red[1][1][lane]) + red[2][1][lane]) + red[3][1][lane];
            Quad<T> q;
#pragma unroll
            for (int i = 0; i < 4; ++i) q.v[i] = from_f32<T>(gate_up_of(v[i], up[i], alpha, limit));
            *(Quad<T> *)(out_t + (size_t)dst * out_stride + tile0 * 8 + 4 * g) = q;
        } else {
            const int col = (tile0 + wave) * 16 + 4 * g; // (N is a multiple of 4)
            if (col >= N) return;
            if constexpr (MODE == MOE_UP) {
                Quad<T> q;
#pragma unroll
                for (int i = 0; i < 4; ++i) q.v[i] = from_f32<T>(gelu_erf(v[i]));
                *(Quad<T> *)(out_t + (size_t)dst * out_stride + col) = q;
            } else {
                f32x4 *o = (f32x4 *)(out_f + (size_t)dst * out_stride + col);
                *o = add ? *o + v : v;
            }
        }
    };
    pass(Int<8>(), 0);
    for (int r0 = 16; r0 < count; r0 += 16) pass(Int<2>(), r0);
}

// Many rows an expert (prompts): tiles of up to 32, 64, 96 or 128 rows; a block of four waves takes a tile and 128 features, a wave 32 of them with all
// rows.  The rows go through LDS in steps of 128 bytes of k, in two buffers in turn with one barrier a step; no two waves want the same piece of the
// matrix, so each loads its own straight into registers.  Both are two steps ahead.  MT: tiles of 16 rows that are multiplied.
// What bounds it are the turns of loads, LDS and barrier of the two blocks that a compute unit holds (half the matrix instructions take as long) and, up
// to 50 rows an expert, the matrices out of memory.  Tiles of 64 rows whose matrices went through LDS too took, per pass of both products, 16 experts
// of 2048 x 2048 with 2,014 tokens of two each 241 us, now 155; gated, 2 x 1024: 180 and 132; 200 tokens of two 77 and 51.  (Rows copied into LDS by the
// loads themselves, four buffers, the barrier in the middle of the instructions: the same times; 64 rows and three blocks: 5 to 30 % longer.)
template <class T, int MODE, bool PACKED, int MT>
__device__ __forceinline__ void moe_many_tile(T *__restrict__ xs, const T *__restrict__ x, int x_stride, const T *__restrict__ we, int N, int K,
                                              const int *__restrict__ sorted_to_flat, const float *__restrict__ wts, int n0, int row0, int rows,
                                              T *__restrict__ out_t, float *__restrict__ out_f, int out_stride, int top, int add, float alpha, float limit) {
    typedef Mma<T> M;
    typedef typename M::frag frag;
    constexpr int PL = M::PER_LANE;                 // elements in 16 bytes
    constexpr int KS = 128 / sizeof(T);             // elements of k a step
    constexpr int CH = KS / PL;                     // 16-byte pieces of a row a step: 8
    constexpr int SS = KS / M::KSTEP;               // units of k a step: 2
    constexpr int XP = MT / 2;                      // rows that a thread copies
    const int tid = threadIdx.x, wave = tid / WAVE, lane = tid % WAVE, g = lane / 16, l16 = lane % 16;
    const int ch = tid % CH;                        // this thread's piece of k in every row it copies
    unsigned xrow[XP];                              // (a row's number, not its address: registers are short)
    float xsc[XP];
#pragma unroll
    for (int i = 0; i < XP; ++i) {
        const int r = tid / CH + 32 * i;
        const int srow = row0 + (r < rows ? r : 0), flat = MODE != MOE_DOWN ? sorted_to_flat[srow] : srow;
        xrow[i] = MODE != MOE_DOWN ? flat / top : flat;
        xsc[i] = MODE == MOE_UP ? wts[flat] : 1.f;
    }
    const int units = (K + M::KSTEP - 1) / M::KSTEP, steps = (units + SS - 1) / SS, tile0 = n0 / 16 + 2 * wave;
    const Unit<T, PACKED> w0(we, tile0, N, K, units, lane), w1(we, tile0 + 1, N, K, units, lane);
    frag xreg[2][XP], a[2][SS][2];
    const int full = K / KS;                        // steps that are all within K
    // every load is issued, with a place that exists: beyond the last step it is the last step's, beyond K the last piece of the row
    auto rows_of = [&](auto buf, int step) {
        const unsigned k = min(min(step, steps - 1) * KS + ch * PL, K - PL);
#pragma unroll
        for (int i = 0; i < XP; ++i) xreg[decltype(buf)::value][i] = M::load(x + ((size_t)xrow[i] * (unsigned)x_stride + k));
    };
    auto weights_of = [&](auto buf, int step) {
#pragma unroll
        for (int u = 0; u < SS; ++u) {
            const int s = min(min(step, steps - 1) * SS + u, units - 1);
            a[decltype(buf)::value][u][0] = w0.cached(s);
            a[decltype(buf)::value][u][1] = w1.cached(s);
        }
    };
    auto rows_to_lds = [&](auto buf, int step) {
        constexpr int B = decltype(buf)::value;
        if (step >= full) {                         // the last step, partly beyond K (a branch, no select in every step)
            asm volatile("");
            if (step * KS + ch * PL >= K)
#pragma unroll
                for (int i = 0; i < XP; ++i) xreg[B][i] = M::zero();
        }
#pragma unroll
        for (int i = 0; i < XP; ++i) {
            frag v = xreg[B][i];
            if (MODE == MOE_UP) v = M::scaled(v, xsc[i]);
            *(frag *)(xs + (B * 16 * MT + tid / CH + 32 * i) * KS + (ch ^ (tid / CH % 8)) * PL) = v;
        }
    };
    f32x4 acc[2][MT], sum[2][MT];
#pragma unroll
    for (int ft = 0; ft < 2; ++ft)
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[ft][m] = sum[ft][m] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int part = quarter_steps(units) / SS;     // steps of a part of K
    int left = part;                                // of this part that are left
    auto one = [&](auto buf, int step) {
        constexpr int B = decltype(buf)::value;
        lds_barrier();                              // this step's rows are there, the step before has been read
        rows_of(buf, step + 2);
        if (left == 0) {
            left = part;
#pragma unroll
            for (int ft = 0; ft < 2; ++ft)
#pragma unroll
                for (int m = 0; m < MT; ++m) {
                    sum[ft][m] += acc[ft][m];
                    acc[ft][m] = f32x4{0.f, 0.f, 0.f, 0.f};
                }
        }
        --left;
        if (step >= full) {
            asm volatile("");
#pragma unroll
            for (int u = 0; u < SS; ++u)
                if (step * SS + u >= units || (!PACKED && (step * SS + u) * M::KSTEP + g * PL >= K)) a[B][u][0] = a[B][u][1] = M::zero();
        }
        __builtin_amdgcn_sched_barrier(0);
        // piece p of row r lies at p ^ (r % 8) of the row: whichever lanes the LDS serves together, they are in different banks
        frag b[SS * MT];
#pragma unroll
        for (int i = 0; i < SS * MT; ++i)
            b[i] = *(const frag *)(xs + (B * 16 * MT + 16 * (i % MT) + l16) * KS + ((i / MT * 4 + g) ^ (l16 % 8)) * PL);
#pragma unroll
        for (int i = 0; i < SS * MT; ++i) {
            const int u = i / MT, m = i % MT;
            acc[0][m] = M::mma(a[B][u][0], b[i], acc[0][m]);
            acc[1][m] = M::mma(a[B][u][1], b[i], acc[1][m]);
        }
        // RA reads of rows are always on their way ahead of the products
        constexpr int RA = 4, PER = 2 * (sizeof(T) == 4 ? 4 : 1);
        __builtin_amdgcn_sched_group_barrier(0x100, RA, 0);
#pragma unroll
        for (int i = RA; i < SS * MT; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, PER, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x008, PER * RA, 0);
        __builtin_amdgcn_sched_barrier(0);
        weights_of(buf, step + 2);
        rows_to_lds(Int<1 - B>(), step + 1);
    };
    rows_of(Int<0>(), 0);
    weights_of(Int<0>(), 0);
    rows_of(Int<1>(), 1);
    weights_of(Int<1>(), 1);
    rows_to_lds(Int<0>(), 0);
    int step = 0;
    for (; step + 1 < steps; step += 2) {
        one(Int<0>(), step);
        one(Int<1>(), step + 1);
    }
    if (step < steps) one(Int<0>(), step);
#pragma unroll
    for (int ft = 0; ft < 2; ++ft)
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[ft][m] = sum[ft][m] + acc[ft][m];
    // The results go out through LDS, 64 rows at a time: a wave then stores whole lines (from where the products leave them a store was 64 separate words, and the
    // activation's code stood here 64 times).  Four neighbouring features q of row r lie at q ^ (r % 8).  One MI355X, 4,096 pairs, us: K of 64, all but the loop, up with gelu to
    // 2,048 features 24.5, now 19.1, down 26.9 and 14.5; both products of 2048 x 2048 185 and 155.
    constexpr int EP = MT < 4 ? MT : 4, QUADS = MODE == MOE_UP_GATED ? 16 : 32, ROWS = 256 / QUADS;      // quads of features of a row, rows stored at a time
    float *out_rows = (float *)xs;
    const int q = tid % QUADS, r_in = tid / QUADS, col = n0 / (32 / QUADS) + 4 * q;
    int dst[16 * MT / ROWS];
    if (MODE == MOE_DOWN) {
#pragma unroll
        for (int i = 0; i < 16 * MT / ROWS; ++i) {
            dst[i] = sorted_to_flat[row0 + min(r_in + ROWS * i, rows - 1)];
            if (add) dst[i] /= top;
        }
    }
#pragma unroll
    for (int m0 = 0; m0 < MT; m0 += EP) {
        lds_barrier();                              // what lay there has been read
#pragma unroll
        for (int m = m0; m < m0 + EP && m < MT; ++m)
#pragma unroll
            for (int ft = 0; ft < 2; ++ft) *(f32x4 *)(out_rows + (16 * (m - m0) + l16) * 128 + 4 * ((8 * wave + 4 * ft + g) ^ (l16 % 8))) = acc[ft][m];
        lds_barrier();
        auto at = [&](int r, int quad) { return *(const f32x4 *)(out_rows + r * 128 + 4 * (quad ^ (r % 8))); };
        const int here = min(rows - 16 * m0, 16 * EP);
        if constexpr (MODE == MOE_DOWN) {
#pragma unroll
            for (int i = 0; i < 16 * (MT - m0 < EP ? MT - m0 : EP) / ROWS; ++i) {
                const int r = r_in + ROWS * i;
                if (r >= here || col >= N) continue;
                pair_f32x4_at *o = (pair_f32x4_at *)(out_f + (size_t)dst[16 * m0 / ROWS + i] * out_stride + col);
                const f32x4 v = at(r, q);
                *o = add ? *o + v : v;
            }
        } else {
#pragma unroll 1
            for (int r = r_in; r < here; r += ROWS) {
                Quad<T> to;
                if constexpr (MODE == MOE_UP_GATED) {       // a wave's first 16 features are a gate block, its second the up block that meets it
                    const f32x4 gate = at(r, 8 * (q / 4) + q % 4), up = at(r, 8 * (q / 4) + 4 + q % 4);
#pragma unroll
                    for (int i = 0; i < 4; ++i) to.v[i] = from_f32<T>(gate_up_of(gate[i], up[i], alpha, limit));
                } else {
                    const f32x4 v = at(r, q);
#pragma unroll
                    for (int i = 0; i < 4; ++i) to.v[i] = from_f32<T>(gelu_erf(v[i]));
                }
                if (col < (MODE == MOE_UP_GATED ? N / 2 : N)) *(Quad<T> *)(out_t + (size_t)(row0 + 16 * m0 + r) * out_stride + col) = to;
            }
        }
    }
}

template <class T, int MODE, bool PACKED>
__global__ void __launch_bounds__(256, 2)
moe_gemm_many_kernel(const T *__restrict__ x, int x_stride, const T *__restrict__ w, size_t w_expert_stride, int N, int K,
                     const int *__restrict__ sorted_to_flat, const float *__restrict__ wts,
                     const int *__restrict__ tile_expert, const int *__restrict__ tile_begin,
                     const int *__restrict__ tile_rows, const int *__restrict__ n_tiles, T *__restrict__ out_t,
                     float *__restrict__ out_f, int out_stride, int top, int add, float alpha, float limit) {
    __shared__ __attribute__((aligned(16))) T xs[2 * MOE_TILE_ROWS * 128 / sizeof(T)];
    // Workgroups go to the chip's eight dies in turn (workgroup i to die i % 8), and each die has an L2 of its own.  The work, in the order
    // four tiles after four tiles, their feature blocks, the tiles, is cut into eight pieces: what a die has at hand at a time are a few
    // tiles' rows and a few experts' matrices, and each comes to one die (at the pieces' borders two).
    // (By feature blocks, every die read every row: 16 experts, 200 tokens of two 65 us, 51 so; 2,040 tokens 157 and 142.)
    const int n_fb = (N + 127) / 128, tiles = n_tiles[0], each = (tiles * n_fb + 7) / 8, at = blockIdx.x / 8, item = blockIdx.x % 8 * each + at;
    if (at >= each || item >= tiles * n_fb) return;
    const int first = item / (4 * n_fb) * 4, rest = item - first * n_fb, side = min(4, tiles - first), fb = rest / side, tile = first + rest % side;
    const T *we = w + (size_t)tile_expert[tile] * w_expert_stride;
    const int row0 = tile_begin[tile], rows = tile_rows[tile];
#define TILE(MT) moe_many_tile<T, MODE, PACKED, MT>(xs, x, x_stride, we, N, K, sorted_to_flat, wts, fb * 128, row0, rows, out_t, out_f, out_stride, top, add, alpha, limit)
    if (rows > 96) TILE(8);
    else if (rows > 64) TILE(6);
    else if (rows > 32) TILE(4);
    else TILE(2);
#undef TILE
}

// out[t] = the token's sum (pair_sum.h).  Four columns a thread; d is a multiple of 4.
template <class T>
__global__ void __launch_bounds__(256)
moe_combine_kernel(float *out, PairSum p, int n, int d) {
    const int c = (blockIdx.x * blockDim.x + threadIdx.x) * 4;
    if (c >= d) return;
    for (size_t t = blockIdx.y; t < (size_t)n; t += gridDim.y) *(pair_f32x4_at *)(out + t * d + c) = pair_sum4<T>(p, t, c, d);
}

// out: [n, d] 32-bit (p->base may be the same memory); p: in host memory.
LCU_API int lcu_moe_combine(float *out, const PairSum *p, int type, int n, int d, hipStream_t stream) {
    if (n <= 0) return LCU_OK;
    if (!out || !p || !pair_sum_ok(*p, d) || (type != LCU_F32 && type != LCU_BF16)) return LCU_BAD_ARGUMENT;
    const dim3 gc((d + 1023) / 1024, n < 65535 ? n : 65535), block(256);
    if (type == LCU_BF16) moe_combine_kernel<bf16_t><<<gc, block, 0, stream>>>(out, *p, n, d);
    else moe_combine_kernel<float><<<gc, block, 0, stream>>>(out, *p, n, d);
    LCU_LAUNCH_CHECK();
    return LCU_OK;
}

// Rows of a tile for n * top pairs over so many experts: while an expert has 16 rows or fewer on average the kernel for few rows, with no
// tiles up to MOE_LIST pairs (0; MOE_LIST_F32 in 32 bits) and tiles of 16 beyond.  In 32 bits 32 then: the products are bound by their matrix instructions, and small tiles
// are shared out evenly over the compute units.  In bfloat16 what should take least: the two products' workgroups (a tile and 128 features each) in turns of as many as there are compute
// units, a turn as long as the K of its product times the rows that a workgroup multiplies and what it spends besides, 60 rows' time; as many tiles as there are where every
// token chooses evenly, with one and a half times their deviation, and workgroups of the rows of the largest expert of so many.
// Measured with 2 to 64 experts of 520 x 272 to 4096 x 4096 and 17 to 1,024 rows each on average, evenly and with a few experts taking most, 288 shapes: bfloat16 0.9 % (3.9 % unevenly)
// more than the best of the four sizes, 17 % at most, 32 bits 2.8 % and 0.2 %, 16 % at most.  Always 96, but 128 for 80 to 120 rows, was 11 % and 10 % more, 32 bits 31 % and 51 %; tiles of
// 64 10 % and 9 %, 32 bits 15 % and 24 %.  (us a pass of both products, with 32, 64, 96 and 128 rows: 16 experts, gated, of 1024 x 512, 88 rows 30, 27, 32, 34, 252 rows 53, 50, 45, 50; of 2048 x
// 1024, 88 rows 71, 55, 65, 55, 252 rows 135, 111, 100, 109; 32 bits, 8 of 1024 x 1024, 88 rows: 59, 94, 131, 165.  The 60 rows' time: over 40 shapes 20 to 70 were tried, 50 and 60 are best.)
// The caller sizes its scratch with it: max_tiles = min(total, total / rows + experts), or 0.
LCU_API int lcu_moe_tile_rows(int type, int total, int experts, int up_rows, int d, int ff) {
    if ((long long)total <= 16ll * experts) return total > (type == LCU_F32 ? MOE_LIST_F32 : MOE_LIST) ? 16 : 0;
    if (type == LCU_F32) return 32;
    const double mean = (double)total / experts, deviation = sqrt(mean), most = mean + (1 + log2((double)experts) / 6) * deviation;
    int best = 0;
    double least = 0;
    for (int tile = most <= 32 ? 64 : 32; tile <= MOE_TILE_ROWS; tile += 32) {      // (half empty tiles take no longer than full ones of half the rows, and hold an expert that has a few rows more)
        const int all = (int)fmax((mean - 6 * deviation) / tile, 1);      // tiles that every expert has
        double per = all, spread = 0;                // tiles of an expert and their variance
        for (int j = all; j <= (int)(most / tile) + 2; ++j) {
            const double beyond = 0.5 * erfc((j * tile + 0.5 - mean) / deviation * 0.70710678118654752);   // the share of the experts with more than j tiles' rows
            per += beyond;
            spread += beyond * (1 - beyond);
        }
        const double tiles = fmin(experts * ceil(most / tile), experts * per + 1.5 * sqrt(experts * spread)), rows = fmin(tile, ceil(most / ceil(mean / tile) / 32) * 32);
        auto turns = [&](int features) { return ceil(tiles * ((features + 127) / 128) / 256); };
        const double time = (turns(up_rows) * d + turns(d) * ff) * (60 + rows);
        if (!best || time < least) { best = tile; least = time; }
    }
    return best;
}

// h: [n, d] of `type`; router: [experts, d] 32-bit; ids, wts: [n * top].
// bias: null or [experts] 32-bit; mode 0: sigmoid weights, 1: softmax over the chosen; extra, gates: see the kernel
// (router then has experts + extra rows).
LCU_API int lcu_moe_route(const void *h, int type, const float *router, const float *bias, int *ids, float *wts, float *gates,
                          int n, int d, int experts, int top, int mode, int extra, int groups, int keep, int renorm, float scale,
                          hipStream_t stream) {
    if (n <= 0) return LCU_OK;
    if (d <= 0 || experts <= 0 || experts > MOE_MAX_EXPERTS || top <= 0 || top > experts || mode < 0 || mode > 2 ||
        extra < 0 || extra > MOE_MAX_EXTRA || (extra && !gates) || groups < 1 ||
        (groups > 1 && (mode != 2 || experts % groups || keep < 1 || keep > groups || top > keep * (experts / groups))))
        return LCU_BAD_ARGUMENT;
    const bool few = n <= 256 && experts > 4;
    if (type != LCU_F32 && type != LCU_BF16) return LCU_BAD_ARGUMENT;
#define ARGS experts, top, mode, extra, groups, keep, renorm, scale
#define GENERAL(T, TH) moe_route_kernel<T, TH><<<dim3(n), dim3(TH), 0, stream>>>((const T *)h, router, bias, ids, wts, gates, d, ARGS)
#define ROWS(T, CHUNKS, TOKENS)                                                                                                                          \
    case 8 * CHUNKS + TOKENS:                                                                                                                             \
        moe_route_rows_kernel<T, CHUNKS, TOKENS><<<dim3((n + TOKENS - 1) / TOKENS), dim3(ROUTE_THREADS), TOKENS * 3 * (experts + extra) * sizeof(float), stream>>>( \
            (const T *)h, router, bias, ids, wts, gates, n, ARGS);                                                                                        \
        break;
#define GO(T)                                                                                                                                            \
    do {                                                                                                                                                  \
        if (few) GENERAL(T, 1024);                                                                                                                        \
        else switch (8 * chunks + tokens) {                                                                                                               \
            ROWS(T, 1, 1) ROWS(T, 1, 2) ROWS(T, 1, 4) ROWS(T, 2, 1) ROWS(T, 2, 2) ROWS(T, 2, 4) ROWS(T, 3, 1) ROWS(T, 3, 2) ROWS(T, 3, 4)                   \
            ROWS(T, 4, 1) ROWS(T, 4, 2) ROWS(T, 4, 4) ROWS(T, 5, 2) ROWS(T, 6, 2) ROWS(T, 7, 2) ROWS(T, 8, 2) ROWS(T, 8, 4)                                 \
            default: GENERAL(T, 256);                                                                                                                     \
        }                                                                                                                                                 \
    } while (0)
    const int chunks = d / 512, tokens = d % 512 || chunks > ROUTE_CHUNKS ? 0 : route_tokens(n, chunks, experts + extra, type);
    if (type == LCU_F32) GO(float);
    else GO(bf16_t);
#undef GO
#undef ROWS
#undef GENERAL
#undef ARGS
    LCU_LAUNCH_CHECK();
    return LCU_OK;
}

// tile_rows: what lcu_moe_tile_rows says, or beyond 16 another multiple of 16 up to MOE_TILE_ROWS (the results are the same).
// ints: scratch of total + 3 * max_tiles + 1 entries, laid out as sorted_to_flat, tile_expert, tile_begin,
// tile_rows, n_tiles (null with tile_rows 0).
// w_up: [experts, ff, d], w_down: [experts, d, ff] of `type`; packed_up, packed_down: in the order of Unit.  act: scratch [total, ff] of `type`; y: scratch
// [total, d] 32-bit (only read and written when top > 1 or gated).  out: [n, d] 32-bit, added to.
// gated: w_up is [experts, 2 * ff, d], in turns 16 rows of the gate matrix and the 16 rows of the up matrix that meet
// them (ff a multiple of 16); act = silu(gate h) * (up h), and the weight scales what comes out; fresh: out is written
// and not added to; limit > 0: the limited activation (gate_act.h) with alpha and limit instead of silu.  identity: ids may name experts + identity experts; the last `identity` have no matrices and return the
// token's input.  shared (null or
// [n, d] of `type`) with shared_gate (null or [n] 32-bit): rows that are added beside the experts', times the gate.  shared_up,
// shared_down (null, or the matrices [2 * shared_ff, d] and [d, shared_ff] of a shared expert that is computed here, with silu, in the order of Unit
// like w_up and w_down; only with tile_rows 16 or 0): act then holds n * shared_ff elements more and y n rows more.
// defer: with top > 1 or gated, and any tile_rows, the sum is left to whoever reads y, and out is not used.
LCU_API int lcu_moe_experts(const void *h, int type, const int *ids, const float *wts, int tile_rows, int *ints, int max_tiles,
                            const void *w_up, int packed_up, const void *w_down, int packed_down, void *act, float *y, float *out, int n, int d, int ff,
                            int experts, int top, int gated, const void *shared, const float *shared_gate, const void *shared_up,
                            const void *shared_down, int shared_ff, int fresh, int identity, float alpha, float limit, int defer, hipStream_t stream) {
    if (n <= 0) return LCU_OK;
    const int per = type == LCU_BF16 ? 8 : 4;
    if (d <= 0 || ff <= 0 || d % per || ff % per || experts <= 0 || experts > MOE_MAX_EXPERTS || top <= 0 ||
        (type != LCU_F32 && type != LCU_BF16) || (gated && ff % 16) || (shared && !gated) || (fresh && !gated) || identity < 0 ||
        (identity && !gated) || experts + identity > MOE_MAX_EXPERTS)
        return LCU_BAD_ARGUMENT;
    const int total = n * top;
    const bool few = tile_rows <= 16;
    if (tile_rows < 0 || tile_rows > MOE_TILE_ROWS || tile_rows % 16 || (!tile_rows && total > (type == LCU_F32 ? MOE_LIST_F32 : MOE_LIST))) return LCU_BAD_ARGUMENT;
    if (shared_up && (!shared_down || shared || !gated || !few || !packed_up || !packed_down || shared_ff <= 0 || shared_ff % 16)) return LCU_BAD_ARGUMENT;
    const int add = top == 1 && !gated;
    float *down_to = add ? out : y;
    if (!add && !y) return LCU_BAD_ARGUMENT;
    const int up_rows = gated ? 2 * ff : ff;                  // rows of an expert's first matrix
    const int kstep = type == LCU_BF16 ? 32 : 16;             // elements an expert's matrix takes
    auto elems = [&](int rows, int k, int packed) { return packed ? (size_t)((rows + 15) / 16 * 16) * ((k + kstep - 1) / kstep * kstep) : (size_t)rows * k; };
    const size_t up_stride = elems(up_rows, d, packed_up), down_stride = elems(d, ff, packed_down);
#define TYPED(GO, ...)                                                                                             \
    if (type == LCU_BF16) { if (packed) GO(bf16_t, true, __VA_ARGS__); else GO(bf16_t, false, __VA_ARGS__); }       \
    else { if (packed) GO(float, true, __VA_ARGS__); else GO(float, false, __VA_ARGS__); }                          \
    LCU_LAUNCH_CHECK()
    int *sorted = nullptr, *t_exp = nullptr, *t_beg = nullptr, *t_rows = nullptr, *n_tiles = nullptr;
    if (!ids) return LCU_BAD_ARGUMENT;
    if (tile_rows) {
        if (!ints || max_tiles <= 0) return LCU_BAD_ARGUMENT;
        sorted = ints;
        t_exp = ints + total;
        t_beg = t_exp + max_tiles;
        t_rows = t_beg + max_tiles;
        n_tiles = t_rows + max_tiles;
        moe_group_kernel<<<dim3(1), dim3(1024), 0, stream>>>(ids, total, experts + identity, sorted, t_exp, t_beg, t_rows, n_tiles, max_tiles, tile_rows, experts);
        LCU_LAUNCH_CHECK();
    }
    if (few) {
        // one more expert, the shared one: its activations lie behind the pairs' (act [total, ff], then [n, shared_ff]), its outputs too
        const int with = (tile_rows ? max_tiles : experts) + (shared_up ? 1 : 0), s_rows = 2 * shared_ff, wider = shared_up && s_rows > up_rows ? s_rows : up_rows;
        const size_t act_end = (size_t)total * ff;
        const dim3 block(256), gu((wider + 31) / 32, with), gd((d + 31) / 32, with);
        const int slots = total < experts ? total : experts;
        const dim3 su(gu.x, slots + (shared_up ? 1 : 0)), sd(gd.x, su.y);
        const bool up_slots = !tile_rows && moe_slots_take(n, top, experts, up_rows), down_slots = !tile_rows && moe_slots_take(n, top, experts, d);
#define UP_SLOTS(T, PACKED, MODE) moe_gemm_slots_kernel<T, MODE, PACKED><<<su, dim3(512), 0, stream>>>((const T *)h, d, (const T *)w_up, up_stride, up_rows, d, \
                                                ids, total, wts, (T *)act, nullptr, ff, top, 0, alpha, limit, experts, slots, \
                                                (const T *)h, (const T *)shared_up, s_rows, d, (T *)act + act_end, nullptr)
#define DOWN_SLOTS(T, PACKED, MODE) moe_gemm_slots_kernel<T, MODE, PACKED><<<sd, dim3(512), 0, stream>>>((const T *)act, ff, (const T *)w_down, down_stride, d, ff, \
                                                ids, total, wts, nullptr, down_to, d, top, add, 0.f, 0.f, experts, slots, \
                                                (const T *)act + act_end, (const T *)shared_down, d, shared_ff, nullptr, y + (size_t)total * d)
#define UP(T, PACKED, MODE) moe_gemm_few_kernel<T, MODE, PACKED><<<gu, block, 0, stream>>>((const T *)h, d, (const T *)w_up, up_stride, up_rows, d, \
                                                ids, total, wts, (T *)act, nullptr, ff, top, 0, alpha, limit, experts, \
                                                (const T *)h, (const T *)shared_up, s_rows, d, (T *)act + act_end, nullptr, sorted, t_exp, t_beg, t_rows, n_tiles, max_tiles)
#define DOWN(T, PACKED, MODE) moe_gemm_few_kernel<T, MODE, PACKED><<<gd, block, 0, stream>>>((const T *)act, ff, (const T *)w_down, down_stride, d, ff, \
                                                ids, total, wts, nullptr, down_to, d, top, add, 0.f, 0.f, experts, \
                                                (const T *)act + act_end, (const T *)shared_down, d, shared_ff, nullptr, y + (size_t)total * d, sorted, t_exp, t_beg, t_rows, n_tiles, max_tiles)
        int packed = packed_up;
        if (up_slots) {
            if (gated) { TYPED(UP_SLOTS, MOE_UP_GATED); } else { TYPED(UP_SLOTS, MOE_UP); }
        } else {
            if (gated) { TYPED(UP, MOE_UP_GATED); } else { TYPED(UP, MOE_UP); }
        }
        packed = packed_down;
        if (down_slots) { TYPED(DOWN_SLOTS, MOE_DOWN); } else { TYPED(DOWN, MOE_DOWN); }
#undef UP_SLOTS
#undef DOWN_SLOTS
#undef UP
#undef DOWN
    } else {
        // flat grids: the kernel shares them out over the dies itself
        const dim3 block(256), gu((max_tiles * ((up_rows + 127) / 128) + 7) / 8 * 8), gd((max_tiles * ((d + 127) / 128) + 7) / 8 * 8);
#define UP(T, PACKED, MODE) moe_gemm_many_kernel<T, MODE, PACKED><<<gu, block, 0, stream>>>((const T *)h, d, (const T *)w_up, up_stride, up_rows, d, \
                                                sorted, wts, t_exp, t_beg, t_rows, n_tiles, (T *)act, nullptr, ff, top, 0, alpha, limit)
#define DOWN(T, PACKED, MODE) moe_gemm_many_kernel<T, MODE, PACKED><<<gd, block, 0, stream>>>((const T *)act, ff, (const T *)w_down, down_stride, d, ff, \
                                                sorted, wts, t_exp, t_beg, t_rows, n_tiles, nullptr, down_to, d, top, add, 0.f, 0.f)
        int packed = packed_up;
        if (gated) { TYPED(UP, MOE_UP_GATED); } else { TYPED(UP, MOE_UP); }
        packed = packed_down;
        TYPED(DOWN, MOE_DOWN);
#undef UP
#undef DOWN
    }
#undef TYPED
    if (!add && !defer) {
        const PairSum p = {fresh ? nullptr : out, y, gated ? wts : nullptr, shared, shared_up ? y + (size_t)total * d : nullptr, shared_gate, identity ? ids : nullptr, h, top, experts};
        return lcu_moe_combine(out, &p, type, n, d, stream);
    }
    return LCU_OK;
}
