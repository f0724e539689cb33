// Y[M, N] = X[M, K] * W[N, K]^T for few rows (decoding: M <= 32), bfloat16 operands,
// 32-bit accumulation on the matrix cores.  The work is streaming W once from HBM, so
// the kernel is laid out around W's loads:
//
//   * a workgroup of 4 or 8 waves owns NT tiles of 16 output features (rows of W) and walks
//     the whole K: no sum crosses workgroups, results do not depend on the grid, and
//     the epilogue can be fused;
//   * K goes in macro-steps of 128; the waves take macro-steps in turn; in a macro-step
//     lane group g of a wave reads the 64 contiguous bytes k0 + 32g .. k0 + 32g + 31 of
//     its row as four 16-byte loads, one per matrix instruction (which k a slot of the
//     instruction holds is free, as long as W and X agree), so the four waves read 1 KB
//     of a row back to back;
//   * a wave keeps the loads of several macro-steps in flight while it multiplies one;
//   * v_mfma_f32_16x16x32_bf16 with A = W tile, B = X^T: the 16 columns are 16 tokens,
//     MT such tiles for up to 32 tokens (more rows go to gemm_mid.hip, which shares them through LDS).
//     X comes in by quads of lanes and is turned into the operands' order in registers (quad_rows.h).
// The waves' partial sums are added in LDS in a fixed order.
//
// One MI355X, packed weights out of memory, us a product (in brackets with X loaded in the operands' order, a cycle of a compute unit for every
// lane): 2048 x 2048 4.0 (4.2) at 1 row, 4.4 (4.8) at 8, 5.2 (6.2) at 16; 4096 x 4096 7.8 (8.3) at 8, 9.1 (10.7) at 16; 4096 x 14336 22.0 (22.6) at
// 1, 22.7 (25.3) at 8, 25.0 (32.9) at 16; SwiGLU of 28672 x 4096 41.1 (41.8) at 8, 42.0 (43.8) at 16.
//
// W may also be given packed (lcu_pack_weight / the wrapper's pack_weight): the 16 x 128 block
// of a tile and a macro-step lies in 4 KB of its own, ordered [j][lane][8] as the lanes load it,
// the blocks of a tile one after the other.  Then every load instruction of a wave reads 1 KB
// in one piece and a workgroup streams one contiguous run of memory, which HBM serves
// faster than pieces of 256 bytes out of 16 or 32 rows that lie kilobytes apart.
//
// Epilogues: store bfloat16; store float32 (logits); add into float32 (the residual
// stream); SwiGLU, where the workgroup's two tiles are the gate rows n and the up rows
// n + N/2 of one matrix and silu(gate) * up (or the limited form, gate_act.h) is stored.
//
// Grouped: W is several matrices of group_rows rows one above the other, and each multiplies rows of X of its own
// (group g reads X + g * x_group_stride): one product per head, or several projections of differently mixed rows, in
// one launch.  Their outputs may be multiplied by the sigmoid of a gate [M, N] on the way out.
#include <type_traits>
#include "common.h"
#include "lane_moves.h"
#include "gate_act.h"
#include "kv_layout.h"
#include "qkv_store.h"
#include "quad_rows.h"
#include "stream_steps.h"

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;

constexpr int SK_MAX_LDX = 1 << 24;
enum { EPI_BF16 = 0, EPI_F32 = 1, EPI_ADD_F32 = 2, EPI_SWIGLU = 3, EPI_ADD_NORM = 4, EPI_QKV_ROPE = 5, EPI_STREAMS = 6 };

// What two epilogues need beside Y, so that no kernel stands between a projection that ends
// a branch and the product that follows the next norm:
//   EPI_ADD_NORM: Y is the float32 residual stream and takes the product in; the new rows times
//     the norm's weight go to h_out as bfloat16, *not yet normalised*, and the workgroup's
//     share of each row's sum of squares goes to sumsq_out[row][workgroup].
//   EPI_STREAMS: the same for several residual streams side by side (Y [M, streams * N]): x_t <- sum_s mix[s, t] x_s + out_w[t] *
//     product, all t at once, and h_out and sumsq_out are made of sum_s read[s] x_s (read null: ones).  The rows of X may wait for
//     their normalisation.
//   row scale (any other epilogue, sumsq_in not null): the rows of X are such rows; a row of
//     the product is multiplied by rsqrt(sum of its shares / norm_width + eps) before the
//     epilogue (the normalisation is a factor per row, so it commutes with the product).
//   EPI_QKV_ROPE: W holds the q, k and v projections (rows q heads, k heads, v heads, head_dim
//     each).  A workgroup's two tiles are 16 dims of a head and the 16 dims head_dim/2 further,
//     the pairs of the rotation (half-split pairing over the whole head): the epilogue rotates q
//     and k by the token's position, writes q to q_out and k and v straight into the token's
//     place in the paged cache.  No rotation kernel runs after this product.
// The shares are added in a fixed order: no atomics, results do not depend on timing.
struct SkinnyExtra {
    const void *norm_w;        // [N] norm weight of EPI_ADD_NORM
    int norm_w_type;           // LCU_F32 or LCU_BF16
    bf16_t *h_out;             // [M, N] rows ldh apart
    int ldh;
    float *sumsq_out;          // [M][gridDim.x]
    const float *sumsq_in;     // [M][n_in] or null
    int n_in;
    int norm_width;
    float eps;
    QkvStore qkv;              // EPI_QKV_ROPE
    // EPI_ADD_NORM: what the product is multiplied by before it is added to the residual stream
    float res_scale;
    // EPI_SWIGLU: limit > 0 asks for the limited activation (gate_act.h)
    float act_alpha, act_limit;
    // EPI_STREAMS
    int streams;
    const float *mix, *out_w, *read;
    // grouped products (group_rows 0: one matrix, one X)
    int group_rows;
    size_t x_group_stride;
    const void *gate;          // [M, N] rows ldg apart, or null
    int gate_type, ldg;
};

__device__ __forceinline__ f32x4 mfma16(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// LOADS: loads of 128 k of the last tile's rows of X (quad_rows.h), fewer than four for up to eight of them; the tiles before take four.
template <int NT, int MT, int LOADS>
struct Frag {
    u32x4 w[NT][4];
    u32x4 x[MT][4];
};

// A weight is read once per product and never again before the caches have turned over: the loads of a packed
// weight are marked non-temporal, so that they do not displace what is used again (the rows, the next kernel's
// operands).  A kernel that only reads memory moves 6.2 to 6.4 TB/s of a 235 MB stretch with such loads and 5.7
// with ordinary ones.  Only where a load instruction of a wave takes whole 128-byte lines, as it does from a packed
// weight: from plain rows, where eight instructions share a line, such loads fetch the line again and again (the
// decode step of 8 requests took 5.5 ms with them and plain rows).
__device__ __forceinline__ u32x4 stream_load(const u32x4 *p) { return __builtin_nontemporal_load(p); }

// The lane's loads of macro-step s: W's k = 128 s + 32 grp + 8 j .. + 7 for j = 0..3; X as quad_rows.h says, through a buffer that ends with the
// last row's k (rows beyond it read zeros; WHOLE: K has no partial step), x_place the lane's place in its first four rows and x_four the bytes of four rows.
template <int NT, int MT, bool PACKED, int LOADS, bool WHOLE>
__device__ __forceinline__ void load_frag(Frag<NT, MT, LOADS> &f, const bf16_t *const (&wrow)[NT], __amdgpu_buffer_rsrc_t xb, uint32_t x_place,
                                          uint32_t x_four, int s, int lane, int K) {
    const int grp = lane >> 4, kb = 128 * s + 32 * grp;
    const u32x4 zero = u32x4{0u, 0u, 0u, 0u};
    if (WHOLE || 128 * (s + 1) <= K) {
        // packed: wrow is the lane's place in the tile's first block; blocks are 2048 elements,
        // the four loads of a block 512 apart
        const int w0 = PACKED ? 2048 * s : kb, wj = PACKED ? 512 : 8;
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                f.w[t][j] = PACKED ? stream_load((const u32x4 *)(wrow[t] + w0 + wj * j)) : *(const u32x4 *)(wrow[t] + w0 + wj * j);
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int i = 0; i < (m < MT - 1 ? 4 : LOADS); ++i)
                f.x[m][i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(xb, x_place + (4 * m + i) * x_four + 256u * s, 0, 0));
    } else {                                   // the last, partial macro-step (K is a multiple of 8)
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int j = 0; j < 4; ++j) f.w[t][j] = (kb + 8 * j + 8 <= K) ? *(const u32x4 *)(wrow[t] + kb + 8 * j) : zero;
        const bool in = 128 * s + quad_k(lane) + 8 <= K;         // (what lies behind a row's k may be NaN)
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int i = 0; i < (m < MT - 1 ? 4 : LOADS); ++i)
                f.x[m][i] = in ? __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(xb, x_place + (4 * m + i) * x_four + 256u * s, 0, 0)) : zero;
    }
}

template <int NT, int MT, int LOADS>
__device__ __forceinline__ void mul_frag(const Frag<NT, MT, LOADS> &f, f32x4 (&acc)[NT][MT]) {
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        u32x4 x[4];
        if (m < MT - 1) quad_operands<4>(f.x[m], x);
        else {
            u32x4 few[LOADS];
#pragma unroll
            for (int i = 0; i < LOADS; ++i) few[i] = f.x[m][i];
            quad_operands<LOADS>(few, x);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int t = 0; t < NT; ++t) acc[t][m] = mfma16(f.w[t][j], x[j], acc[t][m]);
    }
}

template <int NT, int MT, int EPI, int SK_WAVES, bool PACKED, int LOADS>
__global__ void __launch_bounds__(SK_WAVES *WAVE, SK_WAVES == 8 && NT * MT == 1 && LOADS <= 2 ? 4 : 1)
gemm_skinny_kernel(const bf16_t *__restrict__ X, int ldx, const bf16_t *__restrict__ W, int ldw, void *__restrict__ Y,
                   int ldy, int M, int N, int K, SkinnyExtra ex) {
    __shared__ float red[SK_WAVES][NT * MT * 4][WAVE];
    __shared__ float row_scale[16 * MT];
    const int lane = threadIdx.x & (WAVE - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const int l16 = lane & 15, grp = lane >> 4;
    // the rows of W of tile t: for SwiGLU tile 0 are gate rows, tile 1 the up rows N/2 further
    const int n_out = EPI == EPI_SWIGLU ? N / 2 : N;                 // width of Y
    // SwiGLU: the first NT/2 tiles are gate rows, the other NT/2 the up rows N/2 further
    const int n0 = blockIdx.x * 16 * (EPI == EPI_SWIGLU ? NT / 2 : NT);
    // q/k/v with rotation: workgroup b has, of head b / (head_dim/32), the dims 16 c .. and head_dim/2 + 16 c ..
    const int rope_head = EPI == EPI_QKV_ROPE ? blockIdx.x / (ex.qkv.head_dim / 32) : 0;
    const int rope_c = EPI == EPI_QKV_ROPE ? blockIdx.x % (ex.qkv.head_dim / 32) : 0;
    const bf16_t *wrow[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int half = t / (NT / 2 > 0 ? NT / 2 : 1);              // 0: gate tiles, 1: up tiles (SwiGLU)
        int row = EPI == EPI_SWIGLU ? n0 + 16 * (t % (NT / 2 > 0 ? NT / 2 : 1)) + l16 + half * n_out : n0 + 16 * t + l16;
        if (EPI == EPI_QKV_ROPE) row = rope_head * ex.qkv.head_dim + t * (ex.qkv.head_dim / 2) + 16 * rope_c + l16;
        const int limit = EPI == EPI_SWIGLU ? (half + 1) * n_out : N;
        row = row < limit ? row : limit - 1;                          // a row beyond the end is read, not stored
        wrow[t] = PACKED ? W + ((size_t)(row / 16) * (K / 128)) * 2048 + (size_t)lane * 8   // (the tile of the row)
                           : W + (size_t)row * ldw;
    }
    if (ex.group_rows > 0) X += (size_t)(n0 / ex.group_rows) * ex.x_group_stride;      // (a workgroup's rows lie in one group)
    const __amdgpu_buffer_rsrc_t xb = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t *>(X), 0, (uint32_t)((M - 1) * ldx + K) * 2u, 0x00020000);
    uint32_t x_place = (uint32_t)(quad_load_row(0, lane) * ldx + quad_k(lane)) * 2u;
    asm("" : "+v"(x_place));                    // (else every tile's place is multiplied out in front of the loop, a register each)
    const uint32_t x_four = 8u * ldx;
    const int col = quad_row(l16);              // the token of the tile that the lane's column of the products is
    f32x4 acc[NT][MT];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[t][m] = f32x4{0.f, 0.f, 0.f, 0.f};

    // The rows' factors, by the last wave before it starts on its share of K.  Lane group g adds
    // the g-th quarter of a row's shares, eight 16-byte loads in flight at a time (one load after
    // the other would hold the wave back for tens of microseconds); the quarters' sums are added
    // in the order of the shuffles.  Always the same order: no dependence on timing.
    if (EPI != EPI_ADD_NORM && ex.sumsq_in != nullptr && wave == SK_WAVES - 1) {
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const int tok = 16 * m + l16;
            const float *p = ex.sumsq_in + (size_t)(tok < M ? tok : 0) * ex.n_in;
            float ss = 0.f;
            if ((ex.n_in & 15) == 0) {
                const int q4 = ex.n_in / 16;                       // float4s in a quarter
                const f32x4 *p4 = (const f32x4 *)p + grp * q4;
                for (int i = 0; i < q4; i += 8) {
                    f32x4 v[8];
#pragma unroll
                    for (int e = 0; e < 8; ++e) v[e] = p4[i + e < q4 ? i + e : q4 - 1];
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        if (i + e < q4) ss += (v[e][0] + v[e][1]) + (v[e][2] + v[e][3]);
                }
            } else {
                for (int i = grp; i < ex.n_in; i += 4) ss += p[i];
            }
            ss += __shfl_xor(ss, 16, WAVE);
            ss += __shfl_xor(ss, 32, WAVE);
            if (grp == 0) row_scale[tok] = rsqrtf(ss / (float)ex.norm_width + ex.eps);
        }
    }

    // A ring of STAGES macro-steps in flight per wave: with few workgroups per compute unit
    // (small N) this is what keeps enough bytes on their way from HBM.  Packed rows go through it without a condition (stream_steps.h; with one the wave waited for the whole
    // ring once in STAGES steps): passes of the 8B shape, one request 7.10 -> 6.99 ms, eight 7.80 -> 7.68.  Four waves a SIMD, as before, for one tile of few rows (129 registers
    // otherwise).
    // Two tiles of rows with four of features: two as well while the second tile has up to eight rows (25 to 32 rows want the registers).  SwiGLU, us, 17 to 24 rows with two stages (with
    // one, and all eight loads of rows): 7168 x 8192 33.0 to 34.1 (37.2 to 38.1), 2048 x 6144 23.3 to 24.3 (27.0 to 27.4), 7680 x 16384 65.8 to 67.9 (74.8 to 75.2).
    constexpr int STAGES = NT * MT == 1 ? 4 : NT * MT == 2 ? 3 : NT * MT == 8 && SK_WAVES == 8 && LOADS == 4 ? 1 : 2;
    const int nsteps = (K + 127) / 128;
    Frag<NT, MT, LOADS> f[STAGES];
    if constexpr (PACKED) {                                            // (K is a multiple of 128)
        stream_steps<STAGES>(
            wave < nsteps ? (nsteps - 1 - wave) / SK_WAVES + 1 : 0,
            [&](int u, int i) { load_frag<NT, MT, true, LOADS, true>(f[u], wrow, xb, x_place, x_four, wave + i * SK_WAVES, lane, K); },
            [&](int u, int) { mul_frag<NT, MT, LOADS>(f[u], acc); });
    } else {
        int s = wave;
#pragma unroll
        for (int i = 0; i < STAGES; ++i)
            if (s + i * SK_WAVES < nsteps) load_frag<NT, MT, false, LOADS, false>(f[i], wrow, xb, x_place, x_four, s + i * SK_WAVES, lane, K);
        for (; s < nsteps; s += STAGES * SK_WAVES) {
#pragma unroll
            for (int i = 0; i < STAGES; ++i) {
                const int cur = s + i * SK_WAVES;
                if (cur < nsteps) {
                    mul_frag<NT, MT, LOADS>(f[i], acc);
                    if (cur + STAGES * SK_WAVES < nsteps)
                        load_frag<NT, MT, false, LOADS, false>(f[i], wrow, xb, x_place, x_four, cur + STAGES * SK_WAVES, lane, K);
                }
            }
        }
    }
    // ---- the waves' sums, added in the order 0, 1, 2, ...
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int r = 0; r < 4; ++r) red[wave][(t * MT + m) * 4 + r][lane] = acc[t][m][r];
    __syncthreads();
    if (wave != 0) return;
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int i = (t * MT + m) * 4 + r;
                float sum = red[0][i][lane];
#pragma unroll
                for (int w = 1; w < SK_WAVES; ++w) sum += red[w][i][lane];
                acc[t][m][r] = sum;
            }
    // ---- epilogue: the lane holds, per tile, features 4 grp + r of token 16 m + col
    if (EPI != EPI_ADD_NORM && ex.sumsq_in != nullptr) {
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const float rs = row_scale[16 * m + col];
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[t][m][r] *= rs;
        }
    }
    if (EPI == EPI_QKV_ROPE) {
        // the lane holds dims i = 16 c + 4 grp + r (tile 0) and i + head_dim/2 (tile 1) of token 16 m + col
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const int tok = 16 * m + col;
            if (tok >= M) continue;
            const float lo[4] = {acc[0][m][0], acc[0][m][1], acc[0][m][2], acc[0][m][3]}, hi[4] = {acc[NT - 1][m][0], acc[NT - 1][m][1], acc[NT - 1][m][2], acc[NT - 1][m][3]};
            qkv_store(ex.qkv, rope_head, tok, 16 * rope_c + 4 * grp, lo, hi);
        }
        return;
    }
    if (EPI == EPI_STREAMS) {
        constexpr int MOST = 8;
        const int S = ex.streams;
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const int tok = 16 * m + col;
            float ss = 0.f;
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const int c = n0 + 16 * t + 4 * grp;          // (N is a multiple of 4)
                if (tok >= M || c >= N) continue;
                float *res = (float *)Y + (size_t)tok * ldy + c;
                f32x4 xs[MOST], u = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int s = 0; s < MOST; ++s)
                    if (s < S) xs[s] = *(const f32x4 *)(res + (size_t)s * N);
#pragma unroll
                for (int to = 0; to < MOST; ++to) {
                    if (to >= S) break;
                    f32x4 n = acc[t][m] * ex.out_w[to];
#pragma unroll
                    for (int s = 0; s < MOST; ++s)
                        if (s < S) n += ex.mix[s * S + to] * xs[s];
                    *(f32x4 *)(res + (size_t)to * N) = n;
                    u += (ex.read ? ex.read[to] : 1.f) * n;
                }
                const f32x4 w = *(const f32x4 *)((const float *)ex.norm_w + c);
#pragma unroll
                for (int r = 0; r < 4; ++r) ss += u[r] * u[r];
                uint2 h;
                h.x = pack2_bf16(u[0] * w[0], u[1] * w[1]);
                h.y = pack2_bf16(u[2] * w[2], u[3] * w[3]);
                *(uint2 *)(ex.h_out + (size_t)tok * ex.ldh + c) = h;
            }
            ss += __shfl_xor(ss, 16, WAVE);               // every lane takes part: the others bring zero
            ss += __shfl_xor(ss, 32, WAVE);
            if (grp == 0 && tok < M) ex.sumsq_out[(size_t)tok * gridDim.x + blockIdx.x] = ss;
        }
        return;
    }
    if (EPI == EPI_ADD_NORM) {
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const int tok = 16 * m + col;
            float ss = 0.f;
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int n = n0 + 16 * t + 4 * grp + r;
                    if (tok >= M || n >= N) continue;
                    float *res = (float *)Y + (size_t)tok * ldy + n;
                    const float xn = fmaf(ex.res_scale, acc[t][m][r], *res);
                    *res = xn;
                    ss += xn * xn;
                    const float wn = ex.norm_w_type == LCU_F32 ? ((const float *)ex.norm_w)[n] : to_f32(((const bf16_t *)ex.norm_w)[n]);
                    ex.h_out[(size_t)tok * ex.ldh + n] = from_f32<bf16_t>(xn * wn);
                }
            ss += __shfl_xor(ss, 16, WAVE);               // every lane takes part: the others bring zero
            ss += __shfl_xor(ss, 32, WAVE);
            if (grp == 0 && tok < M) ex.sumsq_out[(size_t)tok * gridDim.x + blockIdx.x] = ss;
        }
        return;
    }
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        const int tok = 16 * m + col;
        if (tok >= M) continue;
        if (EPI == EPI_SWIGLU) {
#pragma unroll
            for (int t = 0; t < NT / 2; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int n = n0 + 16 * t + 4 * grp + r;
                    if (n >= n_out) continue;
                    const float gate = acc[t][m][r], up = acc[t + NT / 2][m][r];
                    ((bf16_t *)Y)[(size_t)tok * ldy + n] = from_f32<bf16_t>(gate_up_of(gate, up, ex.act_alpha, ex.act_limit));
                }
        } else {
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int n = n0 + 16 * t + 4 * grp + r;
                    if (n >= N) continue;
                    const size_t at = (size_t)tok * ldy + n;
                    if (EPI == EPI_BF16 && ex.gate != nullptr) {
                        const size_t ga = (size_t)tok * ex.ldg + n;
                        const float z = ex.gate_type == LCU_F32 ? ((const float *)ex.gate)[ga] : to_f32(((const bf16_t *)ex.gate)[ga]);
                        acc[t][m][r] *= 1.0f / (1.0f + expf(-z));
                    }
                    if (EPI == EPI_BF16) ((bf16_t *)Y)[at] = from_f32<bf16_t>(acc[t][m][r]);
                    else if (EPI == EPI_F32) ((float *)Y)[at] = acc[t][m][r];
                    else ((float *)Y)[at] += acc[t][m][r];
                }
        }
    }
}

// (a last tile of few rows takes fewer loads where it is the only tile or where that leaves registers for a second stage.  Plain matrices, us at 1, 4 and 8 rows with that and with
// four loads: 2048 x 2048 4.7, 4.7, 4.9 and 5.3, 5.3, 5.4, 14336 x 4096 24.4, 24.5, 26.2 and 27.5, 27.7, 28.8)
#define RUN(E, GRID, BLOCK)                                                            \
    do {                                                                               \
        if (packed) RUN_LOADS(E, GRID, BLOCK, true, MT == 1 || (NT * MT == 8 && WAVES == 8)); \
        else RUN_LOADS(E, GRID, BLOCK, false, MT == 1);                                \
    } while (0)
#define RUN_LOADS(E, GRID, BLOCK, PACKED, FEW)                                         \
    do {                                                                               \
        if constexpr (!(FEW)) RUN_AS(E, GRID, BLOCK, PACKED, 4);                       \
        else if (M - 16 * (MT - 1) <= 4) RUN_AS(E, GRID, BLOCK, PACKED, 1);            \
        else if (M - 16 * (MT - 1) <= 8) RUN_AS(E, GRID, BLOCK, PACKED, 2);            \
        else RUN_AS(E, GRID, BLOCK, PACKED, 4);                                        \
    } while (0)
#define RUN_AS(E, GRID, BLOCK, PACKED, LOADS)                                                                                \
    gemm_skinny_kernel<NT, MT, E, WAVES, PACKED, LOADS><<<GRID, BLOCK, 0, stream>>>((const bf16_t *)X, ldx, (const bf16_t *)W, ldw, Y, ldy, M, N, K, ex)

template <int NT, int MT, int WAVES>
static int launch_epi(const void *X, int ldx, const void *W, int ldw, void *Y, int ldy, int M, int N, int K, int epi,
                      int packed, const SkinnyExtra &ex, hipStream_t stream) {
    dim3 block(WAVES * WAVE);
    const dim3 grid((N + 16 * NT - 1) / (16 * NT));
#define GO(E)                                                                                                                      \
    do {                                                                                                                           \
        RUN(E, grid, block);                                                                                                       \
    } while (0)
    switch (epi) {
    case EPI_BF16: GO(EPI_BF16); break;
    case EPI_F32: GO(EPI_F32); break;
    case EPI_ADD_F32: GO(EPI_ADD_F32); break;
    case EPI_ADD_NORM:
        if constexpr (MT <= 2 && NT <= 2) { GO(EPI_ADD_NORM); break; }      // made for decoding: at most 32 rows
        return LCU_UNSUPPORTED;
    case EPI_STREAMS:
        if constexpr (MT <= 2 && NT <= 2) { GO(EPI_STREAMS); break; }
        return LCU_UNSUPPORTED;
    case EPI_QKV_ROPE:
        if constexpr (MT <= 2 && NT == 2) {
            const dim3 rgrid((ex.qkv.heads + 2 * ex.qkv.kv_heads) * (ex.qkv.head_dim / 32));
            RUN(EPI_QKV_ROPE, rgrid, block);
            break;
        }
        return LCU_UNSUPPORTED;
    default: return LCU_BAD_ARGUMENT;
    }
#undef GO
    LCU_LAUNCH_CHECK();
    return LCU_OK;
}

template <int NT, int MT, int WAVES>
static int launch_swiglu(const void *X, int ldx, const void *W, int ldw, void *Y, int ldy, int M, int N, int K,
                         int packed, const SkinnyExtra &ex, hipStream_t stream) {
    const int groups = (N / 2 + 8 * NT - 1) / (8 * NT);
    RUN(EPI_SWIGLU, dim3(groups), dim3(WAVES * WAVE));
    LCU_LAUNCH_CHECK();
    return LCU_OK;
}
#undef RUN
#undef RUN_LOADS

// X: [M, K] bfloat16 rows ldx apart; W: [N, K] bfloat16 rows ldw apart; Y: [M, N] rows ldy
// apart (for the SwiGLU epilogue [M, N/2]: W holds N/2 gate rows, then N/2 up rows).
// M <= 32; K, ldx and ldw multiples of 8 (16-byte loads); tiles: output tiles of 16
// features per workgroup (1, 2 or 4; more tiles reuse X more, fewer give more workgroups);
// waves: 4 or 8 waves share a workgroup's K.
static int skinny_bf16(const void *X, int ldx, const void *W, int ldw, void *Y, int ldy, int M, int N, int K, int epilogue,
                       int tiles, int waves, int packed, const SkinnyExtra &ex, hipStream_t stream) {
    if (M <= 0 || N <= 0) return LCU_OK;
    // a packed weight is whole blocks of 16 rows x 128 k (and for SwiGLU each half is)
    if (packed && (K % 128 || N % 16 || (epilogue == EPI_SWIGLU && N % 32))) return LCU_BAD_ARGUMENT;
    if (M > 32 || K <= 0 || K % 8 || ldx % 8 || ldw % 8 || ldx < K || ldw < K || ldx >= SK_MAX_LDX) return LCU_BAD_ARGUMENT;      // (a load's place in the rows is 32 bits)
    if (waves != 4 && waves != 8) return LCU_BAD_ARGUMENT;
    const int mt = (M + 15) / 16;
    if (epilogue == EPI_SWIGLU) {
        if (N % 2 || ldy < N / 2) return LCU_BAD_ARGUMENT;
        // tiles: gate and up tiles together (2: one of each, 4: two of each)
#define SW(NT_, MT_) return waves == 8 ? launch_swiglu<NT_, MT_, 8>(X, ldx, W, ldw, Y, ldy, M, N, K, packed, ex, stream) \
                                       : launch_swiglu<NT_, MT_, 4>(X, ldx, W, ldw, Y, ldy, M, N, K, packed, ex, stream)
        if (tiles == 4 && mt <= 2) {
            if (mt == 1) SW(4, 1);
            SW(4, 2);
        }
        if (mt == 1) SW(2, 1);
        SW(2, 2);
#undef SW
    }
    if (ldy < N) return LCU_BAD_ARGUMENT;
#define EP(NT_, MT_) return waves == 8 ? launch_epi<NT_, MT_, 8>(X, ldx, W, ldw, Y, ldy, M, N, K, epilogue, packed, ex, stream) \
                                       : launch_epi<NT_, MT_, 4>(X, ldx, W, ldw, Y, ldy, M, N, K, epilogue, packed, ex, stream)
#define PICK(NT_)          \
    if (mt == 1) EP(NT_, 1); \
    EP(NT_, 2);
    if (tiles == 1) { PICK(1) }
    if (tiles == 2) { PICK(2) }
    if (tiles == 4) { PICK(4) }
#undef PICK
#undef EP
    return LCU_BAD_ARGUMENT;
}

LCU_API int lcu_gemm_skinny_bf16(const void *X, int ldx, const void *W, int ldw, void *Y, int ldy, int M, int N, int K,
                                 int epilogue, int tiles, int waves, int w_packed, float act_alpha, float act_limit, hipStream_t stream) {
    if (epilogue == EPI_ADD_NORM || epilogue == EPI_STREAMS) return LCU_BAD_ARGUMENT;
    SkinnyExtra ex = {};
    ex.act_alpha = act_alpha; ex.act_limit = act_limit;
    return skinny_bf16(X, ldx, W, ldw, Y, ldy, M, N, K, epilogue, tiles, waves, w_packed, ex, stream);
}

// Grouped: rows g * group_rows .. of W multiply the rows X + g * x_group_stride (M rows ldx apart); Y [M, N] takes all groups
// side by side, bfloat16 or float32 (epilogue).  gate (bfloat16 output only; may be null): [M, N] rows ldg apart of
// gate_type, the product is multiplied by its sigmoid before it is rounded.  group_rows a multiple of 16 * tiles.
LCU_API int lcu_gemm_skinny_bf16_grouped(const void *X, int ldx, long long x_group_stride, const void *W, int ldw, int group_rows, void *Y,
                                         int ldy, int M, int N, int K, int epilogue, int tiles, int waves, int w_packed,
                                         const void *gate, int gate_type, int ldg, hipStream_t stream) {
    if ((epilogue != EPI_BF16 && epilogue != EPI_F32) || group_rows <= 0 || tiles <= 0 || group_rows % (16 * tiles) || N % group_rows ||
        x_group_stride < 0 || x_group_stride % 8)
        return LCU_BAD_ARGUMENT;
    if (gate && (epilogue != EPI_BF16 || ldg < N || (gate_type != LCU_F32 && gate_type != LCU_BF16))) return LCU_BAD_ARGUMENT;
    SkinnyExtra ex = {};
    ex.group_rows = group_rows; ex.x_group_stride = (size_t)x_group_stride;
    ex.gate = gate; ex.gate_type = gate_type; ex.ldg = ldg;
    return skinny_bf16(X, ldx, W, ldw, Y, ldy, M, N, K, epilogue, tiles, waves, w_packed, ex, stream);
}

// The product that ends a branch, the residual sum and the next norm's weight in one kernel:
// res[M, N] (float32, rows ldres apart) += res_scale * (X W^T); h_out[M, N] = bfloat16(res * norm_w), not yet
// normalised; sumsq_out[M][ceil(N / (16 tiles))] = each workgroup's share of the rows' sums of
// squares.  At most 32 rows, tiles 1 or 2.
LCU_API int lcu_gemm_skinny_bf16_add_norm(const void *X, int ldx, const void *W, int ldw, float *res, int ldres, int M, int N,
                                          int K, const void *norm_w, int norm_w_type, void *h_out, int ldh, float *sumsq_out,
                                          int sumsq_cols, int tiles, int waves, int w_packed, float res_scale, hipStream_t stream) {
    if (M > 32 || (tiles != 1 && tiles != 2) || !res || !norm_w || !h_out || !sumsq_out || ldh < N || ldres < N ||
        (norm_w_type != LCU_F32 && norm_w_type != LCU_BF16) || sumsq_cols != (N + 16 * tiles - 1) / (16 * tiles))
        return LCU_BAD_ARGUMENT;
    SkinnyExtra ex = {};
    ex.norm_w = norm_w; ex.norm_w_type = norm_w_type; ex.h_out = (bf16_t *)h_out; ex.ldh = ldh; ex.sumsq_out = sumsq_out;
    ex.res_scale = res_scale;
    return skinny_bf16(X, ldx, W, ldw, res, ldres, M, N, K, EPI_ADD_NORM, tiles, waves, w_packed, ex, stream);
}

// The same between several residual streams: x [M, streams * N] (float32, rows ldx_s apart, N a multiple of 4); mix [streams, streams]
// (from, to), out_w and read [streams] (read may be null), norm_w [N], all float32.  sumsq_in (may be null): the rows of X
// wait for their normalisation.
LCU_API int lcu_gemm_skinny_bf16_streams(const void *X, int ldx, const void *W, int ldw, float *x, int ldx_s, int streams, int M, int N, int K,
                                         const float *mix, const float *out_w, const float *read, const float *norm_w, void *h_out, int ldh,
                                         float *sumsq_out, int sumsq_cols, int tiles, int waves, int w_packed, const float *sumsq_in, int n_in,
                                         int norm_width, float eps, hipStream_t stream) {
    if (M > 32 || (tiles != 1 && tiles != 2) || !x || !mix || !out_w || !norm_w || !h_out || !sumsq_out || streams < 1 || streams > 8 || N % 4 ||
        ldh < N || ldh % 4 || ldx_s < streams * N || ldx_s % 4 || (uintptr_t)x % 16 || (uintptr_t)norm_w % 16 || (uintptr_t)h_out % 8 ||
        sumsq_cols != (N + 16 * tiles - 1) / (16 * tiles) || (sumsq_in && (n_in <= 0 || norm_width <= 0)))
        return LCU_BAD_ARGUMENT;
    SkinnyExtra ex = {};
    ex.norm_w = norm_w; ex.norm_w_type = LCU_F32; ex.h_out = (bf16_t *)h_out; ex.ldh = ldh; ex.sumsq_out = sumsq_out;
    ex.streams = streams; ex.mix = mix; ex.out_w = out_w; ex.read = read;
    ex.sumsq_in = sumsq_in; ex.n_in = n_in; ex.norm_width = norm_width; ex.eps = eps;
    return skinny_bf16(X, ldx, W, ldw, x, ldx_s, M, N, K, EPI_STREAMS, tiles, waves, w_packed, ex, stream);
}

// A product whose rows of X wait for their normalisation: row i of the product is multiplied by
// rsqrt(sum(sumsq_in[i][0 .. n_in)) / norm_width + eps) before the epilogue (not EPI_ADD_NORM).
LCU_API int lcu_gemm_skinny_bf16_scaled(const void *X, int ldx, const void *W, int ldw, void *Y, int ldy, int M, int N, int K,
                                        int epilogue, int tiles, int waves, int w_packed, const float *sumsq_in, int n_in,
                                        int norm_width, float eps, float act_alpha, float act_limit, hipStream_t stream) {
    if (epilogue == EPI_ADD_NORM || epilogue == EPI_STREAMS || !sumsq_in || n_in <= 0 || norm_width <= 0) return LCU_BAD_ARGUMENT;
    SkinnyExtra ex = {};
    ex.sumsq_in = sumsq_in; ex.n_in = n_in; ex.norm_width = norm_width; ex.eps = eps;
    ex.act_alpha = act_alpha; ex.act_limit = act_limit;
    return skinny_bf16(X, ldx, W, ldw, Y, ldy, M, N, K, epilogue, tiles, waves, w_packed, ex, stream);
}


// The q, k and v projections with the rotation and the cache write in the epilogue.  W: [(heads +
// 2 kv_heads) * head_dim, K] (q heads, then k heads, then v heads).  q_out: [M, heads * head_dim]
// rows ldq apart takes the rotated queries; the rotated keys and the values go to cache (this
// layer's pages, laid out as kv_layout.h says) at slots[m] (page * page_size + place; -1: nothing
// is stored).  cos_t, sin_t: [max_pos, head_dim / 2] float32; pairs are (i, i + head_dim / 2).
// At most 32 rows; head_dim a multiple of 32.  sumsq_in (may be null): the rows of X wait for
// their normalisation, as in lcu_gemm_skinny_bf16_scaled.
LCU_API int lcu_gemm_skinny_bf16_qkv_rope(const void *X, int ldx, const void *W, int ldw, int M, int K, void *q_out, int ldq,
                                          const int *positions, const int *slots, const float *cos_t, const float *sin_t,
                                          int max_pos, void *cache, int heads, int kv_heads, int head_dim, int page,
                                          int waves, int w_packed, const float *sumsq_in, int n_in, int norm_width, float eps,
                                          hipStream_t stream) {
    if (M <= 0) return LCU_OK;
    if (M > 32 || heads <= 0 || kv_heads <= 0 || head_dim <= 0 || head_dim % 32 || page <= 0 || page % 8 || !q_out ||
        !positions || !cos_t || !sin_t || max_pos <= 0 || !cache || ldq < heads * head_dim ||
        (sumsq_in && (n_in <= 0 || norm_width <= 0)))
        return LCU_BAD_ARGUMENT;
    SkinnyExtra ex = {};
    ex.sumsq_in = sumsq_in; ex.n_in = n_in; ex.norm_width = norm_width; ex.eps = eps;
    ex.qkv = {positions, slots, cos_t, sin_t, max_pos, (bf16_t *)cache, (bf16_t *)q_out, ldq, heads, kv_heads, head_dim, page};
    const int N = (heads + 2 * kv_heads) * head_dim;
    return skinny_bf16(X, ldx, W, ldw, q_out, N, M, N, K, EPI_QKV_ROPE, 2, waves, w_packed, ex, stream);
}


// ============================================================================ float32
// The same weight-streaming layout for float32 operands, with v_mfma_f32_16x16x4_f32: a true
// 32-bit matrix product (32-bit multiplies and adds; no reduced-precision mode).  A lane's
// 16-byte load holds four k of its row, one per instruction, and the four lane groups' loads of a row lie side by side.  K goes in
// macro-steps of 64; the
// waves of a workgroup take macro-steps in turn and their sums are added in a fixed order, so
// a token's result depends on K and the number of waves only: not on M, not on which tile of
// 16 or 64 tokens (grid.y) it is in, not on the other tokens.
//
// The products that begin and end a branch of a 32-bit model do more, so that no norm or activation kernel runs between them: the
// rows may wait for their normalisation (sumsq_in), the result may go into the residual stream, with the next norm's weight on its
// way out (norm_w), and gate and up rows may meet in SwiGLU (PAIR: the matrix tile's sixteen rows are eight gate rows and the eight up rows
// that meet them, so that there are as many workgroups as without).  What
// bounds it at few tokens is latency (a launch, one round of loads, 0.9 us of matrix instructions), not the matrix: us at 2 tokens, matrices out of
// memory, 1024 x 1024 4.5, SwiGLU of 2816 x 1024 5.4; 32000 x 1024 25 (5.2 TB/s).  At 250 tokens 1024 x 1024 10.3, 2048 x 2048 31.5.  With both operands loaded
// in the operands' order (a cycle a lane, quad_rows.h) and a condition of the lanes' at every load they were 5.3, 5.9, 31.5, 14.9 and 49.3; with the first of the two mended 5.1, 6.1, 26.9, 11.4 and
// 34.1 (and longer than before it where K is no multiple of 64: 4096 x 1000 at 1 row 5.7, 6.4, now 5.7).  Rows that begin between lines and are short remain: 512 x 272 2.9, now 3.1.
constexpr int F32_WAVES = 8, COMPUTE_UNITS = 256;

struct F32Extra {
    int accumulate;
    float scale;                                             // of the product before it is added (accumulate, norm_w)
    const float *sumsq_in; int n_in, norm_width; float eps;  // null, or [M, n_in] shares of the rows' sums of squares
    const float *norm_w; float *h_out; int ldh; float *sumsq_out;      // null, or: Y += ..., h_out = Y * norm_w, sumsq_out [M, N / 16 rounded up]
    float act_alpha, act_limit;
};

// Both operands come in by quads of lanes (quad_rows.h, four k where bfloat16 has eight): W's load i brings lane (g, a, b) row 4 a + i, so that
// the operands' rows are in order, X's row 4 i + a, so that few rows take fewer loads; operand j then holds k = 64 s + 16 g + 4 j .. of its row.
// PAIR: SwiGLU; SCALED: with sumsq_in; ADDS: accumulate or norm_w; TWO: sixteen rows in 128 registers, for grids of more workgroups than compute units
template <int MT, bool PAIR, bool SCALED, bool ADDS, int LOADS, bool TWO = false>
__global__ void __launch_bounds__(F32_WAVES *WAVE, MT == 1 && (LOADS < 4 || TWO) ? 4 : 2)      // (up to eight rows, or TWO: two workgroups a compute unit)
gemm_skinny_f32_kernel(const float *__restrict__ X, int ldx, const float *__restrict__ W, int ldw, float *__restrict__ Y,
                       int ldy, int M, int N, int K, F32Extra ex) {
    __shared__ f32x4 red[F32_WAVES][MT][WAVE];
    __shared__ float factor[16 * MT];
    const int lane = threadIdx.x & (WAVE - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const int l16 = lane & 15, grp = lane >> 4, col = quad_row(l16);      // (the token of the tile that the lane's column is)
    const int n0 = blockIdx.x * (PAIR ? 8 : 16), m0 = blockIdx.y * 16 * MT;
    // (a row beyond the end is read, not stored)
    const float *wrow[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int r = 4 * ((lane >> 2) & 3) + i;
        wrow[i] = W + (size_t)(PAIR ? min(n0 + (r & 7), N - 1) + (r < 8 ? 0 : N) : min(n0 + r, N - 1)) * ldw;
    }
    // X's rows from the workgroup's first on, up to the last one's k: rows beyond it read zeros
    const __amdgpu_buffer_rsrc_t xb = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(X + (size_t)m0 * ldx), 0,
                                                                       (uint32_t)(min(M - 1 - m0, 16 * MT - 1) * ldx + K) * 4u, 0x00020000);
    uint32_t x_place = (uint32_t)(quad_load_row(0, lane) * ldx + 16 * (lane >> 4) + 4 * (lane & 3)) * 4u;
    asm("" : "+v"(x_place));                                 // (else every tile's place is multiplied out in front of the loop, a register each)
    const uint32_t x_four = 16u * ldx;
    f32x4 acc[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[m] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int nsteps = (K + 63) / 64;
    // a wave stores sixteen tokens in the end; what it adds to, and the norm's weights, are on their way meanwhile
    const int tok = m0 + 16 * wave + col;
    float old[4] = {}, nw[4] = {};
    if (ADDS && wave < MT) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int n = n0 + 4 * grp + r;
            if (tok < M && n < N) {
                old[r] = Y[(size_t)tok * ldy + n];
                if (ex.norm_w) nw[r] = ex.norm_w[n];
            }
        }
    }
    // macro-steps whose loads are on their way: of the matrix two, of up to eight rows two, of more rows a tile's next when it is used.  Every load is issued under
    // no condition of a lane's, with a place that exists, and what lies beyond K is taken out when it is used: with the condition at the load the ring's
    // waits were for everything on its way
    constexpr int ROWS_AHEAD = LOADS < 4 ? 2 : 1, AHEAD = 2;
    quad_u32x4 w[AHEAD][4], x[ROWS_AHEAD][MT][LOADS];
    const int k_lane = 16 * grp + 4 * (lane & 3);            // (K is a multiple of 4)
    auto load_w = [&](int u, int s) {
        const int k = min(64 * s + k_lane, K - 4);
#pragma unroll
        for (int i = 0; i < 4; ++i) w[u][i] = *(const quad_u32x4 *)(wrow[i] + k);
    };
    auto load_x = [&](int u, int m, int s) {
#pragma unroll
        for (int i = 0; i < LOADS; ++i) x[u][m][i] = __builtin_bit_cast(quad_u32x4, __builtin_amdgcn_raw_buffer_load_b128(xb, x_place + (4 * m + i) * x_four + 256u * s, 0, 0));
    };
    auto load_rows = [&](int u, int s) {
#pragma unroll
        for (int m = 0; m < MT; ++m) load_x(u, m, s);
    };
    // operand j: k = 64 s + 16 grp + 4 j ..
    auto within_k = [&](quad_u32x4 (&v)[4], int s) {
        if (64 * s + 64 <= K) return;
        asm volatile("");                                    // (a branch, no selection where there is nothing to take out)
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = 64 * s + 16 * grp + 4 * j + 4 <= K ? v[j] : quad_u32x4{0u, 0u, 0u, 0u};
    };
    // macro-step s out of w[U]; MORE_W, MORE_X: the loads that take its registers are asked for
    auto step = [&](auto U, int s, auto MORE_W, auto MORE_X) {
        constexpr int u = decltype(U)::value, ux = u % ROWS_AHEAD;
        quad_u32x4 wt[4];
        quad_operands<4, TWO>(w[u], wt);
        within_k(wt, s);
        if constexpr (decltype(MORE_W)::value) load_w(u, s + AHEAD * F32_WAVES);
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            quad_u32x4 xt[4];
            quad_operands<LOADS, TWO>(x[ux][m], xt);
            within_k(xt, s);
            if constexpr (decltype(MORE_X)::value) load_x(ux, m, s + ROWS_AHEAD * F32_WAVES);
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    acc[m] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(wt[j][e]), __uint_as_float(xt[j][e]), acc[m], 0, 0, 0);
        }
    };
    auto factors = [&]() {
        if constexpr (SCALED) {
            for (int r = wave; r < 16 * MT && m0 + r < M; r += F32_WAVES) {
                float t = 0.f;
                for (int i = lane; i < ex.n_in; i += WAVE) t += ex.sumsq_in[(size_t)(m0 + r) * ex.n_in + i];
                t = wave_sum_in_place(t);
                if (lane == 0) factor[r] = rsqrtf(t / (float)ex.norm_width + ex.eps);
            }
        }
    };
    constexpr std::integral_constant<int, 0> at0;
    constexpr std::integral_constant<int, 1> at1;
    constexpr std::true_type more;
    constexpr std::false_type last;
    constexpr std::bool_constant<ROWS_AHEAD == 1> rows_more;
    int s = wave, left = (nsteps - wave + F32_WAVES - 1) / F32_WAVES;      // the wave's macro-steps
    if (left >= 2) {
        load_w(0, s);
        load_rows(0, s);
        load_w(1, s + F32_WAVES);
        if constexpr (ROWS_AHEAD == 2) load_rows(1, s + F32_WAVES);
        factors();
        for (; left >= 4; left -= 2, s += 2 * F32_WAVES) {
            step(at0, s, more, more);
            step(at1, s + F32_WAVES, more, more);
        }
        if (left == 3) {
            step(at0, s, more, more);
            step(at1, s + F32_WAVES, last, rows_more);
            step(at0, s + 2 * F32_WAVES, last, last);
        } else {
            step(at0, s, last, rows_more);
            step(at1, s + F32_WAVES, last, last);
        }
    } else {
        if (left > 0) {
            load_w(0, s);
            load_rows(0, s);
        }
        factors();
        if (left > 0) step(at0, s, last, last);
    }
    asm volatile("s_nop 3" : "+v"(acc[MT - 1]));             // the last matrix instruction's wait, which the compiler leaves a state short behind the branches
#pragma unroll
    for (int m = 0; m < MT; ++m) red[wave][m][lane] = acc[m];
    __syncthreads();
    if (wave >= MT) return;
    f32x4 sum = red[0][wave][lane];
#pragma unroll
    for (int w = 1; w < F32_WAVES; ++w) sum += red[w][wave][lane];
    if constexpr (SCALED) sum *= factor[16 * wave + col];
    if constexpr (PAIR) {                                    // the up rows' sums are 32 lanes further
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const unsigned u = __float_as_uint(sum[r]);
            const float up = __uint_as_float(__builtin_amdgcn_permlane32_swap(u, u, false, false)[1]);
            const int n = n0 + 4 * grp + r;
            if (grp < 2 && tok < M && n < N) Y[(size_t)tok * ldy + n] = gate_up_of(sum[r], up, ex.act_alpha, ex.act_limit);
        }
        return;
    }
    float ss = 0.f;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int n = n0 + 4 * grp + r;
        if (tok >= M || n >= N) continue;
        const float v = ADDS ? old[r] + ex.scale * sum[r] : sum[r];
        Y[(size_t)tok * ldy + n] = v;
        if (ADDS && ex.norm_w) {
            ex.h_out[(size_t)tok * ex.ldh + n] = v * nw[r];
            ss += v * v;
        }
    }
    if (ADDS && ex.norm_w) {                                 // every lane takes part: the others bring zero
        ss += __shfl_xor(ss, 16, WAVE);
        ss += __shfl_xor(ss, 32, WAVE);
        if (grp == 0 && tok < M) ex.sumsq_out[(size_t)tok * gridDim.x + blockIdx.x] = ss;
    }
}

// X: [M, K] float32, W: [N, K] float32, Y: [M, N] float32 (accumulate: Y += scale X W^T).  Any M
// (tiles of 16 or 64 tokens; W is read once per tile); K, ldx, ldw multiples of 4, X and W 16-byte aligned.
// swiglu: W holds N gate rows, then N up rows.  sumsq_in: null, or [M, n_in] shares of the rows' sums of squares: the product's rows are
// multiplied by rsqrt(sum / norm_width + eps).  norm_w: null, or [N]: Y += scale X W^T, h_out [M, ldh] = Y norm_w, sumsq_out [M, ceil(N / 16)] the
// shares of the new rows' sums of squares.
LCU_API int lcu_gemm_skinny_f32(const float *X, int ldx, const float *W, int ldw, float *Y, int ldy, int M, int N,
                                int K, int accumulate, float scale, int swiglu, const float *sumsq_in, int n_in, int norm_width, float eps,
                                const float *norm_w, float *h_out, int ldh, float *sumsq_out, float act_alpha, float act_limit, hipStream_t stream) {
    if (M <= 0 || N <= 0) return LCU_OK;
    if (K <= 0 || K % 4 || ldx % 4 || ldw % 4 || ldx < K || ldw < K || ldy < N || ldx >= SK_MAX_LDX) return LCU_BAD_ARGUMENT;
    if ((sumsq_in && (n_in <= 0 || norm_width <= 0)) || (norm_w && (!h_out || !sumsq_out || ldh < N || swiglu)) || (swiglu && accumulate))
        return LCU_BAD_ARGUMENT;
    F32Extra ex = {accumulate, scale, sumsq_in, n_in, norm_width, eps, norm_w, h_out, ldh, sumsq_out, act_alpha, act_limit};
    // 16 tokens a workgroup, each of which reads its rows of W (from the L2 caches, but for the first), while the matrix instructions are
    // what takes the time: up to 32 tokens, and up to three workgroups a compute unit.  One MI355X, us with 16 / 64 tokens a
    // workgroup: 1024 x 1024 at 62 tokens 6.1 / 10.4, at 128 8.1 / 10.5, at 250 (1,024 workgroups) 13.8 / 10.8; 1536 x 1024 at 128 (768) 11.4 / 11.4; SwiGLU of
    // 2816 x 1024 at 62 (704) 12.1 / 11.8; 32000 x 1024 at 62 96 / 83, at 32 58 / 81; 2048 x 2048 at 62 (512) 14.5 / 18.3, at 128 (1,024) 22.8 / 18.8.
    const int rows = M <= 32 || ((N + 15) / 16) * ((M + 15) / 16) <= 768 ? 16 : 64;
    const int tiles = (M + rows - 1) / rows;
    if (tiles > 65535) return LCU_BAD_ARGUMENT;
    const dim3 grid(swiglu ? (N + 7) / 8 : (N + 15) / 16, tiles), block(F32_WAVES * WAVE);
    // What a product does besides is known when it is compiled: a form that looks at F32Extra for it, behind the loads that are on their way, took
    // 4.9 us for two rows of 1024 x 1024 with the matrix in the caches and 2.5 for 64 x 64, now 4.6 and 2.3.
#define GO(MT, PAIR, SCALED, ADDS, LOADS, TWO) gemm_skinny_f32_kernel<MT, PAIR, SCALED, ADDS, LOADS, TWO><<<grid, block, 0, stream>>>(X, ldx, W, ldw, Y, ldy, M, N, K, ex)
#define ROWS(MT, PAIR, ADDS, LOADS, TWO) do { if (sumsq_in) GO(MT, PAIR, true, ADDS, LOADS, TWO); else GO(MT, PAIR, false, ADDS, LOADS, TWO); } while (0)
#define FORMS(MT, LOADS, TWO) do { if (swiglu) ROWS(MT, true, false, LOADS, TWO); else if (accumulate || norm_w) ROWS(MT, false, true, LOADS, false); else ROWS(MT, false, false, LOADS, TWO); } while (0)
    // Two workgroups a compute unit where there are more than compute units; registers to spare where not.  us, two and one: 32000 x 1024 at 9 / 16 / 32 rows 28.7, 30.5, 51.3 and 34.8, 36.3, 61.4,
    // 520 x 272 at 128 (264 workgroups) 4.8 and 5.7; 1024 x 1024 at 9 / 16 (64) 5.7, 5.8 and 5.2, 5.2.  (What it adds to leaves no registers for it.)
    const bool two = (long long)grid.x * grid.y > COMPUTE_UNITS;
    if (rows > 16) FORMS(4, 4, false);
    else if (M <= 4) FORMS(1, 1, false);
    else if (M <= 8) FORMS(1, 2, false);
    else if (two) FORMS(1, 4, true);
    else FORMS(1, 4, false);
#undef FORMS
#undef ROWS
#undef GO
    LCU_LAUNCH_CHECK();
    return LCU_OK;
}
