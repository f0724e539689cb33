// Y[M, N] = X[M, K] * W[N, K]^T for up to 64 rows and weights of some tens of megabytes at most, bfloat16 operands, 32-bit sums.
//
// The weight-streaming kernel (gemm_skinny.hip) ends at 32 rows, the one that shares the rows through LDS (gemm_mid.hip) wants a weight of
// many features; a layer of width 2048 has products of 2 to 8 thousand features, 8 to 34 MB, which take 2 to 6 us out of memory, and the
// time goes into latency and idle compute units.  Here a workgroup takes 16 or 32 features (for SwiGLU 16 gate rows and the 16 up rows
// that meet them) and all rows; its eight waves share out K, a wave has all or most of its loads on their way at once, and the eight
// partial sums are added through LDS in a fixed order.  W is streamed once (packed as gemm_skinny.hip describes it: 4 KB for 16 rows x
// 128 k; whole lines, non-temporal); every workgroup reads all of X, out of the L2 caches: N / 32 times M K elements, which is why the
// rows and features end where they do.
//
// One MI355X, weights out of memory, beside the weight-streaming kernel, the row-sharing one (its sums in planes) and the library's, us a product
// (graph of products one after the other); in brackets as it was with the rows loaded in the operand's order (quad_rows.h says what that costs) and two
// macro-steps of them ahead of the second step's weights: 2048 x 2048: 4.4 (4.9) / 4.4 / - / 8.1 at 8 rows, 5.9 (7.3) / 8.2 / 5.4 / 11.4 at 32, 8.3
// (11.3) / - / 7.0 / 11.7 at 64; 8192 x 2048: 7.9 (8.1) / 8.1 / - / 12.9 at 8, 9.5 (10.0) / 11.3 / 10.2 / 13.2 at 32; 4096 x 4096: 8.6 (9.1) / 9.1 / - / - at
// 16, 10.7 (12.2) / 14.4 / 10.5 / 13.2 at 32, 14.7 (19.9) / - / 13.5 / 15.3 at 64; SwiGLU of 5632 x 2048: 7.1 (7.4) / 10.3 / - / - at 8, 8.8 (10.1) / 14.5 / 8.8 / 12.4
// (and the activation) at 32, 11.0 (16.6) / - / 16.2 / 13.0 at 64.  Bound by latency up to 16 rows; beyond, every 16 rows at K = 2048 are 1.1 us, half of it the
// operands' transposition, a quarter the way from the L2 caches.  Groups with a gate (a latent's heads): 16 of 128 x 512 2.9 / 3.1 / - / - at 8 rows, 3.4 / 3.9 / -
// / 8.6 at 32, 4.4 / - / - / 8.9 at 64.
//
// Groups: X is [groups][M, K], group g's rows x_group elements further, and multiplies the rows g * N / groups .. of W.
#include "common.h"
#include "gate_act.h"
#include "lane_moves.h"
#include "qkv_store.h"
#include "quad_rows.h"

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;

enum { GW_EPI_BF16 = 0, GW_EPI_F32 = 1, GW_EPI_SWIGLU = 2, GW_EPI_GATED = 3, GW_EPI_QKV = 4 };     // GATED: bf16, times sigmoid(gate); QKV: q, k and v, rotated and put where they belong

constexpr int GW_WAVES = 8, GW_MAX_ROWS = 64, GW_MAX_LDX = 1 << 24;

// NT: tiles of 16 features a workgroup; MT: tiles of 16 rows; LOADS: loads of 128 k of a tile's rows (quad_rows.h; fewer than four with one tile).
template <int NT, int MT, int EPI, int LOADS = 4>
__global__ void __launch_bounds__(GW_WAVES *WAVE)
gemm_wavek_kernel(const bf16_t *__restrict__ X, int ldx, size_t x_group, int group_tiles, const bf16_t *__restrict__ W, void *__restrict__ Y,
                  int ldy, const bf16_t *__restrict__ gate, int ldg, int M, int N, int K, const float *__restrict__ sumsq, int n_in,
                  int norm_width, float eps, float alpha, float limit, QkvStore store) {
    constexpr int AHEAD = 2;                         // macro-steps (128 k) whose weights are on their way; a tile's next rows are when it is used
    __shared__ f32x4 red[GW_WAVES][NT * MT][WAVE];
    __shared__ float factor[16 * MT];
    const int waves = blockDim.x >> 6;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), g = lane >> 4, l16 = lane & 15;
    const int macros = K / 128, per = (macros + waves - 1) / waves, m0 = min(macros, wave * per), m1 = min(macros, m0 + per);
    static_assert(LOADS == 4 || MT == 1, "few rows are one tile");
    // q, k, v: a rotation pairs dim i of a head with dim i + head_dim / 2: sixteen of the one and sixteen of the other
    const int per_head = EPI == GW_EPI_QKV ? store.head_dim / 32 : 1, qkv_head = EPI == GW_EPI_QKV ? blockIdx.x / per_head : 0, qkv_c = blockIdx.x - qkv_head * per_head;
    const bf16_t *wp[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) {
        int tile = EPI == GW_EPI_SWIGLU ? blockIdx.x + n * (N / 32) : min((int)blockIdx.x * NT + n, N / 16 - 1);
        if (EPI == GW_EPI_QKV) tile = qkv_head * 2 * per_head + qkv_c + n * per_head;
        wp[n] = W + (size_t)tile * 16 * K + lane * 8;
    }
    X += (size_t)(blockIdx.x * NT / group_tiles) * x_group;
    // a buffer that ends with the last row's k: rows beyond it read zeros, and a load's address is one register for all tiles
    const __amdgpu_buffer_rsrc_t xb = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t *>(X), 0, (uint32_t)((M - 1) * ldx + K) * 2u, 0x00020000);
    uint32_t place = (uint32_t)(quad_load_row(0, lane) * ldx + quad_k(lane)) * 2u;
    asm("" : "+v"(place));                           // (else every tile's place is multiplied out in front of the loop, a register each)
    const uint32_t four = 8u * ldx;
    f32x4 acc[NT][MT];
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[n][m] = f32x4{0.f, 0.f, 0.f, 0.f};
    u32x4 a[AHEAD][NT][4], b[MT][LOADS];
    auto fetch_w = [&](int u, int s) {
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
            for (int j = 0; j < 4; ++j) a[u][n][j] = __builtin_nontemporal_load((const u32x4 *)(wp[n] + (size_t)s * 2048 + 512 * j));
    };
    auto fetch_x = [&](int m, int s) {
#pragma unroll
        for (int i = 0; i < LOADS; ++i)
            b[m][i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(xb, place + (4 * m + i) * four + 256u * s, 0, 0));
    };
    auto multiply = [&](int u, int m) {
        u32x4 x[4];
        quad_operands<LOADS>(b[m], x);
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int n = 0; n < NT; ++n)
                acc[n][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a[u][n][j]), __builtin_bit_cast(bf16x8, x[j]), acc[n][m], 0, 0, 0);
    };
    // the last matrix instructions' wait, which the compiler leaves a state short behind the branches of the loop
    auto wait_for_sums = [&]() {
#pragma unroll
        for (int n = 0; n < NT; ++n) asm volatile("s_nop 3" : "+v"(acc[n][MT - 1]));
    };
#pragma unroll
    for (int u = 0; u < AHEAD; ++u)
        if (m0 + u < m1) fetch_w(u, m0 + u);
    if (m0 < m1) {
#pragma unroll
        for (int m = 0; m < MT; ++m) fetch_x(m, m0);
    }
    if (sumsq) {                                     // the rows wait for their normalisation: a factor each, from its shares added in a fixed order
        for (int r = wave; r < 16 * MT; r += waves) {
            float t = 0.f;
            for (int i = lane; i < n_in; i += WAVE) t += sumsq[(size_t)min(r, M - 1) * n_in + i];
            t = wave_sum_in_place(t);
            if (lane == 0) factor[r] = rsqrtf(t / (float)norm_width + eps);
        }
    }
    for (int s = m0; s < m1; s += AHEAD) {
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) {
            if (s + u >= m1) break;
            if (s + u + 1 < m1) {
#pragma unroll
                for (int m = 0; m < MT; ++m) {
                    multiply(u, m);
                    fetch_x(m, s + u + 1);
                }
                wait_for_sums();
                if (s + u + AHEAD < m1) fetch_w(u, s + u + AHEAD);
            } else {
#pragma unroll
                for (int m = 0; m < MT; ++m) multiply(u, m);
                wait_for_sums();
            }
        }
    }
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int m = 0; m < MT; ++m) red[wave][n * MT + m][lane] = acc[n][m];
    __syncthreads();
    auto total = [&](int t) {
        f32x4 v = red[0][t][lane];
        for (int w = 1; w < waves; ++w) v += red[w][t][lane];
        return sumsq ? v * factor[16 * (t % MT) + quad_row(l16)] : v;
    };
    // a wave stores a tile: four neighbouring features of a row a lane
    for (int t = wave; t < (EPI == GW_EPI_SWIGLU || EPI == GW_EPI_QKV ? MT : NT * MT); t += waves) {
        if constexpr (EPI == GW_EPI_SWIGLU) {
            const int row = 16 * t + quad_row(l16);
            const f32x4 v = total(t), up = total(MT + t);
            float o[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) o[i] = gate_up_of(v[i], up[i], alpha, limit);
            if (row < M) *(uint2 *)((bf16_t *)Y + (size_t)row * ldy + blockIdx.x * 16 + 4 * g) = make_uint2(pack2_bf16(o[0], o[1]), pack2_bf16(o[2], o[3]));
        } else if constexpr (EPI == GW_EPI_QKV) {
            const int row = 16 * t + quad_row(l16);
            const f32x4 a = total(t), b = total(MT + t);
            const float lo[4] = {a[0], a[1], a[2], a[3]}, hi[4] = {b[0], b[1], b[2], b[3]};
            if (row < M) qkv_store(store, qkv_head, row, 16 * qkv_c + 4 * g, lo, hi);
        } else {
            const int n = t / MT, row = 16 * (t % MT) + quad_row(l16), tile = blockIdx.x * NT + n, col = tile * 16 + 4 * g;
            f32x4 v = total(t);
            if (row >= M || tile * 16 >= N) continue;
            if constexpr (EPI == GW_EPI_F32) {
                *(f32x4 *)((float *)Y + (size_t)row * ldy + col) = v;
            } else {
                if constexpr (EPI == GW_EPI_GATED) {
                    const uint2 in = *(const uint2 *)(gate + (size_t)row * ldg + col);
                    const float z[4] = {__uint_as_float(in.x << 16), __uint_as_float(in.x & 0xffff0000u), __uint_as_float(in.y << 16), __uint_as_float(in.y & 0xffff0000u)};
#pragma unroll
                    for (int i = 0; i < 4; ++i) v[i] *= 1.0f / (1.0f + expf(-z[i]));
                }
                *(uint2 *)((bf16_t *)Y + (size_t)row * ldy + col) = make_uint2(pack2_bf16(v[0], v[1]), pack2_bf16(v[2], v[3]));
            }
        }
    }
}

static int wavek_launch(const void *X, int ldx, long long x_group, int groups, const void *W, void *Y, int ldy, const void *gate, int ldg,
                        int M, int N, int K, int epi, int wide, const float *sumsq, int n_in, int norm_width, float eps, float alpha, float limit,
                        const QkvStore &store, hipStream_t stream) {
    if (M <= 0) return LCU_OK;
    // (a load's place in the rows is 32 bits)
    if (M > GW_MAX_ROWS || N <= 0 || K <= 0 || N % 16 || K % 128 || ldx < 0 || ldx >= GW_MAX_LDX || groups < 1 || N % (16 * groups) || epi < 0 || epi > GW_EPI_QKV ||
        ((epi == GW_EPI_SWIGLU || epi == GW_EPI_QKV) && (N % 32 || groups != 1)) || (epi == GW_EPI_GATED && !gate) ||
        (sumsq && (n_in <= 0 || norm_width <= 0)))
        return LCU_BAD_ARGUMENT;
    const bool pairs = epi == GW_EPI_SWIGLU || epi == GW_EPI_QKV, two = pairs || (wide && (groups == 1 || N / groups % 32 == 0));
    const int tiles = N / 16, group_tiles = pairs ? tiles : tiles / groups;
    const dim3 grid(two ? (tiles + 1) / 2 : tiles), block((K / 128 < GW_WAVES ? K / 128 : GW_WAVES) * WAVE);
#define GO(NT, MT, EPI, LOADS) gemm_wavek_kernel<NT, MT, EPI, LOADS><<<grid, block, 0, stream>>>((const bf16_t *)X, ldx, (size_t)x_group, group_tiles, (const bf16_t *)W, Y, ldy, (const bf16_t *)gate, ldg, M, N, K, sumsq, n_in, norm_width, eps, alpha, limit, store)
#define ROWS(NT, EPI)                                  \
    do {                                               \
        if (M <= 4) GO(NT, 1, EPI, 1);                 \
        else if (M <= 8) GO(NT, 1, EPI, 2);            \
        else if (M <= 16) GO(NT, 1, EPI, 4);           \
        else if (M <= 32) GO(NT, 2, EPI, 4);           \
        else if (M <= 48) GO(NT, 3, EPI, 4);           \
        else GO(NT, 4, EPI, 4);                        \
    } while (0)
#define TILES(EPI) do { if (two) ROWS(2, EPI); else ROWS(1, EPI); } while (0)
    if (epi == GW_EPI_SWIGLU) ROWS(2, GW_EPI_SWIGLU);
    else if (epi == GW_EPI_QKV) ROWS(2, GW_EPI_QKV);
    else if (epi == GW_EPI_BF16) TILES(GW_EPI_BF16);
    else if (epi == GW_EPI_F32) TILES(GW_EPI_F32);
    else TILES(GW_EPI_GATED);
#undef GO
#undef ROWS
#undef TILES
    LCU_LAUNCH_CHECK();
    return LCU_OK;
}

// X: [M, ldx] (a group's rows x_group elements behind the last one's), 16-byte aligned rows; W: packed, [N, K]; Y: [M, ldy], rows aligned for
// four of its elements.  epi as above but for QKV (SWIGLU: W holds N / 2 gate rows, then the up rows, Y has N / 2 columns; GATED: gate [M, ldg] bfloat16).
// wide: 32 features a workgroup instead of 16.  sumsq: null, or [M, n_in] shares of the rows' sums of squares: the rows are multiplied by
// rsqrt(sum / norm_width + eps).
LCU_API int lcu_gemm_wavek(const void *X, int ldx, long long x_group, int groups, const void *W, void *Y, int ldy, const void *gate, int ldg,
                           int M, int N, int K, int epi, int wide, const float *sumsq, int n_in, int norm_width, float eps, float alpha, float limit,
                           hipStream_t stream) {
    if (epi == GW_EPI_QKV) return LCU_BAD_ARGUMENT;
    return wavek_launch(X, ldx, x_group, groups, W, Y, ldy, gate, ldg, M, N, K, epi, wide, sumsq, n_in, norm_width, eps, alpha, limit, QkvStore{}, stream);
}

// The q, k, v product of an attention layer with the rotation and the cache write in its epilogue (qkv_store.h): W packed, [(heads + 2 kv_heads) *
// head_dim, K], head_dim a multiple of 32.
LCU_API int lcu_gemm_wavek_qkv_rope(const void *X, int ldx, const void *W, int M, int K, void *q_out, int ldq, const int *positions, const int *slots,
                                    const float *cos_t, const float *sin_t, int max_pos, void *cache, int heads, int kv_heads, int head_dim, int page,
                                    hipStream_t stream) {
    if (M <= 0) return LCU_OK;
    if (heads <= 0 || kv_heads <= 0 || head_dim <= 0 || head_dim % 32 || page <= 0 || page % 8 || !q_out || !positions || !cos_t || !sin_t || max_pos <= 0 ||
        !cache || ldq < heads * head_dim || ldx % 8 || ldx < K || (uintptr_t)X % 16 || (uintptr_t)W % 16)
        return LCU_BAD_ARGUMENT;
    const QkvStore store = {positions, slots, cos_t, sin_t, max_pos, (bf16_t *)cache, (bf16_t *)q_out, ldq, heads, kv_heads, head_dim, page};
    return wavek_launch(X, ldx, 0, 1, W, nullptr, 0, nullptr, 0, M, (heads + 2 * kv_heads) * head_dim, K, GW_EPI_QKV, 1, nullptr, 0, 0, 0.f, 0.f, 0.f, store, stream);
}
