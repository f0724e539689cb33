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
// One MI355X, weights out of memory, beside the weight-streaming kernel, the row-sharing one and the library's, us a product (graph of
// products one after the other): 2048 x 2048: 5.0 / 4.8 / - / 8.1 at 8 rows, 7.1 / 8.2 / 7.8 / 8.3 at 32, 10.9 / - / 12.1 / 8.7 at 64;
// 8192 x 2048: 7.4 / 7.8 / - / 12.9 at 8, 9.4 / 11.0 / 9.4 / 13.0 at 32; SwiGLU of 5632 x 2048: 6.8 / 9.9 / - / 14 at 8, 7.4 / 10.7 / - / 14 at
// 16, 9.2 / 14.5 / 8.5 / 14 at 32, 15.1 / - / 16.1 / 15 at 64; 4096 x 4096: 9.9 / 8.0 at 8 (a wave's share of K and X grow: the
// weight-streaming kernel).  What bounds it is latency up to 16 rows, beyond it the rows' way from the L2 caches: 1.6 us for every 16 of
// them at K = 2048.  Groups with a gate (a latent's heads): 16 of 128 x 512 3.5 / 4.1 / - / 12.3 at 8 rows, 4.2 / 5.9 / - / 10.9 at 32, 5.4 / - / - / 11.3 at
// 64; 64 of 128 x 512 4.5 / 6.1, 5.3 / 9.1 and 8.1 / 11.6 (library) there.
//
// Groups: X is [groups][M, K], group g's rows x_group elements further, and multiplies the rows g * N / groups .. of W.
#include "common.h"
#include "gate_act.h"
#include "lane_moves.h"

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;

enum { GW_EPI_BF16 = 0, GW_EPI_F32 = 1, GW_EPI_SWIGLU = 2, GW_EPI_GATED = 3 };     // GATED: bf16, times sigmoid(gate)

constexpr int GW_WAVES = 8, GW_MAX_ROWS = 64;

// A macro-step's rows come from memory as whole pieces of 64 bytes: load i brings lane group q the eight k from 32 i + 8 q on.  The packed
// weight's load j holds for lane group q the k from 32 q + 8 j on.  So x[j], group q = r[q], group j: a transposition between the loads
// and the four groups of 16 lanes, in the vector unit.  (Rows loaded in the weight's order touch four times as many lines: 16 us at 64
// rows of 2048 with 2048 features, now 10.9.)
__device__ __forceinline__ void by_groups(const u32x4 (&r)[4], u32x4 (&x)[4]) {
#pragma unroll
    for (int d = 0; d < 4; ++d) {
        const auto ab = __builtin_amdgcn_permlane32_swap(r[0][d], r[2][d], false, false);      // (r0.0 r0.1 r2.0 r2.1), (r0.2 r0.3 r2.2 r2.3)
        const auto cd = __builtin_amdgcn_permlane32_swap(r[1][d], r[3][d], false, false);
        const auto lo = __builtin_amdgcn_permlane16_swap(ab[0], cd[0], false, false);          // (r0.0 r1.0 r2.0 r3.0), (r0.1 r1.1 r2.1 r3.1)
        const auto hi = __builtin_amdgcn_permlane16_swap(ab[1], cd[1], false, false);
        x[0][d] = lo[0];
        x[1][d] = lo[1];
        x[2][d] = hi[0];
        x[3][d] = hi[1];
    }
}

// NT: tiles of 16 features a workgroup; MT: tiles of 16 rows.
template <int NT, int MT, int EPI>
__global__ void __launch_bounds__(GW_WAVES *WAVE)
gemm_wavek_kernel(const bf16_t *__restrict__ X, int ldx, size_t x_group, int group_tiles, const bf16_t *__restrict__ W, void *__restrict__ Y,
                  int ldy, const bf16_t *__restrict__ gate, int ldg, int M, int N, int K, const float *__restrict__ sumsq, int n_in,
                  int norm_width, float eps, float alpha, float limit) {
    constexpr int AHEAD = 2;                         // macro-steps (128 k) whose loads are on their way
    __shared__ f32x4 red[GW_WAVES][NT * MT][WAVE];
    __shared__ float factor[16 * MT];
    const int waves = blockDim.x >> 6;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, g = lane >> 4, l16 = lane & 15;
    const int macros = K / 128, per = (macros + waves - 1) / waves, m0 = min(macros, wave * per), m1 = min(macros, m0 + per);
    const bf16_t *wp[NT], *xp[MT];
#pragma unroll
    for (int n = 0; n < NT; ++n) {
        const int tile = EPI == GW_EPI_SWIGLU ? blockIdx.x + n * (N / 32) : min((int)blockIdx.x * NT + n, N / 16 - 1);
        wp[n] = W + (size_t)tile * 16 * K + lane * 8;
    }
    X += (size_t)(blockIdx.x * NT / group_tiles) * x_group;
#pragma unroll
    for (int m = 0; m < MT; ++m) xp[m] = X + (size_t)min(16 * m + l16, M - 1) * ldx + 8 * g;
    f32x4 acc[NT][MT];
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[n][m] = f32x4{0.f, 0.f, 0.f, 0.f};
    u32x4 a[AHEAD][NT][4], b[AHEAD][MT][4];
    auto fetch = [&](int u, int s) {
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
            for (int j = 0; j < 4; ++j) a[u][n][j] = __builtin_nontemporal_load((const u32x4 *)(wp[n] + (size_t)s * 2048 + 512 * j));
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int j = 0; j < 4; ++j) b[u][m][j] = *(const u32x4 *)(xp[m] + 128 * s + 32 * j);
    };
#pragma unroll
    for (int u = 0; u < AHEAD; ++u)
        if (m0 + u < m1) fetch(u, m0 + u);
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
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                u32x4 x[4];
                by_groups(b[u][m], x);
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int n = 0; n < NT; ++n)
                        acc[n][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a[u][n][j]), __builtin_bit_cast(bf16x8, x[j]), acc[n][m], 0, 0, 0);
            }
            if (s + u + AHEAD < m1) fetch(u, s + u + AHEAD);
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
        return sumsq ? v * factor[16 * (t % MT) + l16] : v;
    };
    // a wave stores a tile: four neighbouring features of a row a lane
    for (int t = wave; t < (EPI == GW_EPI_SWIGLU ? MT : NT * MT); t += waves) {
        if constexpr (EPI == GW_EPI_SWIGLU) {
            const int row = 16 * t + l16;
            const f32x4 v = total(t), up = total(MT + t);
            float o[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) o[i] = gate_up_of(v[i], up[i], alpha, limit);
            if (row < M) *(uint2 *)((bf16_t *)Y + (size_t)row * ldy + blockIdx.x * 16 + 4 * g) = make_uint2(pack2_bf16(o[0], o[1]), pack2_bf16(o[2], o[3]));
        } else {
            const int n = t / MT, row = 16 * (t % MT) + l16, tile = blockIdx.x * NT + n, col = tile * 16 + 4 * g;
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

// X: [M, ldx] (a group's rows x_group elements behind the last one's), 16-byte aligned rows; W: packed, [N, K]; Y: [M, ldy], rows aligned for
// four of its elements.  epi as above (SWIGLU: W holds N / 2 gate rows, then the up rows, Y has N / 2 columns; GATED: gate [M, ldg] bfloat16).
// wide: 32 features a workgroup instead of 16.  sumsq: null, or [M, n_in] shares of the rows' sums of squares: the rows are multiplied by
// rsqrt(sum / norm_width + eps).
LCU_API int lcu_gemm_wavek(const void *X, int ldx, long long x_group, int groups, const void *W, void *Y, int ldy, const void *gate, int ldg,
                           int M, int N, int K, int epi, int wide, const float *sumsq, int n_in, int norm_width, float eps, float alpha, float limit,
                           hipStream_t stream) {
    if (M <= 0) return LCU_OK;
    if (M > GW_MAX_ROWS || N <= 0 || K <= 0 || N % 16 || K % 128 || groups < 1 || N % (16 * groups) || epi < 0 || epi > GW_EPI_GATED ||
        (epi == GW_EPI_SWIGLU && (N % 32 || groups != 1)) || (epi == GW_EPI_GATED && !gate) ||
        (sumsq && (n_in <= 0 || norm_width <= 0)))
        return LCU_BAD_ARGUMENT;
    const bool two = epi == GW_EPI_SWIGLU || (wide && N / groups % 32 == 0);
    const int tiles = N / 16, group_tiles = epi == GW_EPI_SWIGLU ? tiles : tiles / groups, mt = (M + 15) / 16;
    const dim3 grid(two ? tiles / 2 : tiles), block((K / 128 < GW_WAVES ? K / 128 : GW_WAVES) * WAVE);
#define GO(NT, MT, EPI) gemm_wavek_kernel<NT, MT, EPI><<<grid, block, 0, stream>>>((const bf16_t *)X, ldx, (size_t)x_group, group_tiles, (const bf16_t *)W, Y, ldy, (const bf16_t *)gate, ldg, M, N, K, sumsq, n_in, norm_width, eps, alpha, limit)
#define ROWS(NT, EPI)                                  \
    do {                                               \
        if (mt == 1) GO(NT, 1, EPI);                   \
        else if (mt == 2) GO(NT, 2, EPI);              \
        else if (mt == 3) GO(NT, 3, EPI);              \
        else GO(NT, 4, EPI);                           \
    } while (0)
#define TILES(EPI) do { if (two) ROWS(2, EPI); else ROWS(1, EPI); } while (0)
    if (epi == GW_EPI_SWIGLU) ROWS(2, GW_EPI_SWIGLU);
    else if (epi == GW_EPI_BF16) TILES(GW_EPI_BF16);
    else if (epi == GW_EPI_F32) TILES(GW_EPI_F32);
    else TILES(GW_EPI_GATED);
#undef GO
#undef ROWS
#undef TILES
    LCU_LAUNCH_CHECK();
    return LCU_OK;
}
