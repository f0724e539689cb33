// Y[M, N] = X[M, K] * W[N, K]^T for many rows (prompts), bfloat16 operands, 32-bit sums, W as its file holds it; SwiGLU in the epilogue if asked for.
//
// A workgroup has a tile of F features and T tokens.  Both operands come by loads that write into LDS themselves, 64 k a step, features and tokens in rings of
// their own (SF and ST steps: 160 KB leave room for three steps of the one and two of the other, and the weights come from further away).  A wave multiplies 32 FT
// features and 32 TT tokens by v_mfma_f32_32x32x16_bf16.  One barrier a step, in the middle of it: when a wave has read the last slice of a step (16 k) it
// waits for its loads of the next step, then all do; the products of that last slice, and then of each slice, run while the next slice is read, so the matrix
// cores have work on both sides of the barrier, and the step's loads are spread over three of the four slices (all at once they held the waves up where the
// loads are taken: 4096 x 14336, 2,048 rows, 221 us, so 207).
//
// What bounds it: LDS and the matrix cores alike (256 x 256: 1,536 cycles of a compute unit for the reads and 512 for what the loads write a step, 2,048 for
// the products), at the clock that the card's power limit leaves, about 1.6 GHz; below a full round of workgroups one step's latency.  One MI355X, random
// numbers, us, the library's and this: 4096 x 14336 800 rows 128 / 103; 2048 x 2048 1,100 rows 20.5 / 16.7, 2,014 21.9 / 22.4; 2560 x 2048 2,014 rows 27.8 /
// 25.0; SwiGLU (the library's with the activation kernel) 5632 x 2048 1,100 rows 38.2 / 31.4, 2,014 59.7 / 52.4.  The library is ahead where tiles of 256 x 256
// fill whole rounds (8192 x 2048 2,014 rows 52 / 58, 28672 x 4096 354 / 399): the caller chooses (ops.tiles_choice).  Four waves of 128 x 128 read less from
// LDS and take 388 there, but with one wave a SIMD the epilogue of SwiGLU takes 37 us instead of 10.
#include <utility>
#include <type_traits>
#include "common.h"
#include "gate_act.h"

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;

enum { GT_EPI_BF16 = 0, GT_EPI_F32 = 1, GT_EPI_SWIGLU = 2 };

template <int LEFT>
__device__ __forceinline__ void gt_wait_loads() {
    static_assert(LEFT >= 0 && LEFT < 64, "vmcnt has six bits");
    __builtin_amdgcn_s_waitcnt((LEFT & 15) | ((LEFT >> 4) << 14) | (7 << 4) | (15 << 8));
}

template <int FT_, int TT_, int WF_, int WT_, int SF_, int ST_> struct GtShape {
    static constexpr int FT = FT_, TT = TT_, WF = WF_, WT = WT_, SF = SF_, ST = ST_;
    static constexpr int WAVES = WF * WT, THREADS = WAVES * WAVE, F = 32 * FT * WF, T = 32 * TT * WT, BK = 64, PIECES = 8, SLICES = 4;
    static constexpr int LF = F / 8 / WAVES, LT = T / 8 / WAVES;       // loads of a wave a stage: features, tokens (8 rows each)
    static constexpr int LDS = (SF * F + ST * T) * PIECES;             // pieces
    static constexpr int LEFT = (SF > ST ? LF : 0) + (ST - 2) * (LF + LT);        // loads that may be on their way when a step begins
    static_assert(FT % 2 == 0 && F % (8 * WAVES) == 0 && T % (8 * WAVES) == 0 && SF >= ST && ST >= 2 && LDS * 16 <= 160 * 1024, "whole loads, and room for the stages");
};

// where piece c of row r stands in its row
template <class S> __device__ __forceinline__ int gt_place(int r, int c) { return c ^ (r & 7); }

template <class S> struct GtFrags { u32x4 f[S::FT], t[S::TT]; };

template <class S>
__device__ __forceinline__ void gt_read(u32x4 &to, const u32x4 *from) {
    to = *from;
    __builtin_amdgcn_sched_barrier(0);
}

// The last slice of one step's products while the first one of the next is read, and so on through that step's slices but the last, whose operands are in registers in
// the end.  nf, nt: the next step's stages; df, dt: the stages that the loads of a later step go to (parameters of one function with __restrict__: else the
// compiler lets every read from LDS wait for every load in flight).
template <class S, class IssueT, class IssueF>
__device__ __forceinline__ void gt_turn(const u32x4 *__restrict__ nf, const u32x4 *__restrict__ nt, u32x4 *__restrict__ df, u32x4 *__restrict__ dt, IssueT &&issue_t, IssueF &&issue_f,
                                        const int (&at)[S::SLICES], GtFrags<S> (&op)[2], f32x16 (&acc)[S::FT][S::TT]) {
#pragma unroll
    for (int s = 0; s < S::SLICES; ++s) {
        // operands of slice s - 1 (s == 0: the last of the step before) are in op[(s + 1) & 1]
        GtFrags<S> &use = op[(s + 1) & 1], &get = op[s & 1];
#pragma unroll
        for (int i = 0; i < S::FT * S::TT; ++i) {
            const int f = i / S::TT, t = i % S::TT;
            acc[f][t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, use.f[f]), __builtin_bit_cast(bf16x8, use.t[t]), acc[f][t], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            {
                constexpr int ALL = S::FT * S::TT * (S::SLICES - 1), L = S::LF + S::LT;
                const int n = s * S::FT * S::TT + i, l0 = n * L / ALL, l1 = (n + 1) * L / ALL;
#pragma unroll
                for (int l = l0; l < l1; ++l) {
                    if (l < S::LT) issue_t(dt, l);
                    else if (l < L) issue_f(df, l - S::LT);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            constexpr int READS = S::FT + S::TT;
            const int r0 = i * READS / (S::FT * S::TT), r1 = (i + 1) * READS / (S::FT * S::TT);
#pragma unroll
            for (int r = r0; r < r1; ++r) {
                if (r < S::TT) gt_read<S>(get.t[r], nt + at[s] + 32 * S::PIECES * r);
                else gt_read<S>(get.f[r - S::TT], nf + at[s] + 32 * S::PIECES * (r - S::TT));
            }
        }
    }
}

template <class S, int EPI>
__global__ void __launch_bounds__(S::THREADS, 1)
gemm_tiles_kernel(const bf16_t *__restrict__ X, int ldx, const bf16_t *__restrict__ W, void *__restrict__ Y, int ldy, int M, int N, int K, int up_rows, float alpha,
                  float limit) {
    extern __shared__ __attribute__((aligned(16))) u32x4 gt_lds[];
    constexpr int FT = S::FT, TT = S::TT, PIECES = S::PIECES;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l32 = lane & 31, hi = lane >> 5;
    const int wf = wave % S::WF, wt = wave / S::WF;
    // ---- which tile: workgroups go to the eight dies in turn; a die takes a run of tiles, those of a few feature tiles side by side
    const int t_tiles = (M + S::T - 1) / S::T, f_tiles = (N + S::F - 1) / S::F, tiles = t_tiles * f_tiles;
    const int each = (tiles + 7) / 8, item = blockIdx.x % 8 * each + blockIdx.x / 8;
    if ((int)blockIdx.x / 8 >= each || item >= tiles) return;
    const int ft0 = item / t_tiles, tt0 = item - ft0 * t_tiles;
    // ---- the loads of a stage: load i of wave w takes eight rows from (i * WAVES + w) * 8 on
    const __amdgpu_buffer_rsrc_t wb = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t *>(W), 0, (uint32_t)N * K * 2u, 0x00020000);
    const __amdgpu_buffer_rsrc_t xb = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t *>(X), 0, (uint32_t)((M - 1) * ldx + K) * 2u, 0x00020000);
    uint32_t from_f[S::LF], from_t[S::LT];
#pragma unroll
    for (int i = 0; i < S::LF; ++i) {
        const int r = (i * S::WAVES + wave) * 8 + lane / 8;
        const int row = EPI == GT_EPI_SWIGLU ? (r / 32 & 1) * up_rows + ft0 * (S::F / 2) + r / 64 * 32 + r % 32 : ft0 * S::F + r;     // SwiGLU: in turns 32 gate rows and the up rows that meet them
        from_f[i] = (uint32_t)row * (uint32_t)K * 2u + 16u * gt_place<S>(r, lane % 8);
    }
#pragma unroll
    for (int i = 0; i < S::LT; ++i) {
        const int r = (i * S::WAVES + wave) * 8 + lane / 8;
        from_t[i] = (uint32_t)(tt0 * S::T + r) * (uint32_t)ldx * 2u + 16u * gt_place<S>(r, lane % 8);
    }
    const int steps = K / S::BK;
    u32x4 *const lds_f = gt_lds, *const lds_t = gt_lds + S::SF * S::F * PIECES;
    auto issue_f = [&](u32x4 *dst, int step, int i) {
        auto *to = (__attribute__((address_space(3))) void *)(dst + (i * S::WAVES + wave) * WAVE);
        const uint32_t from = from_f[i] + (uint32_t)min(step, steps - 1) * (S::BK * 2u);      // (a plain variable: the compiler's pass for the host refuses the builtin with a type that depends on a template)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(wb, to, 16, from, 0, 0, 0);
    };
    auto issue_t = [&](u32x4 *dst, int step, int i) {
        auto *to = (__attribute__((address_space(3))) void *)(dst + (i * S::WAVES + wave) * WAVE);
        const uint32_t from = from_t[i] + (uint32_t)min(step, steps - 1) * (S::BK * 2u);      // (a plain variable: the compiler's pass for the host refuses the builtin with a type that depends on a template)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(xb, to, 16, from, 0, 0, 0);
    };
    // ---- where the lane's operands stand in a stage: row l32 of a tile, k 8 hi .. + 7 of a slice
    int at[S::SLICES];
#pragma unroll
    for (int s = 0; s < S::SLICES; ++s) at[s] = l32 * PIECES + gt_place<S>(l32, 2 * s + hi);
    const int of_f = wf * 32 * FT * PIECES, of_t = wt * 32 * TT * PIECES;
    f32x16 acc[FT][TT];
#pragma unroll
    for (int f = 0; f < FT; ++f)
#pragma unroll
        for (int t = 0; t < TT; ++t)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[f][t][i] = 0.f;
    GtFrags<S> op[2];
#pragma unroll
    for (int f = 0; f < FT; ++f) op[1].f[f] = u32x4{0u, 0u, 0u, 0u};
#pragma unroll
    for (int t = 0; t < TT; ++t) op[1].t[t] = u32x4{0u, 0u, 0u, 0u};
    // what SF - 1 turns before the first would have asked for
#pragma unroll
    for (int j = 1 - S::SF; j < 0; ++j) {
        if (j + S::ST - 1 >= 0) {
#pragma unroll
            for (int i = 0; i < S::LT; ++i) issue_t(lds_t + (j + S::ST - 1) * S::T * PIECES, j + S::ST - 1, i);
        }
#pragma unroll
        for (int i = 0; i < S::LF; ++i) issue_f(lds_f + (j + S::SF - 1) * S::F * PIECES, j + S::SF - 1, i);
    }
    int rf = 0, rt = 0, df = S::SF - 1, dt = S::ST - 1;
    for (int t = 0; t < steps; ++t) {
        gt_wait_loads<S::LEFT>();                              // this step's stages are there
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        gt_turn<S>(lds_f + rf * S::F * PIECES + of_f, lds_t + rt * S::T * PIECES + of_t, lds_f + df * S::F * PIECES, lds_t + dt * S::T * PIECES,
                   [&](u32x4 *dst, int i) { issue_t(dst, t + S::ST - 1, i); }, [&](u32x4 *dst, int i) { issue_f(dst, t + S::SF - 1, i); }, at, op, acc);
        rf = rf + 1 == S::SF ? 0 : rf + 1;
        rt = rt + 1 == S::ST ? 0 : rt + 1;
        df = df + 1 == S::SF ? 0 : df + 1;
        dt = dt + 1 == S::ST ? 0 : dt + 1;
    }
    // the last slice
#pragma unroll
    for (int i = 0; i < FT * TT; ++i)
        acc[i / TT][i % TT] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, op[1].f[i / TT]), __builtin_bit_cast(bf16x8, op[1].t[i % TT]), acc[i / TT][i % TT], 0, 0, 0);
    gt_wait_loads<0>();                                        // (the copies that nobody reads have landed before LDS is used otherwise)
    __syncthreads();
    // ---- out: a wave turns 32 tokens at a time through LDS of its own, and stores whole rows of its features
    constexpr int OUT_F = EPI == GT_EPI_SWIGLU ? 16 * FT : 32 * FT, ELEM = EPI == GT_EPI_F32 ? 4 : 2, PITCH = OUT_F * ELEM + 16, CH = OUT_F * ELEM / 16;
    static_assert(S::WAVES * 32 * PITCH <= S::LDS * 16, "room for the waves' rows");
    char *mine = (char *)gt_lds + wave * 32 * PITCH;
    const int out_n = EPI == GT_EPI_SWIGLU ? up_rows : N, f0 = (EPI == GT_EPI_SWIGLU ? ft0 * (S::F / 2) : ft0 * S::F) + wf * OUT_F;
#pragma unroll
    for (int t = 0; t < TT; ++t) {
#pragma unroll
        for (int f = 0; f < (EPI == GT_EPI_SWIGLU ? FT / 2 : FT); ++f)
#pragma unroll
            for (int q = 0; q < 4; ++q) {                      // features 32 f + 8 q + 4 hi ..
                char *to = mine + l32 * PITCH + (32 * f + 8 * q + 4 * hi) * ELEM;
                if constexpr (EPI == GT_EPI_F32) {
                    *(f32x4 *)to = f32x4{acc[f][t][4 * q], acc[f][t][4 * q + 1], acc[f][t][4 * q + 2], acc[f][t][4 * q + 3]};
                } else {
                    float o[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        o[e] = EPI == GT_EPI_SWIGLU ? gate_up_of(acc[2 * f][t][4 * q + e], acc[2 * f + 1][t][4 * q + e], alpha, limit) : acc[f][t][4 * q + e];
                    *(uint2 *)to = make_uint2(pack2_bf16(o[0], o[1]), pack2_bf16(o[2], o[3]));
                }
            }
        const int tok0 = tt0 * S::T + wt * 32 * TT + 32 * t;
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
        for (int x = 0; x < 32 * CH / WAVE; ++x) {
            const int i = x * WAVE + lane, row = i / CH, c = i % CH, col = f0 + c * (16 / ELEM);
            const u32x4 v = *(const u32x4 *)(mine + row * PITCH + c * 16);
            if (tok0 + row < M && col < out_n) *(u32x4 *)((char *)Y + ((size_t)(tok0 + row) * ldy + col) * ELEM) = v;
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
}

template <class S, int EPI>
static int gt_go(const void *X, int ldx, const void *W, void *Y, int ldy, int M, int N, int K, float alpha, float limit, hipStream_t stream) {
    const int up_rows = N / 2;
    const int tiles = ((M + S::T - 1) / S::T) * ((N + S::F - 1) / S::F);
    constexpr int bytes = S::LDS * 16;
    static_assert(bytes > 64 * 1024, "more LDS than a launch gets unasked");
    static bool asked = false;
    if (!asked) {
        const hipError_t e = hipFuncSetAttribute((const void *)gemm_tiles_kernel<S, EPI>, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
        if (e != hipSuccess) return (int)e;
        asked = true;
    }
    gemm_tiles_kernel<S, EPI><<<dim3((tiles + 7) / 8 * 8), dim3(S::THREADS), bytes, stream>>>((const bf16_t *)X, ldx, (const bf16_t *)W, Y, ldy, M, N, K, up_rows, alpha, limit);
    LCU_LAUNCH_CHECK();
    return LCU_OK;
}

// X: [M, ldx], W: [N, K], both 16-byte aligned, K a multiple of 64, ldx and N of 8; Y: [M, ldy], 16-byte aligned rows.  epi: GT_EPI_*; SWIGLU: W holds N / 2 gate rows
// (a multiple of 8), then the up rows, Y has N / 2 columns.  shape: 0 to 2, tiles of features x tokens: 128 x 128, 128 x 256, 256 x 256.
LCU_API int lcu_gemm_tiles(const void *X, int ldx, const void *W, void *Y, int ldy, int M, int N, int K, int epi, int shape, float alpha, float limit, hipStream_t stream) {
    if (M <= 0) return LCU_OK;
    const int cols = epi == GT_EPI_SWIGLU ? N / 2 : N, elem = epi == GT_EPI_F32 ? 4 : 2;
    // (a load's place is 32 bits, rows of the last tiles beyond the matrices' ends too)
    if (N <= 0 || K <= 0 || K % 64 || ldx < K || ldx % 8 || cols % 8 || (epi == GT_EPI_SWIGLU && N % 16) || ldy < cols || ldy * elem % 16 || !X || !W || !Y ||
        ((uintptr_t)X | (uintptr_t)W | (uintptr_t)Y) % 16 || (unsigned long long)(M + 256ll) * ldx * 2 >= 1ull << 32 || (unsigned long long)(N + 256ll) * K * 2 >= 1ull << 32)
        return LCU_BAD_ARGUMENT;
#define GO(...)                                                                                                                        \
    do {                                                                                                                              \
        typedef GtShape<__VA_ARGS__> S;                                                                                                \
        if (epi == GT_EPI_BF16) return gt_go<S, GT_EPI_BF16>(X, ldx, W, Y, ldy, M, N, K, alpha, limit, stream);                        \
        if (epi == GT_EPI_F32) return gt_go<S, GT_EPI_F32>(X, ldx, W, Y, ldy, M, N, K, alpha, limit, stream);                          \
        if (epi == GT_EPI_SWIGLU) return gt_go<S, GT_EPI_SWIGLU>(X, ldx, W, Y, ldy, M, N, K, alpha, limit, stream);                    \
        return LCU_BAD_ARGUMENT;                                                                                                      \
    } while (0)
    if (shape == 0) GO(2, 2, 2, 2, 4, 4);
    if (shape == 1) GO(2, 2, 2, 4, 3, 3);
    if (shape == 2) GO(4, 2, 2, 4, 3, 2);
#undef GO
    return LCU_BAD_ARGUMENT;
}
