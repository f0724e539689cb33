// The delta rules over portions of many tokens: chunks of 64 tokens side by side on the 32-bit matrix instruction.
//
// A token maps a head's state by S <- diag(w) S - al (u^T S) + k v^T, o = S^T r (gated: w one number, al = beta g u, k = u).  Within
// a chunk, with G_t the product of the decays up to t (per key channel), c_t = u_t^T S_(t-1) and the rows
//   u~_t = u_t G_(t-1),  r~_t = r_t G_t,  k~_s = k_s / G_s,  al~_s = al_s / G_s
// the chunk is  c = T (u~ S + tril(u~ k~^T, -1) v),  T = (I + tril(u~ al~^T, -1))^-1,
//               o = r~ S + tril(r~ k~^T) v - tril(r~ al~^T) c,    S <- G_C (S + k~^T v - al~^T c),
// which is affine in the state that the chunk finds:  S <- F S + H,  o = P S + Q, with
//   M = T u~, N = T tril(u~ k~^T, -1) v;   F = G_C (I - al~^T M),  H = G_C (k~^T v - al~^T N),  P = r~ - tril(r~ al~^T) M,
//   Q = tril(r~ k~^T) v - tril(r~ al~^T) N.
// Two kernels: `maps` makes F, H, P and Q of every chunk and head at once; `chain` walks a request's chunks, 16 value columns a
// workgroup, and applies them.  A token alone (delta_scan_kernel) is a chain of 0.55 us a token, 0.9 us and more where the decay is per
// channel; a chunk is one of 2.3 us.  2,048 tokens of one request, 16 heads of 128: gated 1,100 us scanned, maps 68 and chain 79 us in
// chunks; with decays per channel 1,800 to 2,400 us scanned, 106 and 79 us in chunks.  64 tokens (the fewest that come here) gated 32
// us scanned, 35 in chunks, with decays per channel 58 and more against 54.
//
// What bounds them: `maps` runs 4,300 (channel-wise 6,300) matrix instructions of 32 cycles a chunk and head, 14 (21) us on a compute
// unit's four SIMDs, of which it takes 30 (48): one workgroup of 8 waves fits a compute unit beside its LDS.  `chain` is its 96 matrix
// instructions a SIMD and chunk (1.3 us) and the round through LDS; the affine form costs `maps` a third more products than c, o and S
// in turn would, but leaves one product instead of two, one after the other, on the chain.
//
// The decays per channel are at least exp(-exp(-1/2)) = 0.545 a token, so G over a chunk stays above 1e-17 and 1 / G below 1e17: the
// products u~_t k~_s are of the size of u_t k_s again and lose nothing (a quotient of two rounded numbers).  The gated rule's one decay
// may be as small as it likes: there the products u k^T and r k^T are weighted by exp(L_t - L_s) <= 1, L the sums of log g in 64-bit.
//
// All products are 32-bit with 32-bit sums (v_mfma_f32_16x16x4_f32).  In its operands lane (l, g) of 16 x 4 holds row (or column) l and
// index g of the summed four, in its results column l and rows 4 g .. 4 g + 3: with the summed index permuted alike on both sides
// (step e of a tile of 16 takes the indexes 4 g + e) results are the next product's operand as they are.
#pragma once
#include <mutex>
#include "common.h"

constexpr int DELTA_CHUNK = 64;
constexpr int DELTA_LONG = 64;                   // a request that feeds fewer tokens in a step walks them one by one
constexpr int DELTA_CHUNK_THREADS = 512;
constexpr int DELTA_LDM = DELTA_CHUNK + 4;       // rows of a [64][64] matrix in LDS
constexpr int DELTA_MAX_DEVICES = 16;

typedef __attribute__((ext_vector_type(4))) float dc_f32x4;

struct DeltaChunkArgs {
    const float *prep;                           // [n, heads, 5 dk] (w | al | u | k | r) or, gated, [n, heads, 2 dk + 4] (u | r | g, beta g, log g, 0)
    const void *proj;                            // the values: columns off_v of rows [n, row_stride] of T, or vf [n, heads * dv] if not null
    int row_stride, off_v;
    const float *vf;
    float *f, *h, *p, *q;                        // [slot][head] of [DK][DK], [DK][16 tiles], [64][DK], [64][16 tiles], in tiles of 16 x 16: F
                                                 // and P as left operands [row tile][index tile], H and Q as results [column tile][row tile]
    float *state;
    size_t slot_stride;
    float *o;                                    // [n, heads * dv]
    const int *q_start, *ctx_len, *state_slot;
    int n_req, heads, dk, dv, tiles;             // tiles: of 16 value columns
};

// The chunks that a step of n tokens in n_req requests can have: every long request's last one may be cut short.
__host__ __device__ inline int delta_chunk_slots(int n, int n_req) {
    const int most = n / DELTA_LONG;
    return n / DELTA_CHUNK + (most < n_req ? most : n_req);
}
// Whether a step may hold a long request (every request feeds a token at least).
inline bool delta_chunks_possible(int n, int n_req, int dk) { return dk <= 128 && n - n_req + 1 >= DELTA_LONG; }
inline int delta_padded(int dk) { return dk <= 64 ? 64 : 128; }
inline size_t delta_chunk_floats(int n, int n_req, int heads, int dk, int dv) {
    if (!delta_chunks_possible(n, n_req, dk)) return 0;
    const size_t D = delta_padded(dk), V = (size_t)(dv + 15) / 16 * 16;
    return (size_t)delta_chunk_slots(n, n_req) * heads * (D * D + D * V + DELTA_CHUNK * (D + V));
}

__device__ __forceinline__ dc_f32x4 dc_mma(float4 a, dc_f32x4 b, dc_f32x4 c) {
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.x, b[0], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.y, b[1], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.z, b[2], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.w, b[3], c, 0, 0, 0);
    return c;
}
// Where element (row m, index k) of a tile of 16 x 16 stands in memory: in the order in which a wave's lanes take the tile as the left
// operand, so that the wave reads whole lines.
__device__ __forceinline__ int dc_operand(int tile, int m, int k) { return (tile * WAVE + k / 4 * 16 + m) * 4 + k % 4; }
// Keeps the compiler from holding what it reads from LDS here in registers until it is read again later: that would spill.
__device__ __forceinline__ void dc_forget() { asm volatile("" ::: "memory"); }
__device__ __forceinline__ dc_f32x4 dc_vec(float4 v) { return dc_f32x4{v.x, v.y, v.z, v.w}; }

// LDS of `maps`, in floats: the channel-wise rule holds four [64][DK + 4] arrays, of which the first two make room for the four
// [64][68] matrices; the gated rule two of each.
template <bool GATED, int DK> struct DeltaMapsLds {
    static constexpr int LD = DK + 4, ROWS = DELTA_CHUNK * LD, MAT = DELTA_CHUNK * DELTA_LDM;
    static constexpr int FRONT = GATED ? ROWS : (2 * ROWS > 4 * MAT ? 2 * ROWS : 4 * MAT);      // (gated: u stays)
    static constexpr int REST = GATED ? ROWS + 2 * MAT : 2 * ROWS;
    static constexpr int DINV = 4 * 16 * 20;
    static constexpr int SMALL = 512 + DK;        // gated: the sums of log g in two parts, beta g, weights; G_C
    static constexpr int FLOATS = FRONT + REST + DINV + SMALL;
};

template <class T, bool GATED, int DK>
__global__ void __launch_bounds__(DELTA_CHUNK_THREADS, 1)
delta_maps_kernel(DeltaChunkArgs p) {
    typedef DeltaMapsLds<GATED, DK> L;
    constexpr int C = DELTA_CHUNK, LD = L::LD, LDM = DELTA_LDM, KT = DK / 16, THREADS = DELTA_CHUNK_THREADS, WAVES = THREADS / WAVE;
    extern __shared__ __attribute__((aligned(16))) float dc_lds[];
    float *us = dc_lds, *rs = us + L::ROWS;                                   // u~ and r~ (gated: u and r)
    float *ks = dc_lds + L::FRONT, *as = ks + L::ROWS;                        // k~ and al~ (channel-wise)
    float *m_uk = GATED ? rs + L::ROWS : dc_lds, *m_rk = m_uk + L::MAT, *m_ua = m_rk + L::MAT, *m_ra = m_ua + L::MAT;
    float *dinv = dc_lds + L::FRONT + L::REST, *small = dinv + L::DINV, *g_all = small + 512;
    float *l_hi = small, *l_lo = l_hi + C, *bg = l_lo + C, *w_end = bg + C, *w_start = w_end + C;        // gated, by token
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, g = lane >> 4, l16 = lane & 15, head = blockIdx.y;
    // ---- which request's chunk this is
    int t0 = 0, nt = 0;
    {
        int left = blockIdx.x;
        for (int r = 0; r < p.n_req; ++r) {
            const int a = p.q_start[r], b = p.q_start[r + 1], len = b - a;
            if (len < DELTA_LONG) continue;
            const int chunks = (len + C - 1) / C;
            if (left < chunks) {
                t0 = a + left * C;
                nt = min(C, b - t0);
                break;
            }
            left -= chunks;
        }
        if (nt == 0) return;                                                  // (fewer chunks than the step could have had)
    }
    const int dk = p.dk, dv = p.dv, heads = p.heads;
    const size_t no = (size_t)blockIdx.x * heads + head;
    // ---- the tokens' vectors
    if constexpr (GATED) {
        const int row = 2 * dk + 4;
        if (wave == 0) {
            const float *s = p.prep + ((size_t)(t0 + min(lane, nt - 1)) * heads + head) * row + 2 * dk;
            double l = lane < nt ? (double)fmaxf(s[2], -1e4f) : 0.0;          // (a decay of exp(-1e4) is 0 like any smaller one)
            const float b = lane < nt ? s[1] : 0.f;
#pragma unroll
            for (int off = 1; off < C; off <<= 1) {
                const double before = __shfl_up(l, off, WAVE);
                if (lane >= off) l += before;
            }
            const float hi = (float)l, lo = (float)(l - (double)hi);
            const float end_hi = __shfl(hi, C - 1, WAVE), end_lo = __shfl(lo, C - 1, WAVE);
            l_hi[lane] = hi;
            l_lo[lane] = lo;
            bg[lane] = b;
            w_end[lane] = expf((end_hi - hi) + (end_lo - lo));
            w_start[lane] = expf(hi + lo);
        }
#pragma unroll
        for (int x = tid; x < C * (DK / 4); x += THREADS) {
            const int t = x / (DK / 4), c = x % (DK / 4) * 4;
            const float *s = p.prep + ((size_t)(t0 + min(t, nt - 1)) * heads + head) * row;
            float4 u, r;
            if (dk % 4 == 0) {                                                // (rows of 2 dk + 4 floats: whole pieces of four)
                u = *(const float4 *)(s + min(c, dk - 4));
                r = *(const float4 *)(s + dk + min(c, dk - 4));
                if (t >= nt || c >= dk) u = r = make_float4(0.f, 0.f, 0.f, 0.f);
            } else {
                auto at = [&](int e) { return t < nt && c + e < dk ? s[c + e] : 0.f; };
                u = make_float4(at(0), at(1), at(2), at(3));
                auto rt = [&](int e) { return t < nt && c + e < dk ? s[dk + c + e] : 0.f; };
                r = make_float4(rt(0), rt(1), rt(2), rt(3));
            }
            *(float4 *)(us + t * LD + c) = u;
            *(float4 *)(rs + t * LD + c) = r;
        }
    } else {
        // a thread per channel and group of tokens: the decays' products in 64-bit, first the groups' own
        constexpr int GROUPS = THREADS / DK, PER = C / GROUPS;
        double *part = (double *)dinv;                                        // [GROUPS][DK], not needed any more when dinv is made
        static_assert(2 * GROUPS * DK <= L::DINV, "room for the groups' products");
        const int c = tid % DK, grp = tid / DK, row = 5 * dk;
        const float *s = p.prep + ((size_t)t0 * heads + head) * row + min(c, dk - 1);
        float w[PER];
        double own = 1.0;
#pragma unroll
        for (int e = 0; e < PER; ++e) {
            const int t = grp * PER + e;
            w[e] = s[(size_t)min(t, nt - 1) * heads * row];
            if (t >= nt || c >= dk) w[e] = 1.f;
            own *= (double)w[e];
        }
        part[grp * DK + c] = own;
        __syncthreads();
        double before = 1.0;
        for (int x = 0; x < grp; ++x) before *= part[x * DK + c];
#pragma unroll
        for (int e = 0; e < PER; ++e) {
            const int t = grp * PER + e;
            const float *x = s + (size_t)min(t, nt - 1) * heads * row;
            const bool in = t < nt && c < dk;
            const float al = in ? x[dk] : 0.f, u = in ? x[2 * dk] : 0.f, k = in ? x[3 * dk] : 0.f, r = in ? x[4 * dk] : 0.f;
            us[t * LD + c] = u * (float)before;
            before *= (double)w[e];
            const float inv = (float)(1.0 / before);
            rs[t * LD + c] = r * (float)before;
            ks[t * LD + c] = k * inv;
            as[t * LD + c] = al * inv;
        }
        if (grp == GROUPS - 1) g_all[c] = (float)before;
    }
    __syncthreads();
    // ---- the matrices: waves 0 to 3 a tile of 16 rows of u's, waves 4 to 7 of r's (the longest strips beside the shortest on a SIMD)
    {
        const bool of_r = wave >= 4;
        const int a = of_r ? 3 - (wave & 3) : wave & 3;
        const float *left = of_r ? rs : us;
        dc_f32x4 k4[4], a4[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) k4[c] = a4[c] = dc_f32x4{0.f, 0.f, 0.f, 0.f};
        for (int x = 0; x < KT; ++x) {
            const dc_f32x4 b = dc_vec(*(const float4 *)(left + (16 * a + l16) * LD + 16 * x + 4 * g));
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                if (c > a) continue;
                const int at = (16 * c + l16) * LD + 16 * x + 4 * g;
                k4[c] = dc_mma(*(const float4 *)((GATED ? us : ks) + at), b, k4[c]);
                if constexpr (!GATED) a4[c] = dc_mma(*(const float4 *)(as + at), b, a4[c]);
            }
        }
        // this lane's results: token t (of the strip), tokens 16 c + 4 g + i
        const int t = 16 * a + l16;
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int s = 16 * c + 4 * g + i;
                const bool in = of_r ? s <= t : s < t;
                if constexpr (GATED) {
                    const int from = of_r ? t : max(t - 1, 0);
                    k4[c][i] = in ? k4[c][i] * expf((l_hi[from] - l_hi[s]) + (l_lo[from] - l_lo[s])) : 0.f;
                } else {
                    k4[c][i] = in ? k4[c][i] : 0.f;
                    a4[c][i] = in ? a4[c][i] : 0.f;
                }
            }
        // (channel-wise) u~ and r~ make room: what the column tiles still need of them goes to registers, below
        dc_f32x4 um[4], rm[4];
        if (wave < KT) {
#pragma unroll
            for (int b = 0; b < 4; ++b)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int s = 16 * b + 4 * g + i;
                    um[b][i] = us[s * LD + 16 * wave + l16];
                    rm[b][i] = rs[s * LD + 16 * wave + l16];
                    if constexpr (GATED) {
                        um[b][i] *= s > 0 ? w_start[s - 1] : 1.f;
                        rm[b][i] *= w_start[s];
                    }
                }
        }
        if constexpr (!GATED) __syncthreads();
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            if (c > a) continue;
            *(dc_f32x4 *)((of_r ? m_rk : m_uk) + t * LDM + 16 * c + 4 * g) = k4[c];
            if constexpr (!GATED) *(dc_f32x4 *)((of_r ? m_ra : m_ua) + t * LDM + 16 * c + 4 * g) = a4[c];
        }
        __syncthreads();
        // ---- the inverses of the four diagonal blocks I + tril(., -1), a column a lane; a row is on its way while the one before is used
        if (wave < 4 && lane < 16) {
            const float *m = (GATED ? m_uk : m_ua) + 16 * wave * LDM + 16 * wave;
            float4 next[4], bgs[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                next[j] = *(const float4 *)(m + LDM + 4 * j);
                if constexpr (GATED) bgs[j] = *(const float4 *)(bg + 16 * wave + 4 * j);
            }
            float col[16];
            col[0] = lane == 0 ? 1.f : 0.f;
            dinv[16 * wave * 20 + lane] = col[0];
#pragma unroll
            for (int i = 1; i < 16; ++i) {
                float row[16];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    row[4 * j] = next[j].x; row[4 * j + 1] = next[j].y; row[4 * j + 2] = next[j].z; row[4 * j + 3] = next[j].w;
                    if constexpr (GATED) { row[4 * j] *= bgs[j].x; row[4 * j + 1] *= bgs[j].y; row[4 * j + 2] *= bgs[j].z; row[4 * j + 3] *= bgs[j].w; }
                    if (i < 15) next[j] = *(const float4 *)(m + (i + 1) * LDM + 4 * j);
                }
                float v = i == lane ? 1.f : 0.f;
#pragma unroll
                for (int j = 0; j < i; ++j) v -= row[j] * col[j];
                col[i] = v;
                dinv[(16 * wave + i) * 20 + lane] = v;
            }
        }
        __syncthreads();
        // X = T B for 16 columns: lane (l, g) holds rows 16 a + 4 g + i of column l
        auto solve = [&](dc_f32x4 *x) {
            dc_f32x4 bx[4];
            dc_forget();
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                dc_f32x4 sum = dc_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int c = 0; c < b; ++c) sum = dc_mma(*(const float4 *)((GATED ? m_uk : m_ua) + (16 * b + l16) * LDM + 16 * c + 4 * g), bx[c], sum);
                x[b] -= sum;
                x[b] = dc_mma(*(const float4 *)(dinv + (16 * b + l16) * 20 + 4 * g), x[b], dc_f32x4{0.f, 0.f, 0.f, 0.f});
                bx[b] = x[b];
                if constexpr (GATED) bx[b] *= dc_vec(*(const float4 *)(bg + 16 * b + 4 * g));
            }
        };
        // ---- columns of M, and with them of P and F
        if (wave < KT) {
            float *pp = p.p + no * C * DK, *ff = p.f + no * DK * DK;
            solve(um);
            dc_forget();
            if constexpr (GATED) {
#pragma unroll
                for (int b = 0; b < 4; ++b) um[b] *= dc_vec(*(const float4 *)(bg + 16 * b + 4 * g));
            }
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                dc_f32x4 sum = dc_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int c = 0; c <= b; ++c) sum = dc_mma(*(const float4 *)((GATED ? m_rk : m_ra) + (16 * b + l16) * LDM + 16 * c + 4 * g), um[c], sum);
#pragma unroll
                for (int i = 0; i < 4; ++i) pp[dc_operand(b * KT + wave, 4 * g + i, l16)] = rm[b][i] - sum[i];
            }
            if constexpr (GATED) {
#pragma unroll
                for (int b = 0; b < 4; ++b) um[b] *= dc_vec(*(const float4 *)(w_end + 16 * b + 4 * g));
            }
#pragma unroll 4
            for (int y = 0; y < KT; ++y) {
                if (y % 2 == 0) dc_forget();
                dc_f32x4 sum = dc_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    const float *at = (GATED ? us : as) + (16 * b + 4 * g) * LD + 16 * y + l16;
                    sum = dc_mma(make_float4(at[0], at[LD], at[2 * LD], at[3 * LD]), um[b], sum);
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int key = 16 * y + 4 * g + i;
                    const float one = key == 16 * wave + l16 ? 1.f : 0.f;
                    ff[dc_operand(y * KT + wave, 4 * g + i, l16)] = GATED ? one * w_start[C - 1] - sum[i] : g_all[key] * (one - sum[i]);
                }
            }
        }
        // ---- columns of N, and with them of Q and H
        const int width = p.tiles * 16;
        for (int tile = wave; tile < p.tiles; tile += WAVES) {
            float *qq = p.q + no * C * width, *hh = p.h + no * DK * width;
            const int col = tile * 16 + l16;
            dc_f32x4 v[4], x[4];
            dc_forget();
#pragma unroll
            for (int b = 0; b < 4; ++b)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int s = 16 * b + 4 * g + i;
                    const size_t tok = t0 + min(s, nt - 1);
                    const int cc = head * dv + min(col, dv - 1);
                    const float e = p.vf ? p.vf[tok * heads * dv + cc] : to_f32(((const T *)p.proj)[tok * p.row_stride + p.off_v + cc]);
                    v[b][i] = s < nt && col < dv ? e : 0.f;
                }
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                x[b] = dc_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int c = 0; c <= b; ++c) x[b] = dc_mma(*(const float4 *)(m_uk + (16 * b + l16) * LDM + 16 * c + 4 * g), v[c], x[b]);
            }
            solve(x);
            dc_forget();
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                if constexpr (GATED) v[b] -= x[b] * dc_vec(*(const float4 *)(bg + 16 * b + 4 * g));     // (one product for both: their keys are the same)
                else x[b] = -x[b];
            }
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                dc_f32x4 sum = dc_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int c = 0; c <= b; ++c) {
                    const int at = (16 * b + l16) * LDM + 16 * c + 4 * g;
                    sum = dc_mma(*(const float4 *)(m_rk + at), v[c], sum);
                    if constexpr (!GATED) sum = dc_mma(*(const float4 *)(m_ra + at), x[c], sum);
                }
                *(dc_f32x4 *)(qq + ((size_t)(tile * (C / 16) + b) * WAVE + lane) * 4) = sum;
            }
            if constexpr (GATED) {
#pragma unroll
                for (int b = 0; b < 4; ++b) v[b] *= dc_vec(*(const float4 *)(w_end + 16 * b + 4 * g));
            }
#pragma unroll 4
            for (int y = 0; y < KT; ++y) {
                if (y % 2 == 0) dc_forget();
                dc_f32x4 sum = dc_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    const int at = (16 * b + 4 * g) * LD + 16 * y + l16;
                    const float *kp = (GATED ? us : ks) + at;
                    sum = dc_mma(make_float4(kp[0], kp[LD], kp[2 * LD], kp[3 * LD]), v[b], sum);
                    if constexpr (!GATED) sum = dc_mma(make_float4(as[at], as[at + LD], as[at + 2 * LD], as[at + 3 * LD]), x[b], sum);
                }
                if constexpr (!GATED) sum *= dc_vec(*(const float4 *)(g_all + 16 * y + 4 * g));
                *(dc_f32x4 *)(hh + ((size_t)(tile * KT + y) * WAVE + lane) * 4) = sum;
            }
        }
    }
}

// One workgroup per (request, head, 16 value columns): a wave per 16 key channels, whose part of S stays in registers as the results of
// F S + H and goes through LDS once a chunk, where every wave reads all of it; four more waves make the chunk's outputs, 16 tokens
// each.  The maps of the next three chunks are on their way meanwhile (with one chunk ahead, and rows of F in pieces of 64 bytes, a
// chunk took 3.7 us).  The workgroups of a head lie heads * requests apart in launch order, on one die where that is a multiple of
// eight: F and P come out of its L2 for all but one.
template <int DK>
__global__ void __launch_bounds__((DK / 16 + DELTA_CHUNK / 16) * WAVE)
delta_chain_kernel(DeltaChunkArgs p) {
    constexpr int C = DELTA_CHUNK, KT = DK / 16, LD = DK + 4, AHEAD = 3;
    __shared__ __attribute__((aligned(16))) float st[2][16 * LD];             // S of these columns, a column a row
    const int r = blockIdx.x, head = blockIdx.y, tile = blockIdx.z;
    const int t_first = p.q_start[r], t_end = p.q_start[r + 1], q_len = t_end - t_first;
    if (q_len < DELTA_LONG) return;
    int slot = 0;
    for (int x = 0; x < r; ++x) {
        const int len = p.q_start[x + 1] - p.q_start[x];
        if (len >= DELTA_LONG) slot += (len + C - 1) / C;
    }
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), g = lane >> 4, l16 = lane & 15;
    const int dk = p.dk, dv = p.dv, heads = p.heads, width = p.tiles * 16, col = tile * 16 + l16;
    float *mat = p.state + (size_t)p.state_slot[r] * p.slot_stride + (size_t)head * dk * dv;
    const bool of_state = wave < KT;
    const int y = of_state ? wave : wave - KT, row0 = 16 * y + 4 * g;         // this wave's rows: key channels, or the chunk's tokens
    // the wave's rows of the maps of chunk number `slot + c`
    const float *left = of_state ? p.f + (size_t)y * KT * 256 : p.p + (size_t)y * KT * 256;
    const float *right = of_state ? p.h + (size_t)(tile * KT + y) * 256 : p.q + (size_t)(tile * (C / 16) + y) * 256;
    const size_t left_step = of_state ? DK * DK : C * DK, right_step = (size_t)(of_state ? DK : C) * width;
    const int chunks = (q_len + C - 1) / C;
    dc_f32x4 a[AHEAD][KT], b[AHEAD];
    auto fetch = [&](int c, dc_f32x4 *av, dc_f32x4 &bv) {
        const size_t no = (size_t)(slot + c) * heads + head;
        const float *lp = left + no * left_step + 4 * lane;
#pragma unroll
        for (int x = 0; x < KT; ++x) av[x] = *(const dc_f32x4 *)(lp + 256 * x);
        bv = *(const dc_f32x4 *)(right + no * right_step + 4 * lane);
    };
    dc_f32x4 s = dc_f32x4{0.f, 0.f, 0.f, 0.f};
    if (of_state) {
        const bool fresh = p.ctx_len[r] - q_len == 0;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (!fresh && row0 + i < dk && col < dv) s[i] = mat[(size_t)(row0 + i) * dv + col];
        *(dc_f32x4 *)(st[0] + l16 * LD + row0) = s;
    }
#pragma unroll
    for (int k = 0; k < AHEAD; ++k)
        if (k < chunks) fetch(k, a[k], b[k]);
    lds_barrier();
    int turn = 0;
    for (int c0 = 0; c0 < chunks; c0 += AHEAD) {
#pragma unroll
        for (int k = 0; k < AHEAD; ++k) {
            const int c = c0 + k;
            if (c >= chunks) break;
            dc_f32x4 old[KT], s2 = dc_f32x4{0.f, 0.f, 0.f, 0.f};
            s = b[k];
#pragma unroll
            for (int x = 0; x < KT; ++x) old[x] = *(const dc_f32x4 *)(st[turn] + l16 * LD + 16 * x + 4 * g);
#pragma unroll
            for (int x = 0; x < KT; x += 2)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    s = __builtin_amdgcn_mfma_f32_16x16x4f32(a[k][x][e], old[x][e], s, 0, 0, 0);
                    s2 = __builtin_amdgcn_mfma_f32_16x16x4f32(a[k][x + 1][e], old[x + 1][e], s2, 0, 0, 0);
                }
            s += s2;
            // the sums stand before any branch: behind one that is taken the compiler (ROCm 7.2) counts too few wait states between a
            // matrix instruction and the first use of its result, and the use reads the value of before
            asm volatile("" : "+v"(s));
            if (c + AHEAD < chunks) fetch(c + AHEAD, a[k], b[k]);
            turn ^= 1;
            if (of_state) {
                *(dc_f32x4 *)(st[turn] + l16 * LD + row0) = s;
            } else if (col < dv) {
                const int t0 = t_first + c * C + row0;
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (t0 + i < t_end) p.o[((size_t)(t0 + i) * heads + head) * dv + col] = s[i];
            }
            lds_barrier();
        }
    }
    if (of_state) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (row0 + i < dk && col < dv) mat[(size_t)(row0 + i) * dv + col] = s[i];
    }
}

template <class T, bool GATED, int DK>
static int delta_chunks_dk(const DeltaChunkArgs &p, int slots, hipStream_t stream) {
    constexpr int bytes = DeltaMapsLds<GATED, DK>::FLOATS * (int)sizeof(float);
    // more than 64 KB of LDS must be asked for once, on every device that runs the kernel
    static std::mutex lock;
    static bool allowed[DELTA_MAX_DEVICES] = {};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= DELTA_MAX_DEVICES) return LCU_UNSUPPORTED;
    {
        std::lock_guard<std::mutex> guard(lock);
        if (!allowed[dev]) {
            const hipError_t e = hipFuncSetAttribute((const void *)delta_maps_kernel<T, GATED, DK>, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
            if (e != hipSuccess) return (int)e;
            allowed[dev] = true;
        }
    }
    delta_maps_kernel<T, GATED, DK><<<dim3(slots, p.heads), dim3(DELTA_CHUNK_THREADS), bytes, stream>>>(p);
    LCU_LAUNCH_CHECK();
    delta_chain_kernel<DK><<<dim3(p.n_req, p.heads, p.tiles), dim3((DK / 16 + DELTA_CHUNK / 16) * WAVE), 0, stream>>>(p);
    LCU_LAUNCH_CHECK();
    return LCU_OK;
}

// The long requests of a step; `work` holds delta_chunk_floats floats.
template <class T, bool GATED>
static int delta_chunks_launch(DeltaChunkArgs p, float *work, int n, hipStream_t stream) {
    const int slots = delta_chunk_slots(n, p.n_req);
    const size_t D = delta_padded(p.dk), all = (size_t)slots * p.heads;
    p.tiles = (p.dv + 15) / 16;
    const size_t V = (size_t)p.tiles * 16;
    p.f = work;
    p.p = p.f + all * D * D;
    p.h = p.p + all * DELTA_CHUNK * D;
    p.q = p.h + all * D * V;
    return D == 64 ? delta_chunks_dk<T, GATED, 64>(p, slots, stream) : delta_chunks_dk<T, GATED, 128>(p, slots, stream);
}
