// The delta rules over portions of many tokens: chunks of 64 tokens side by side on the 64-bit matrix instruction.
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
// channel; a chunk is one of 3.6 us.  2,048 tokens of one request, 16 heads of 128, the whole rule with its preparation and output kernels:
// gated 1,170 us scanned, 255 in chunks; with decays per channel 2,420 scanned, 320 in chunks (with 32-bit products 175 and 225, and a larger error,
// below).
//
// What bounds them: `maps` runs 4,300 (channel-wise 6,300) matrix instructions of 64 cycles a chunk and head, 28 (42) us on a compute
// unit's four SIMDs; one workgroup of 8 waves fits a compute unit beside its LDS (560 of them, 2,014 tokens of four requests, channel-wise, are three rounds: 220 us, and 241
// while the vectors and values were asked for a few at a time, each under a condition, and so awaited in turn).  `chain` is its 96 matrix
// instructions a SIMD and chunk (2.6 us) and the round through LDS; the affine form costs `maps` a third more products than c, o and S
// in turn would, but leaves one product instead of two, one after the other, on the chain.
//
// The decays per channel are at least exp(-exp(-1/2)) = 0.545 a token, so G over a chunk stays above 1e-17 and 1 / G below 1e17: the
// products u~_t k~_s are of the size of u_t k_s again and lose nothing (a quotient of two rounded numbers).  The gated rule's one decay
// may be as small as it likes: there the products u k^T and r k^T are weighted by exp(L_t - L_s) <= 1, L the sums of log g in 64-bit.
//
// A chunk multiplies what is not yet there by zeros (the triangles' other halves, tokens beyond the end), which an infinity or NaN does not
// forgive: it would reach the tokens before it.  So a chunk in which something is not finite, or so large (DELTA_TAME) that a product might not be, is
// marked by `maps`, and `chain` walks the tokens of that head and request one by one.
//
// Products and sums are 64-bit (v_mfma_f64_16x16x4_f64, half the rate of the 32-bit instruction), what is held between them is 32-bit, but for
// the state on its way along the chain: one rounding each of u~, r~, k~, al~, the masked matrices and the maps.  Sums of 64 and 128 terms in
// 32 bits, one after the other, would be 2 to 3e-7 off where decays are fast and the scan, whose lanes add in a tree, is only 1e-7 off.
// Measured over 640 tokens of 2 heads of 128 (relative, 2-norm, against 64 bits, scan / chunks), per channel,
// from decays of 0.98 to 0.55 a token: outputs 6.7e-7 / 6.2e-7 to 1.4e-7 / 1.0e-7, states 1.5e-6 / 1.5e-6 to 4.4e-8 / 4.6e-8; gated, decays of
// 0.9999 to 0.05: outputs 6.6e-7 / 1.2e-7 to 1.5e-7 / 1.0e-7, states 1.4e-6 / 1.0e-7 to 7.7e-8 / 6.8e-8.
// In the instruction's operands lane (l, g) of 16 x 4 holds row (or column) l and index g of the summed four, in its results column l and
// rows g, g + 4, g + 8, g + 12.  Step e of a tile of 16 therefore takes the indexes 4 e + g, so that results are the next product's operand as
// they are; in LDS and in the maps the sixteen stand so that a lane's four are neighbours (dc_place).
#pragma once
#include <limits.h>
#include <math.h>
#include <mutex>
#include "common.h"
#include "lane_moves.h"

constexpr int DELTA_CHUNK = 64;
constexpr int DELTA_CHUNK_THREADS = 512;
constexpr int DELTA_LDM = DELTA_CHUNK + 4;       // rows of a [64][64] matrix in LDS
constexpr int DELTA_MAX_DEVICES = 16;
constexpr float DELTA_TAME = 1e12f;              // vectors up to here: products of two, times 1 / G, stay below 1e42 in 64 bits, F and H below 1e28
__device__ __forceinline__ bool dc_wild(float x) { return !(fabsf(x) <= DELTA_TAME); }
__device__ __forceinline__ bool dc_wild(float4 v) { return dc_wild(v.x) || dc_wild(v.y) || dc_wild(v.z) || dc_wild(v.w); }

typedef __attribute__((ext_vector_type(4))) float dc_f32x4;
typedef __attribute__((ext_vector_type(4))) double dc_f64x4;

// Which requests of a step go through chunks: those that feed `line` tokens or more, if all of those take less time so.  The times, in ns, of
// what is measured: a scan is the longest request's chain, and the work of all tokens and heads where they fill the card; chunks are two launches,
// the longest request's chain, and the work of all chunks and heads (a chunk that is cut short counts whole).  Chunks must be faster by a fifth.
// One MI355X, the whole rule, gated heads of 128 / 64 / 16 and per-channel ones, us scanned / in chunks: 16 heads, one request of 130 tokens 82 / 77, 71 / 45 (of 64), 100 /
// 77 (160 tokens); 16 requests of 130 tokens 269 / 371, 8 of 256 340 / 238.  Over 2,130 steps of 1 to 32 requests of 64 to 2,000 tokens, 4 to 64 heads of 16 to 128, this rule
// takes 0.69 of the scan's time (the better one of the two 0.67) and 1.05 at the worst; by the number of tokens alone, 128, and of requests it took 0.70 and 2.2.
// Head sizes for which the scan keeps the state in memory (10 us a token; 40: 646 / 36) go there from 64 tokens on.
struct DeltaLine {
    int line;                                    // INT_MAX: everything is scanned
    int scan, scan_longest, scan_token;          // ns: a step, a token of the longest request, a token
    int chunked, chunked_longest, chunk;
    __host__ __device__ bool chunks_pay(int longest, int tokens, int chunks) const {
        const long long a = scan + (long long)scan_longest * longest + (long long)scan_token * tokens;
        const long long b = chunked + (long long)chunked_longest * ((longest + 63) / 64) + (long long)chunk * chunks;
        return longest >= line && 6 * b < 5 * a;
    }
    // what holds for a step: the least tokens that a request must feed (called by whole waves; sums of less than 2^24, exact in 32-bit)
    __device__ __forceinline__ int of_step(const int *__restrict__ q_start, int n_req) const {
        const int lane = threadIdx.x % WAVE;
        float longest = 0.f, tokens = 0.f, chunks = 0.f;
        for (int r = lane; r < n_req; r += WAVE) {
            const int len = q_start[r + 1] - q_start[r];
            if (len < line) continue;
            longest = fmaxf(longest, (float)len);
            tokens += (float)len;
            chunks += (float)((len + 63) / 64);
        }
        return chunks_pay((int)wave_max_in_place(longest), (int)wave_sum_in_place(tokens), (int)wave_sum_in_place(chunks)) ? line : INT_MAX;
    }
};
inline DeltaLine delta_line(int heads, int dk, int dv, bool gated) {
    const double wide = (double)dv / dk, sq = (double)dk * dk;               // (the work of a token grows with both sizes)
    auto times = [&](double x) { return (int)fmin(x, 1e9); };
    DeltaLine l = {};
    l.line = 64;
    l.scan = 9000;
    l.scan_longest = dk % 16 ? 10000 : times(gated ? 290 + 1.2 * dk : 470 + 2.1 * dk);         // (else the scan has the state in registers)
    l.scan_token = times(heads * wide * (gated ? 0.7 + 2.6e-4 * sq : 0.6 + 9e-4 * sq));
    const bool half = dk <= 64;
    l.chunked = gated ? (half ? 34000 : 54000) : (half ? 38000 : 72000);
    l.chunked_longest = gated ? (half ? 800 : 900) : (half ? 700 : 800);
    l.chunk = times(heads * (0.5 + 0.5 * wide) * (gated ? (half ? 165 : 350) : (half ? 190 : 460)));
    return l;
}

struct DeltaChunkArgs {
    const float *prep;                           // [n, heads, 5 dk] (w | al | u | k | r) or, gated, [n, heads, 2 dk + 4] (u | r | g, beta g, log g, 0)
    const void *proj;                            // the values: columns off_v of rows [n, row_stride] of T, or vf [n, heads * dv] if not null
    int row_stride, off_v;
    const float *vf;
    float *f, *h, *p, *q;                        // [slot][head] of [DK][DK], [DK][16 tiles], [64][DK], [64][16 tiles], in tiles of 16 x 16: F
                                                 // and P as left operands [row tile][index tile], H and Q as results [column tile][row tile]
    int *wild;                                   // [slot][head]: whether the chunk must be walked token by token
    int *done;                                   // [request]: whether it went through chunks
    int gated, bf16;                             // the form of prep; the type of proj
    float *state;
    size_t slot_stride;
    float *o;                                    // [n, heads * dv]
    const int *q_start, *ctx_len, *state_slot;
    int n_req, heads, dk, dv, tiles;             // tiles: of 16 value columns
    DeltaLine line;
};

// The chunks that a step of n tokens in n_req requests can have: every long request's last one may be cut short.
__host__ __device__ inline int delta_chunk_slots(int n, int n_req, int line) {
    const int most = n / line;
    return n / DELTA_CHUNK + (most < n_req ? most : n_req);
}
// Whether a step may hold a long request (every request feeds a token at least).
inline bool delta_chunks_possible(int n, int n_req, int dk, int line) { return dk <= 128 && n - n_req + 1 >= line; }
inline int delta_padded(int dk) { return dk <= 64 ? 64 : 128; }
inline size_t delta_chunk_floats(int n, int n_req, int heads, int dk, int dv, bool gated) {
    const int line = delta_line(heads, dk, dv, gated).line;
    if (!delta_chunks_possible(n, n_req, dk, line)) return 0;
    const size_t D = delta_padded(dk), V = (size_t)(dv + 15) / 16 * 16;
    return (size_t)delta_chunk_slots(n, n_req, line) * heads * (D * D + D * V + DELTA_CHUNK * (D + V) + 1) + n_req;
}

// Where in `work` the kernels leave which requests went through chunks.
inline const int *delta_done(const float *work, int n, int n_req, int heads, int dk, int dv, bool gated) {
    return (const int *)work + delta_chunk_floats(n, n_req, heads, dk, dv, gated) - n_req;
}

__device__ __forceinline__ dc_f64x4 dc_mma(float4 a, dc_f64x4 b, dc_f64x4 c) {
    c = __builtin_amdgcn_mfma_f64_16x16x4f64((double)a.x, b[0], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f64_16x16x4f64((double)a.y, b[1], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f64_16x16x4f64((double)a.z, b[2], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f64_16x16x4f64((double)a.w, b[3], c, 0, 0, 0);
    return c;
}
// The place of index k of a tile of sixteen among them: a lane's 4 e + g are neighbours.  (The places' indexes are found the same way.)
__device__ __forceinline__ int dc_place(int k) { return (k & ~15) + k % 4 * 4 + k % 16 / 4; }
// Where element (row m, index k) of a tile of 16 x 16 stands in memory: in the order in which a wave's lanes take the tile as the left
// operand, so that the wave reads whole lines.
__device__ __forceinline__ int dc_operand(int tile, int m, int k) { return (tile * WAVE + k % 4 * 16 + m) * 4 + k / 4; }
// Keeps the compiler from holding what it reads from LDS here in registers until it is read again later: that would spill.
__device__ __forceinline__ void dc_forget() { asm volatile("" ::: "memory"); }
__device__ __forceinline__ dc_f64x4 dc_vec(float4 v) { return dc_f64x4{v.x, v.y, v.z, v.w}; }
__device__ __forceinline__ dc_f32x4 dc_round(dc_f64x4 v) { return dc_f32x4{(float)v[0], (float)v[1], (float)v[2], (float)v[3]}; }
__device__ __forceinline__ dc_f64x4 dc_zero() { return dc_f64x4{0.0, 0.0, 0.0, 0.0}; }

// LDS of `maps`, in floats: the channel-wise rule holds four [64][DK + 4] arrays, of which the first two make room for the four
// [64][68] matrices; the gated rule two of each.
template <bool GATED, int DK> struct DeltaMapsLds {
    static constexpr int LD = DK + 4, ROWS = DELTA_CHUNK * LD, MAT = DELTA_CHUNK * DELTA_LDM;
    static constexpr int FRONT = GATED ? ROWS : (2 * ROWS > 4 * MAT ? 2 * ROWS : 4 * MAT);      // (gated: u stays)
    static constexpr int REST = GATED ? ROWS + 2 * MAT : 2 * ROWS;
    static constexpr int DINV = 4 * 16 * 20;
    static constexpr int SMALL = 448 + 2 * DK;    // gated: the sums of log g in two parts, beta g, weights in 64 bits; G_C in 64 bits
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
    float *dinv = dc_lds + L::FRONT + L::REST, *small = dinv + L::DINV;
    double *g_all = (double *)small, *w_end = g_all + DK, *w_start = w_end + C;       // by key and by token; g_all and w_end by place
    float *l_hi = (float *)(w_start + C), *l_lo = l_hi + C, *bg = l_lo + C;           // gated, by token, bg by place
    static_assert((L::FRONT + L::REST + L::DINV) % 2 == 0, "64-bit numbers stand at even places");
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, g = lane >> 4, l16 = lane & 15, head = blockIdx.y;
    // ---- which request's chunk this is
    int t0 = 0, nt = 0;
    {
        const int line = p.line.of_step(p.q_start, p.n_req);
        int left = blockIdx.x;
        for (int r = 0; r < p.n_req; ++r) {
            const int a = p.q_start[r], b = p.q_start[r + 1], len = b - a;
            if (len < line) continue;
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
    bool wild = false;
    // ---- the tokens' vectors
    if constexpr (GATED) {
        const int row = 2 * dk + 4;
        if (wave == 0) {
            const float *s = p.prep + ((size_t)(t0 + min(lane, nt - 1)) * heads + head) * row + 2 * dk;
            double l = lane < nt ? (double)fmaxf(s[2], -1e4f) : 0.0;          // (a decay of exp(-1e4) is 0 like any smaller one)
            const float b = lane < nt ? s[1] : 0.f;
            wild |= !(s[2] <= 0.f) || dc_wild(s[1]);
#pragma unroll
            for (int off = 1; off < C; off <<= 1) {
                const double before = __shfl_up(l, off, WAVE);
                if (lane >= off) l += before;
            }
            const float hi = (float)l, lo = (float)(l - (double)hi);
            l_hi[lane] = hi;
            l_lo[lane] = lo;
            bg[dc_place(lane)] = b;
            w_end[dc_place(lane)] = exp(__shfl(l, C - 1, WAVE) - l);
            w_start[lane] = exp(l);
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
            wild |= dc_wild(u) || dc_wild(r);
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
        float w[PER], al[PER], u[PER], k[PER], r[PER];                        // (all asked for before the first is used, and under no condition)
#pragma unroll
        for (int e = 0; e < PER; ++e) w[e] = s[(size_t)min(grp * PER + e, nt - 1) * heads * row];
#pragma unroll
        for (int e = 0; e < PER; ++e) {
            const float *x = s + (size_t)min(grp * PER + e, nt - 1) * heads * row;
            al[e] = x[dk];
            u[e] = x[2 * dk];
            k[e] = x[3 * dk];
            r[e] = x[4 * dk];
        }
        double own = 1.0;
#pragma unroll
        for (int e = 0; e < PER; ++e) {
            const int t = grp * PER + e;
            if (t >= nt || c >= dk) w[e] = 1.f;
            wild |= !(w[e] >= 0.5f && w[e] <= 1.f);
            own *= (double)w[e];
        }
        part[grp * DK + c] = own;
        __syncthreads();
        double before = 1.0;
        for (int x = 0; x < grp; ++x) before *= part[x * DK + c];
#pragma unroll
        for (int e = 0; e < PER; ++e) {
            const int t = grp * PER + e;
            if (t >= nt || c >= dk) al[e] = u[e] = k[e] = r[e] = 0.f;
            wild |= dc_wild(make_float4(al[e], u[e], k[e], r[e]));
            us[t * LD + c] = (float)(u[e] * before);
            before *= (double)w[e];
            const double inv = 1.0 / before;
            rs[t * LD + c] = (float)(r[e] * before);
            ks[t * LD + c] = (float)(k[e] * inv);
            as[t * LD + c] = (float)(al[e] * inv);
        }
        if (grp == GROUPS - 1) g_all[dc_place(c)] = before;
    }
    __syncthreads();
    // ---- the matrices: waves 0 to 3 a tile of 16 rows of u's, waves 4 to 7 of r's (the longest strips beside the shortest on a SIMD)
    {
        const bool of_r = wave >= 4;
        const int a = of_r ? 3 - (wave & 3) : wave & 3;
        const float *left = of_r ? rs : us;
        dc_f64x4 k4[4], a4[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) k4[c] = a4[c] = dc_zero();
        for (int x = 0; x < KT; ++x) {
            const dc_f64x4 b = dc_vec(*(const float4 *)(left + (16 * a + l16) * LD + 16 * x + 4 * g));
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                if (c > a) continue;
                const int at = (16 * c + l16) * LD + 16 * x + 4 * g;
                k4[c] = dc_mma(*(const float4 *)((GATED ? us : ks) + at), b, k4[c]);
                if constexpr (!GATED) a4[c] = dc_mma(*(const float4 *)(as + at), b, a4[c]);
            }
        }
        // this lane's results: token t (of the strip), tokens 16 c + 4 i + g
        const int t = 16 * a + l16;
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int s = 16 * c + 4 * i + g;
                const bool in = of_r ? s <= t : s < t;
                if constexpr (GATED) {
                    const int from = of_r ? t : max(t - 1, 0);
                    k4[c][i] = in ? k4[c][i] * (double)expf((l_hi[from] - l_hi[s]) + (l_lo[from] - l_lo[s])) : 0.0;
                } else {
                    k4[c][i] = in ? k4[c][i] : 0.0;
                    a4[c][i] = in ? a4[c][i] : 0.0;
                }
            }
        // (channel-wise) u~ and r~ make room: what the column tiles still need of them goes to registers, below
        dc_f64x4 um[4], rm[4];
        if (wave < KT) {
#pragma unroll
            for (int b = 0; b < 4; ++b)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int s = 16 * b + 4 * i + g;
                    um[b][i] = us[s * LD + 16 * wave + l16];
                    rm[b][i] = rs[s * LD + 16 * wave + l16];
                    if constexpr (GATED) {
                        um[b][i] *= s > 0 ? w_start[s - 1] : 1.0;
                        rm[b][i] *= w_start[s];
                    }
                }
        }
        if constexpr (!GATED) __syncthreads();
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            if (c > a) continue;
            *(dc_f32x4 *)((of_r ? m_rk : m_uk) + t * LDM + 16 * c + 4 * g) = dc_round(k4[c]);
            if constexpr (!GATED) *(dc_f32x4 *)((of_r ? m_ra : m_ua) + t * LDM + 16 * c + 4 * g) = dc_round(a4[c]);
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
            double col[16];
            col[0] = lane == 0 ? 1.0 : 0.0;
            dinv[16 * wave * 20 + dc_place(lane)] = (float)col[0];
#pragma unroll
            for (int i = 1; i < 16; ++i) {
                double row[16];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    row[j] = next[j].x; row[4 + j] = next[j].y; row[8 + j] = next[j].z; row[12 + j] = next[j].w;
                    if constexpr (GATED) { row[j] *= bgs[j].x; row[4 + j] *= bgs[j].y; row[8 + j] *= bgs[j].z; row[12 + j] *= bgs[j].w; }
                    if (i < 15) next[j] = *(const float4 *)(m + (i + 1) * LDM + 4 * j);
                }
                double v = i == lane ? 1.0 : 0.0;
#pragma unroll
                for (int j = 0; j < i; ++j) v -= row[j] * col[j];
                col[i] = v;
                dinv[(16 * wave + i) * 20 + dc_place(lane)] = (float)v;
            }
        }
        __syncthreads();
        // X = T B for 16 columns: lane (l, g) holds rows 16 a + 4 i + g of column l
        auto solve = [&](dc_f64x4 *x) {
            dc_f64x4 bx[4];
            dc_forget();
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                dc_f64x4 sum = dc_zero();
#pragma unroll
                for (int c = 0; c < b; ++c) sum = dc_mma(*(const float4 *)((GATED ? m_uk : m_ua) + (16 * b + l16) * LDM + 16 * c + 4 * g), bx[c], sum);
                x[b] -= sum;
                x[b] = dc_mma(*(const float4 *)(dinv + (16 * b + l16) * 20 + 4 * g), x[b], dc_zero());
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
                dc_f64x4 sum = dc_zero();
#pragma unroll
                for (int c = 0; c <= b; ++c) sum = dc_mma(*(const float4 *)((GATED ? m_rk : m_ra) + (16 * b + l16) * LDM + 16 * c + 4 * g), um[c], sum);
#pragma unroll
                for (int i = 0; i < 4; ++i) pp[dc_operand(b * KT + wave, 4 * i + g, l16)] = (float)(rm[b][i] - sum[i]);
            }
            if constexpr (GATED) {
#pragma unroll
                for (int b = 0; b < 4; ++b) um[b] *= *(const dc_f64x4 *)(w_end + 16 * b + 4 * g);
            }
#pragma unroll 4
            for (int y = 0; y < KT; ++y) {
                dc_forget();
                dc_f64x4 sum = dc_zero();
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    const float *at = (GATED ? us : as) + (16 * b + g) * LD + 16 * y + l16;
                    sum = dc_mma(make_float4(at[0], at[4 * LD], at[8 * LD], at[12 * LD]), um[b], sum);
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const double one = 16 * y + 4 * i + g == 16 * wave + l16 ? 1.0 : 0.0;
                    ff[dc_operand(y * KT + wave, 4 * i + g, l16)] = (float)(GATED ? one * w_start[C - 1] - sum[i] : g_all[16 * y + 4 * g + i] * (one - sum[i]));
                }
            }
        }
        // ---- columns of N, and with them of Q and H
        const int width = p.tiles * 16;
        for (int tile = wave; tile < p.tiles; tile += WAVES) {
            float *qq = p.q + no * C * width, *hh = p.h + no * DK * width;
            const int col = tile * 16 + l16;
            dc_f64x4 v[4], x[4];
            dc_forget();
            const int cc = head * dv + min(col, dv - 1);
            float value[16];                                                  // all asked for before the first is used: the choice of where from stands outside
            if (p.vf) {
#pragma unroll
                for (int e = 0; e < 16; ++e) value[e] = p.vf[(size_t)(t0 + min(4 * e + g, nt - 1)) * heads * dv + cc];
            } else {
                T raw[16];
#pragma unroll
                for (int e = 0; e < 16; ++e) raw[e] = ((const T *)p.proj)[(size_t)(t0 + min(4 * e + g, nt - 1)) * p.row_stride + p.off_v + cc];
#pragma unroll
                for (int e = 0; e < 16; ++e) value[e] = to_f32(raw[e]);
            }
#pragma unroll
            for (int b = 0; b < 4; ++b)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const bool in = 16 * b + 4 * i + g < nt && col < dv;
                    v[b][i] = in ? (double)value[4 * b + i] : 0.0;
                    wild |= in && dc_wild(value[4 * b + i]);
                }
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                x[b] = dc_zero();
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
                dc_f64x4 sum = dc_zero();
#pragma unroll
                for (int c = 0; c <= b; ++c) {
                    const int at = (16 * b + l16) * LDM + 16 * c + 4 * g;
                    sum = dc_mma(*(const float4 *)(m_rk + at), v[c], sum);
                    if constexpr (!GATED) sum = dc_mma(*(const float4 *)(m_ra + at), x[c], sum);
                }
                *(dc_f32x4 *)(qq + ((size_t)(tile * (C / 16) + b) * WAVE + lane) * 4) = dc_round(sum);
            }
            if constexpr (GATED) {
#pragma unroll
                for (int b = 0; b < 4; ++b) v[b] *= *(const dc_f64x4 *)(w_end + 16 * b + 4 * g);
            }
#pragma unroll 4
            for (int y = 0; y < KT; ++y) {
                dc_forget();
                dc_f64x4 sum = dc_zero();
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    const int at = (16 * b + g) * LD + 16 * y + l16;
                    const float *kp = (GATED ? us : ks) + at;
                    sum = dc_mma(make_float4(kp[0], kp[4 * LD], kp[8 * LD], kp[12 * LD]), v[b], sum);
                    if constexpr (!GATED) sum = dc_mma(make_float4(as[at], as[at + 4 * LD], as[at + 8 * LD], as[at + 12 * LD]), x[b], sum);
                }
                if constexpr (!GATED) sum *= *(const dc_f64x4 *)(g_all + 16 * y + 4 * g);
                *(dc_f32x4 *)(hh + ((size_t)(tile * KT + y) * WAVE + lane) * 4) = dc_round(sum);
            }
        }
    }
    wild = __syncthreads_or(wild);
    if (tid == 0) p.wild[no] = wild;
}

// The tokens t0 .. t1 - 1 of a request one by one (delta_rule.hip's recurrence), for 16 value columns: 256 threads, 16 a column with KT key
// channels each.
template <int KT>
__device__ __forceinline__ void delta_walk(const DeltaChunkArgs &p, float *mat, bool fresh, int t0, int t1, int head, int col, int part) {
    const int dk = p.dk, dv = p.dv, i0 = part * KT, cc = head * dv + min(col, dv - 1);
    float s[KT];
#pragma unroll
    for (int i = 0; i < KT; ++i) s[i] = !fresh && i0 + i < dk && col < dv ? mat[(size_t)(i0 + i) * dv + col] : 0.f;
    for (int t = t0; t < t1; ++t) {
        const float *row = p.prep + ((size_t)t * p.heads + head) * (p.gated ? 2 * dk + 4 : 5 * dk);
        const float v = p.vf ? p.vf[(size_t)t * p.heads * dv + cc] : p.bf16 ? to_f32(((const bf16_t *)p.proj)[(size_t)t * p.row_stride + p.off_v + cc])
                                                                            : ((const float *)p.proj)[(size_t)t * p.row_stride + p.off_v + cc];
        const float g = p.gated ? row[2 * dk] : 1.f, bg = p.gated ? row[2 * dk + 1] : 1.f;
        float u[KT], c = 0.f, o = 0.f;
#pragma unroll
        for (int i = 0; i < KT; ++i) {
            u[i] = i0 + i < dk ? row[(p.gated ? 0 : 2 * dk) + i0 + i] : 0.f;
            c += u[i] * s[i];
        }
        c = sum_over_16(c);
#pragma unroll
        for (int i = 0; i < KT; ++i) {
            if (i0 + i >= dk) continue;
            if (p.gated) s[i] = g * s[i] + u[i] * (v - bg * c);
            else s[i] = row[i0 + i] * s[i] - row[dk + i0 + i] * c + row[3 * dk + i0 + i] * v;
            o += row[(p.gated ? dk : 4 * dk) + i0 + i] * s[i];
        }
        o = sum_over_16(o);
        if (part == 0 && col < dv) p.o[((size_t)t * p.heads + head) * dv + col] = o;
    }
#pragma unroll
    for (int i = 0; i < KT; ++i)
        if (i0 + i < dk && col < dv) mat[(size_t)(i0 + i) * dv + col] = s[i];
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
    __shared__ __attribute__((aligned(16))) double st[2][16 * LD];            // S of these columns, a column a row, by place
    const int r = blockIdx.x, head = blockIdx.y, tile = blockIdx.z;
    const int t_first = p.q_start[r], t_end = p.q_start[r + 1], q_len = t_end - t_first;
    const int line = p.line.of_step(p.q_start, p.n_req);
    if (head == 0 && tile == 0 && threadIdx.x == 0) p.done[r] = q_len >= line;
    if (q_len < line) return;
    int slot = 0;
    for (int x = 0; x < r; ++x) {
        const int len = p.q_start[x + 1] - p.q_start[x];
        if (len >= line) slot += (len + C - 1) / C;
    }
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), g = lane >> 4, l16 = lane & 15;
    const int dk = p.dk, dv = p.dv, heads = p.heads, width = p.tiles * 16, col = tile * 16 + l16;
    float *mat = p.state + (size_t)p.state_slot[r] * p.slot_stride + (size_t)head * dk * dv;
    const bool of_state = wave < KT;
    const int y = of_state ? wave : wave - KT, row0 = 16 * y + g;             // this wave's rows row0 + 4 i: key channels, or the chunk's tokens
    // the wave's rows of the maps of chunk number `slot + c`
    const float *left = of_state ? p.f + (size_t)y * KT * 256 : p.p + (size_t)y * KT * 256;
    const float *right = of_state ? p.h + (size_t)(tile * KT + y) * 256 : p.q + (size_t)(tile * (C / 16) + y) * 256;
    const size_t left_step = of_state ? DK * DK : C * DK, right_step = (size_t)(of_state ? DK : C) * width;
    const int chunks = (q_len + C - 1) / C;
    const bool fresh = p.ctx_len[r] - q_len == 0;
    bool wild = false;
    for (int c = tid; c < chunks; c += blockDim.x) wild |= p.wild[(size_t)(slot + c) * heads + head] != 0;
    if (__syncthreads_or(wild)) {
        if (tid < 256) delta_walk<KT>(p, mat, fresh, t_first, t_end, head, tile * 16 + tid / 16, tid % 16);
        return;
    }
    dc_f32x4 a[AHEAD][KT], b[AHEAD];
    auto fetch = [&](int c, dc_f32x4 *av, dc_f32x4 &bv) {
        const size_t no = (size_t)(slot + c) * heads + head;
        const float *lp = left + no * left_step + 4 * lane;
#pragma unroll
        for (int x = 0; x < KT; ++x) av[x] = *(const dc_f32x4 *)(lp + 256 * x);
        bv = *(const dc_f32x4 *)(right + no * right_step + 4 * lane);
    };
    dc_f64x4 s = dc_zero();
    if (of_state) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (!fresh && row0 + 4 * i < dk && col < dv) s[i] = mat[(size_t)(row0 + 4 * i) * dv + col];
        *(dc_f64x4 *)(st[0] + l16 * LD + 16 * y + 4 * g) = s;
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
            dc_f64x4 s2 = dc_zero();
            s = dc_f64x4{b[k][0], b[k][1], b[k][2], b[k][3]};
#pragma unroll
            for (int x = 0; x < KT; x += 2) {
                const dc_f64x4 old = *(const dc_f64x4 *)(st[turn] + l16 * LD + 16 * x + 4 * g);
                const dc_f64x4 old2 = *(const dc_f64x4 *)(st[turn] + l16 * LD + 16 * x + 16 + 4 * g);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    s = __builtin_amdgcn_mfma_f64_16x16x4f64((double)a[k][x][e], old[e], s, 0, 0, 0);
                    s2 = __builtin_amdgcn_mfma_f64_16x16x4f64((double)a[k][x + 1][e], old2[e], s2, 0, 0, 0);
                }
            }
            s += s2;
            // the sums stand before any branch: behind the one over the next loads the compiler (ROCm 7.2) has left too few wait states where it is
            // taken (3 of 10, with sums in 32 bits; it counted the instructions that the branch passes by), and the use read the value
            // of before.  What holds for every kernel, that no use comes too early on any way, a test reads from the built instructions
            asm volatile("" : "+v"(s));
            if (c + AHEAD < chunks) fetch(c + AHEAD, a[k], b[k]);
            turn ^= 1;
            if (of_state) {
                *(dc_f64x4 *)(st[turn] + l16 * LD + 16 * y + 4 * g) = s;
            } else if (col < dv) {
                const int t0 = t_first + c * C + row0;
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (t0 + 4 * i < t_end) p.o[((size_t)(t0 + 4 * i) * heads + head) * dv + col] = (float)s[i];
            }
            lds_barrier();
        }
    }
    if (of_state) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (row0 + 4 * i < dk && col < dv) mat[(size_t)(row0 + 4 * i) * dv + col] = (float)s[i];
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
    const int slots = delta_chunk_slots(n, p.n_req, p.line.line);
    const size_t D = delta_padded(p.dk), all = (size_t)slots * p.heads;
    p.tiles = (p.dv + 15) / 16;
    const size_t V = (size_t)p.tiles * 16;
    p.f = work;
    p.p = p.f + all * D * D;
    p.h = p.p + all * DELTA_CHUNK * D;
    p.q = p.h + all * D * V;
    p.wild = (int *)(p.q + all * DELTA_CHUNK * V);
    p.done = p.wild + all;
    p.gated = GATED;
    p.bf16 = sizeof(T) == 2;
    return D == 64 ? delta_chunks_dk<T, GATED, 64>(p, slots, stream) : delta_chunks_dk<T, GATED, 128>(p, slots, stream);
}
