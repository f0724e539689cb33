#pragma once
#include "common.h"
#include "rows.h"

// A short causal convolution over many tokens: a thread takes four neighbouring channels and a run of tokens, whose rows (and the taps - 1 before
// them) it asks for all at once, so a row is read 11 / 8 times and in pieces of 16 bytes; a thread a token and channel read it once a tap, one
// element at a time and one tap after the other.  One MI355X, us: 2 sets of 2,000 x 2048 32-bit rows, 4 taps, bfloat16 out
// 12 (37); 2,000 rows of 3072 channels, 32-bit out, with silu 17 (37).
constexpr int CONV_RUN = 8, CONV_RUN_THREADS = 256, CONV_RUN_TAPS = 4;
// Steps of four tokens a request and more, and so many tokens in all.  Against a thread a token and channel, us: 100 requests of one token, 2 x 1024
// channels 6.3 (4.7), 64 tokens of one 4.7 (4.7), at 2048 channels 4.8 (7.2).  Up to 512 channels, where a workgroup walks a row in two steps at most, only
// with CONV_RUN_NARROW values or more: 250 tokens of one, 2 x 64 channels, with the state behind it 6.9 (6.0), 2 x 512 7.1 (7.0); 60 single tokens and a prompt
// of 300 9.3 (8.3), 2 x 1024 10.9 (11.4); 2,000 of one, 2 x 512 8.0 (16.1).
constexpr int CONV_RUN_TOKENS = 64, CONV_RUN_A_REQUEST = 4, CONV_RUN_NARROW = 1 << 19;

// h: the step's first row at the thread's first channel.  emit(k, window, pos, fresh): token k of the run, at position pos of its request, whose
// first row of the step is its first at all if fresh;
// window[j] its taps' rows, oldest first: rows of the step, and before the request's first one state_rows(slot)'s TAPS - 1 rows (d apart).
template <int TAPS, class TI, class STATE, class EMIT>
__device__ __forceinline__ void conv_run(const TI *__restrict__ h, size_t stride, int t0, int count, const int *__restrict__ req_of_token, const int *__restrict__ q_start,
                                         const int *__restrict__ ctx_len, const int *__restrict__ state_slot, size_t d, STATE state_rows, EMIT emit) {
    float row[CONV_RUN + TAPS - 1][4];
#pragma unroll
    for (int k = 0; k < CONV_RUN + TAPS - 1; ++k) load_as_f32<TI, 4>(h + max(t0 - (TAPS - 1) + min(k, count + TAPS - 2), 0) * stride, row[k]);
    // what is looked up is the same for the whole workgroup, the eight tokens' at once
    int r[CONV_RUN], first[CONV_RUN], pos[CONV_RUN], slot[CONV_RUN];
#pragma unroll
    for (int k = 0; k < CONV_RUN; ++k) r[k] = req_of_token[t0 + min(k, count - 1)];
#pragma unroll
    for (int k = 0; k < CONV_RUN; ++k) {
        first[k] = q_start[r[k]];
        pos[k] = ctx_len[r[k]] - (q_start[r[k] + 1] - (t0 + k));
        slot[k] = state_slot[r[k]];
    }
    // four tokens at a time: what their windows want of requests' states is asked for before the first of them is made, so single tokens side by side are
    // two trips to memory and not eight (60 of them and a prompt of 300, 2 x 1024 channels, with the states behind it: 10.9 us, one by one 12.0)
    constexpr int SIDE = 4;
#pragma unroll
    for (int k0 = 0; k0 < CONV_RUN; k0 += SIDE) {
        if (k0 >= count) break;
        float old[SIDE][TAPS - 1][4];
#pragma unroll
        for (int b = 0; b < SIDE; ++b) {
            const int k = k0 + b, into = t0 + k - first[k];      // rows of the request before this one (looked up for the run's last token where there are fewer)
            if (into >= TAPS - 1) continue;
            const float *st = state_rows(slot[k]);
#pragma unroll
            for (int j = 0; j < TAPS - 1; ++j) load_as_f32<float, 4>(st + min(j + into, TAPS - 2) * d, old[b][j]);
        }
#pragma unroll
        for (int b = 0; b < SIDE; ++b) {
            const int k = k0 + b, into = t0 + k - first[k];
            if (k >= count) break;
            if (into >= TAPS - 1) emit(k, &row[k], pos[k], pos[k] == into);
            else {
                float window[TAPS][4];
#pragma unroll
                for (int j = 0; j < TAPS; ++j)
#pragma unroll
                    for (int e = 0; e < 4; ++e) window[j][e] = j + into >= TAPS - 1 || j == TAPS - 1 ? row[k + j][e] : old[b][min(j, TAPS - 2)][e];
                emit(k, window, pos[k], pos[k] == into);
            }
        }
    }
}
