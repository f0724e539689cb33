#pragma once
#include "common.h"
#include "kv_layout.h"

// Where the q, k, v product of an attention layer puts what it makes: the rotated queries in rows of their own, the rotated keys and the values
// in the token's place of its page.
struct QkvStore {
    const int *positions;        // [M]
    const int *slots;            // [M] page * page_size + place, negative or slots null: nothing is stored
    const float *cos_t, *sin_t;  // [max_pos, head_dim / 2]; pairs are (i, i + head_dim / 2)
    int max_pos;
    bf16_t *cache;               // this layer's pages
    bf16_t *q_out;               // [M, heads * head_dim] rows ldq apart
    int ldq;
    int heads, kv_heads, head_dim, page;
};

// Dims i0 .. i0 + 3 and head_dim/2 + i0 .. of one head (the q heads first, then k, then v) of token tok: rounded to bfloat16 before the
// rotation, as a plain product stores them for the rotation kernel, so a token's query and key are made the same way whichever kernel makes them.
__device__ __forceinline__ void qkv_store(const QkvStore &s, int head, int tok, int i0, const float (&lo)[4], const float (&hi)[4]) {
    const int half_dim = s.head_dim / 2;
    const bool is_q = head < s.heads, is_k = !is_q && head < s.heads + s.kv_heads;
    const int pos = s.positions[tok];
    const bool in_table = pos >= 0 && pos < s.max_pos;
    const int slot = s.slots ? s.slots[tok] : -1;
    bf16_t *pg = nullptr;
    int place = 0;
    if (!is_q && slot >= 0) {
        pg = s.cache + (size_t)(slot / s.page) * kv_page_elems(s.kv_heads, s.head_dim, s.page);
        place = slot % s.page;
    }
    bf16_t va[4], vb[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        float a = to_f32(from_f32<bf16_t>(lo[r])), b = to_f32(from_f32<bf16_t>(hi[r]));
        if (is_q || is_k) {
            float cs = __uint_as_float(0x7fc00000u), sn = cs;         // a position outside the table gives NaN
            if (in_table) { cs = s.cos_t[(size_t)pos * half_dim + i0 + r]; sn = s.sin_t[(size_t)pos * half_dim + i0 + r]; }
            float ra, rb;
            rotate_pair(a, b, cs, sn, ra, rb);
            a = ra; b = rb;
        }
        va[r] = from_f32<bf16_t>(a);
        vb[r] = from_f32<bf16_t>(b);
    }
    if (is_q) {
        bf16_t *qo = s.q_out + (size_t)tok * s.ldq + (size_t)head * s.head_dim;
#pragma unroll
        for (int r = 0; r < 4; ++r) { qo[i0 + r] = va[r]; qo[i0 + half_dim + r] = vb[r]; }
    } else if (pg) {
        if (is_k) {
            const int kvh = head - s.heads;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                pg[kv_key_offset(kvh, place, i0 + r, s.head_dim, s.page)] = va[r];
                pg[kv_key_offset(kvh, place, i0 + half_dim + r, s.head_dim, s.page)] = vb[r];
            }
        } else {
            const int kvh = head - s.heads - s.kv_heads;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                pg[kv_value_offset(s.kv_heads, kvh, place, i0 + r, s.head_dim, s.page)] = va[r];
                pg[kv_value_offset(s.kv_heads, kvh, place, i0 + half_dim + r, s.head_dim, s.page)] = vb[r];
            }
        }
    }
}
