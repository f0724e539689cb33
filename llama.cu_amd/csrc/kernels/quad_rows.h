#pragma once
#include "common.h"

// Rows of bfloat16 as the second operand of v_mfma_f32_16x16x32_bf16 (a column of sixteen a row, lane group g of sixteen lanes the k from
// 8 g on), straight from memory into registers.  A compute unit looks a cache line up for every four neighbouring lanes of a 16-byte load:
// lanes that lie side by side in the operand are different rows, so a load in the operand's order takes a cycle for every lane, 16 bytes
// a cycle, where four lanes that read 64 bytes of one row take one cycle together (a product of 16 rows with K = 2048 in every workgroup:
// 1.6 us for the rows in the operand's order, whichever 16 bytes of a row its groups take, 0.4 this way).  So here
//
//   load i (0 .. 3) of 128 k: lane (g, a, b) = (lane / 16, lane / 4 % 4, lane % 4) reads row 4 i + a, k from 32 g + 8 b on,
//
// and a transposition between the loads and the lanes of a quad, in the vector unit (v_cndmask with its operand out of another lane),
// makes operand j of lane (g, a, b) row 4 b + a, k from 32 g + 8 j on: the weights' order, with the columns' rows in another order
// (quad_row).  Up to eight rows take two loads and up to four one; the columns without a row then hold what does not matter.
typedef __attribute__((ext_vector_type(4))) uint32_t quad_u32x4;

// the row of column c (0 .. 15) of the operands
__device__ __forceinline__ int quad_row(int c) { return 4 * (c & 3) + (c >> 2); }
// where lane `lane` begins in its row of load i, and that row
__device__ __forceinline__ int quad_k(int lane) { return 32 * (lane >> 4) + 8 * (lane & 3); }
__device__ __forceinline__ int quad_load_row(int i, int lane) { return 4 * i + ((lane >> 2) & 3); }

// Between registers and lanes the rule is: lo <- where `keep`: lo, else hi of the partner lane; hi <- where `keep`: lo of the partner lane, else
// hi.  The partner is one or two lanes away; keep is the mask of the lanes without that bit.  32 instructions for sixteen rows of 128 k, whose
// operand out of another lane makes them twice as slow as others: 2 us of the 8.3 that 64 rows of 2048 x 2048 take.  (Left to the compiler, a
// move and a selection each: 64.)  The waits: an operand out of another lane wants its register two states old, and so does a matrix
// instruction; the compiler does not look in here.
#define QUAD_1 "quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
#define QUAD_2 "quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
// to <- vcc ? own : other of the partner lane, four registers
#define QUAD_TAKE(TO, OTHER, OWN, P) \
    "v_cndmask_b32_dpp %[" #TO "0], %[" #OTHER "0], %[" #OWN "0], vcc " P "v_cndmask_b32_dpp %[" #TO "1], %[" #OTHER "1], %[" #OWN "1], vcc " P \
    "v_cndmask_b32_dpp %[" #TO "2], %[" #OTHER "2], %[" #OWN "2], vcc " P "v_cndmask_b32_dpp %[" #TO "3], %[" #OTHER "3], %[" #OWN "3], vcc " P
#define QUAD_REGS(HOW, NAME, V) [NAME##0] HOW(V[0]), [NAME##1] HOW(V[1]), [NAME##2] HOW(V[2]), [NAME##3] HOW(V[3])
#define QUAD_KEEP_1 0x5555555555555555ull
#define QUAD_KEEP_2 0x3333333333333333ull

// two registers and the neighbouring lane
__device__ __forceinline__ void quad_swap(const quad_u32x4 &a, const quad_u32x4 &b, quad_u32x4 &lo, quad_u32x4 &hi) {
    uint32_t c[4], d[4];
    asm("s_nop 1\n\t"
        "s_mov_b64 vcc, %[k1]\n\t" QUAD_TAKE(c, b, a, QUAD_1)
        "s_not_b64 vcc, vcc\n\t" QUAD_TAKE(d, a, b, QUAD_1)
        "s_nop 1"
        : QUAD_REGS("=&v", c, c), QUAD_REGS("=&v", d, d)
        : QUAD_REGS("v", a, a), QUAD_REGS("v", b, b), [k1] "s"(QUAD_KEEP_1)
        : "vcc", "scc");
    lo = quad_u32x4{c[0], c[1], c[2], c[3]};
    hi = quad_u32x4{d[0], d[1], d[2], d[3]};
}

// four registers and the four lanes of a quad
__device__ __forceinline__ void quad_transpose(const quad_u32x4 (&r)[4], quad_u32x4 (&x)[4]) {
    uint32_t e[4], f[4], g[4], h[4], m[4], n[4], o[4], p[4];
    asm("s_nop 1\n\t"
        "s_mov_b64 vcc, %[k1]\n\t" QUAD_TAKE(e, b, a, QUAD_1) QUAD_TAKE(g, d, c, QUAD_1)
        "s_not_b64 vcc, vcc\n\t" QUAD_TAKE(f, a, b, QUAD_1) QUAD_TAKE(h, c, d, QUAD_1)
        "s_mov_b64 vcc, %[k2]\n\t" QUAD_TAKE(m, g, e, QUAD_2) QUAD_TAKE(n, h, f, QUAD_2)
        "s_not_b64 vcc, vcc\n\t" QUAD_TAKE(o, e, g, QUAD_2) QUAD_TAKE(p, f, h, QUAD_2)
        "s_nop 1"
        : QUAD_REGS("=&v", e, e), QUAD_REGS("=&v", f, f), QUAD_REGS("=&v", g, g), QUAD_REGS("=&v", h, h),
          QUAD_REGS("=&v", m, m), QUAD_REGS("=&v", n, n), QUAD_REGS("=&v", o, o), QUAD_REGS("=&v", p, p)
        : QUAD_REGS("v", a, r[0]), QUAD_REGS("v", b, r[1]), QUAD_REGS("v", c, r[2]), QUAD_REGS("v", d, r[3]), [k1] "s"(QUAD_KEEP_1), [k2] "s"(QUAD_KEEP_2)
        : "vcc", "scc");
    x[0] = quad_u32x4{m[0], m[1], m[2], m[3]};
    x[1] = quad_u32x4{n[0], n[1], n[2], n[3]};
    x[2] = quad_u32x4{o[0], o[1], o[2], o[3]};
    x[3] = quad_u32x4{p[0], p[1], p[2], p[3]};
}
// the same in two halves, so that the second one's results may have the first one's operands' registers: 16 fewer, a wait more
__device__ __forceinline__ void quad_transpose_in_less(const quad_u32x4 (&r)[4], quad_u32x4 (&x)[4]) {
    uint32_t e[4], f[4], g[4], h[4], m[4], n[4], o[4], p[4];
    asm("s_nop 1\n\t"
        "s_mov_b64 vcc, %[k1]\n\t" QUAD_TAKE(e, b, a, QUAD_1) QUAD_TAKE(g, d, c, QUAD_1)
        "s_not_b64 vcc, vcc\n\t" QUAD_TAKE(f, a, b, QUAD_1) QUAD_TAKE(h, c, d, QUAD_1)
        : QUAD_REGS("=&v", e, e), QUAD_REGS("=&v", f, f), QUAD_REGS("=&v", g, g), QUAD_REGS("=&v", h, h)
        : QUAD_REGS("v", a, r[0]), QUAD_REGS("v", b, r[1]), QUAD_REGS("v", c, r[2]), QUAD_REGS("v", d, r[3]), [k1] "s"(QUAD_KEEP_1)
        : "vcc", "scc");
    asm("s_nop 1\n\t"
        "s_mov_b64 vcc, %[k2]\n\t" QUAD_TAKE(m, g, e, QUAD_2) QUAD_TAKE(n, h, f, QUAD_2)
        "s_not_b64 vcc, vcc\n\t" QUAD_TAKE(o, e, g, QUAD_2) QUAD_TAKE(p, f, h, QUAD_2)
        "s_nop 1"
        : QUAD_REGS("=&v", m, m), QUAD_REGS("=&v", n, n), QUAD_REGS("=&v", o, o), QUAD_REGS("=&v", p, p)
        : QUAD_REGS("v", e, e), QUAD_REGS("v", f, f), QUAD_REGS("v", g, g), QUAD_REGS("v", h, h), [k2] "s"(QUAD_KEEP_2)
        : "vcc", "scc");
    x[0] = quad_u32x4{m[0], m[1], m[2], m[3]};
    x[1] = quad_u32x4{n[0], n[1], n[2], n[3]};
    x[2] = quad_u32x4{o[0], o[1], o[2], o[3]};
    x[3] = quad_u32x4{p[0], p[1], p[2], p[3]};
}
#undef QUAD_1
#undef QUAD_2
#undef QUAD_TAKE
#undef QUAD_REGS
#undef QUAD_KEEP_1
#undef QUAD_KEEP_2

template <int CTRL>
__device__ __forceinline__ quad_u32x4 quad_perm(const quad_u32x4 &v) {
    quad_u32x4 o;
#pragma unroll
    for (int d = 0; d < 4; ++d) o[d] = (uint32_t)__builtin_amdgcn_mov_dpp((int)v[d], CTRL, 0xF, 0xF, true);
    return o;
}

// r: what the loads brought; x: the operands; LESS: in fewer registers
template <int LOADS, bool LESS = false>
__device__ __forceinline__ void quad_operands(const quad_u32x4 (&r)[LOADS], quad_u32x4 (&x)[4]) {
    static_assert(LOADS == 1 || LOADS == 2 || LOADS == 4, "rows in fours");
    if constexpr (LOADS == 1) {
        x[0] = r[0];
        x[1] = quad_perm<0xB1>(r[0]);           // [1, 0, 3, 2]
        x[2] = quad_perm<0x4E>(r[0]);           // [2, 3, 0, 1]
        x[3] = quad_perm<0x1B>(r[0]);           // [3, 2, 1, 0]
    } else if constexpr (LOADS == 2) {
        quad_swap(r[0], r[1], x[0], x[1]);
        x[2] = quad_perm<0x4E>(x[0]);
        x[3] = quad_perm<0x4E>(x[1]);
    } else if constexpr (LESS) {
        quad_transpose_in_less(r, x);
    } else {
        quad_transpose(r, x);
    }
}
