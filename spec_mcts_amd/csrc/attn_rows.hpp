// Row-at-a-time attention arithmetic shared by the decode attention kernels: a 16-lane group owns one
// K/V row of a 128-wide head, scores it against a query held in the same layout and folds it into an
// online-softmax state (base-2 exponentials; the caller pre-scales scores by log2(e)/sqrt(D)).
#pragma once

#include "smh_common.hpp"

namespace smh {

// ---- suffix rows ----------------------------------------------------------------------------------------
// A 16-lane group handles one row at a time; lane c of the group owns head dims 4c..4c+3 ("low half")
// and 64+4c..64+4c+3 ("high half"), held as fp16 pairs in the order (0,2),(1,3) that nibble decoding
// produces.
struct RowRegs { h2 a02, a13, b02, b13; };   // a: dims 4c.., b: dims 64+4c..

// (as it comes from memory, so that a caller can request a row early and wait for it where it is used)
struct RawRow { u32x2 lo, hi; };
__device__ __forceinline__ RawRow raw_row(const half_t *row, int c) {
    return RawRow{*reinterpret_cast<const u32x2 *>(row + 4 * c), *reinterpret_cast<const u32x2 *>(row + 64 + 4 * c)};
}
__device__ __forceinline__ RowRegs row_of_raw(const RawRow &t) {
    RowRegs r;
    r.a02 = as_h2(pack_lo16(t.lo[0], t.lo[1]));
    r.a13 = as_h2(pack_hi16(t.lo[0], t.lo[1]));
    r.b02 = as_h2(pack_lo16(t.hi[0], t.hi[1]));
    r.b13 = as_h2(pack_hi16(t.hi[0], t.hi[1]));
    return r;
}
__device__ __forceinline__ RowRegs row_from_fp16(const half_t *row, int c) { return row_of_raw(raw_row(row, c)); }
// Q4_0 rows.  A walk of them is bound by these instructions, so masks and magic numbers stand in registers that the compiler cannot see through: the nibbles'
// sign bits are flipped and the magic number's bits set by the instruction that masks them (v_bitop3_b32, which takes no literals), and a scale is picked
// by the product's own operand select.  13 instructions for the eight values of a dword; with an XOR, an AND and an OR each and a permute a scale 19.
// (us a step of the 7B architecture behind 512 rows, 10 / 64 / 127 rows of their own, before and now: 37 branches 2406 / 2490 / 2662 and 2391 / 2463 / 2643, 64
// 2716 / 2869 / 3062 and 2691 / 2772 / 2970, 100 3317 / 3592 / 3943 and 3307 / 3551 / 3912; three layers of 64 heads over 8, 100 branches and 90 rows 994 and 972.)
struct RowCodes {
    uint32_t mask_hi = 0x00F000F0u, mask_lo = 0x000F000Fu, magic_hi = 0x54005400u ^ 0x00800080u, magic_lo = MAGIC_1024 ^ 0x00080008u;
    __device__ __forceinline__ RowCodes() {
        asm volatile("" : "+s"(mask_hi), "+s"(mask_lo));
        asm volatile("" : "+v"(magic_hi), "+v"(magic_lo));
    }
};
// bytes: this lane's dword of the packed row; sc: (scale of dims 0..63, scale of dims 64..127).  With u = code + 8: 64 + u and 1024 + u, then the code, then its
// product, rounded once (smh_common.hpp).
__device__ __forceinline__ RowRegs row_from_q40(uint32_t bytes, uint32_t sc, const RowCodes &C) {
    const uint32_t next = bytes >> 8;
    const h2 s = as_h2(sc), s_a = __builtin_shufflevector(s, s, 0, 0), s_b = __builtin_shufflevector(s, s, 1, 1);
    const h2 off_hi = {(half_t)-72.f, (half_t)-72.f}, off_lo = {(half_t)-1032.f, (half_t)-1032.f};
    RowRegs r;
    r.a02 = (as_h2((bytes & C.mask_hi) ^ C.magic_hi) + off_hi) * s_a;
    r.a13 = (as_h2((next & C.mask_hi) ^ C.magic_hi) + off_hi) * s_a;
    r.b02 = (as_h2((bytes & C.mask_lo) ^ C.magic_lo) + off_lo) * s_b;
    r.b13 = (as_h2((next & C.mask_lo) ^ C.magic_lo) + off_lo) * s_b;
    return r;
}
// The same with the masks as literals, for a kernel that lacks the registers (decode_stack_kernel<4>)
__device__ __forceinline__ RowRegs row_from_q40(uint32_t bytes, uint32_t sc) {
    const uint32_t u = bytes ^ NIBBLE_FLIP, u1 = u >> 8;
    const h2 s_a = as_h2(pack_lo16(sc, sc)), s_b = as_h2(pack_hi16(sc, sc));
    RowRegs r;
    r.a02 = codes_high(u) * s_a;
    r.a13 = codes_high(u1) * s_a;
    r.b02 = codes_low(u) * s_b;
    r.b13 = codes_low(u1) * s_b;
    return r;
}
__device__ __forceinline__ float row_dot(const RowRegs &k, const RowRegs &q) {
    float s = __builtin_amdgcn_fdot2(k.a02, q.a02, 0.f, false);
    s = __builtin_amdgcn_fdot2(k.a13, q.a13, s, false);
    s = __builtin_amdgcn_fdot2(k.b02, q.b02, s, false);
    s = __builtin_amdgcn_fdot2(k.b13, q.b13, s, false);
    return row16_sum(s);
}

struct SoftState {
    float m, l;
    float o[8];     // dims 4c+0, 4c+2, 4c+1, 4c+3, 64+4c+0, 64+4c+2, 64+4c+1, 64+4c+3
};
__device__ __forceinline__ void soft_add_row(SoftState &st, float score, const RowRegs &v) {
    const float m_new = fmaxf(st.m, score);
    const float corr = exp2f(st.m - m_new);          // st.m = -inf on first use: exp2(-inf) = 0
    const float pr = exp2f(score - m_new);
    st.m = m_new;
    st.l = st.l * corr + pr;
    st.o[0] = st.o[0] * corr + pr * (float)v.a02.x;
    st.o[1] = st.o[1] * corr + pr * (float)v.a02.y;
    st.o[2] = st.o[2] * corr + pr * (float)v.a13.x;
    st.o[3] = st.o[3] * corr + pr * (float)v.a13.y;
    st.o[4] = st.o[4] * corr + pr * (float)v.b02.x;
    st.o[5] = st.o[5] * corr + pr * (float)v.b02.y;
    st.o[6] = st.o[6] * corr + pr * (float)v.b13.x;
    st.o[7] = st.o[7] * corr + pr * (float)v.b13.y;
}
// The maximum an un-normalised partial is handed on with.  -infinity: it holds no row, and whoever merges may pass it over.  Scores
// that are all NaN have no maximum either, but a sum, which is NaN and has to arrive: the lowest finite number.
__device__ __forceinline__ float partial_max(float m, float l) { return m == -INFINITY && !(l == 0.f) ? -3.402823466e38f : m; }
// fold an un-normalised partial (m2, l2, o2) into st
__device__ __forceinline__ void soft_merge(SoftState &st, float m2, float l2, const float *o2) {
    const float m_new = fmaxf(st.m, m2);
    if (m_new == -INFINITY) return;                  // both empty
    const float c1 = exp2f(st.m - m_new), c2 = exp2f(m2 - m_new);
    st.m = m_new;
    st.l = st.l * c1 + l2 * c2;
#pragma unroll
    for (int j = 0; j < 8; ++j) st.o[j] = st.o[j] * c1 + o2[j] * c2;
}

}  // namespace smh
