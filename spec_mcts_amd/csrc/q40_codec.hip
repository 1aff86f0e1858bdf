// Flat Q4_0 codec kernels: 64-byte rows of packed signed nibbles <-> fp16.
//
// Both kernels are pure streaming (HBM-bound): dequant reads 68 B and writes 256 B per row,
// quantise reads 256 B and writes 68 B per row.  One lane owns 16 bytes of a row, so a row is
// covered by 4 neighbouring lanes and every access is a 128-bit load/store.
#include <type_traits>

#include "q40_matmul.hpp"

namespace smh {

typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));

// out[row*128 + j]      = code(high nibble of byte j) * s[2*row]
// out[row*128 + 64 + j] = code(low  nibble of byte j) * s[2*row+1]      (one fp16 multiply each)
__global__ __launch_bounds__(256) void q40_dequant_kernel(const u32x4 *__restrict__ w,
                                                          const uint32_t *__restrict__ s,
                                                          half_t *__restrict__ out, long rows) {
    long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    long row = t >> 2;
    int c = (int)(t & 3);
    if (row >= rows) return;
    u32x4 v = w[row * 4 + c];
    uint32_t sp = s[row];                       // (s[2row], s[2row+1])
    h2 s_hi = as_h2(pack_lo16(sp, sp));
    h2 s_lo = as_h2(pack_hi16(sp, sp));
    uint32_t hi[8], lo[8];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        uint32_t u = v[j] ^ NIBBLE_FLIP;
        uint32_t u1 = u >> 8;
        // pairs (byte0, byte2) and (byte1, byte3) of this word
        uint32_t h02 = as_u32(codes_high(u) * s_hi), h13 = as_u32(codes_high(u1) * s_hi);
        uint32_t l02 = as_u32(codes_low(u) * s_lo), l13 = as_u32(codes_low(u1) * s_lo);
        hi[2 * j] = pack_lo16(h02, h13);        // (byte0, byte1)
        hi[2 * j + 1] = pack_hi16(h02, h13);    // (byte2, byte3)
        lo[2 * j] = pack_lo16(l02, l13);
        lo[2 * j + 1] = pack_hi16(l02, l13);
    }
    u32x4 *o_hi = reinterpret_cast<u32x4 *>(out + row * 128 + c * 16);
    u32x4 *o_lo = reinterpret_cast<u32x4 *>(out + row * 128 + 64 + c * 16);
    o_hi[0] = u32x4{hi[0], hi[1], hi[2], hi[3]};
    o_hi[1] = u32x4{hi[4], hi[5], hi[6], hi[7]};
    o_lo[0] = u32x4{lo[0], lo[1], lo[2], lo[3]};
    o_lo[1] = u32x4{lo[4], lo[5], lo[6], lo[7]};
}

// One fp16 value -> code with torch's semantics: q = fp16(x / scale); code = rint(q) (to nearest
// even); NaN (0/0) -> 0.  The division is a correctly rounded fp32 division rounded once more to fp16.
__device__ __forceinline__ int q40_code(half_t x, float scale) {
    half_t q = (half_t)((float)x / scale);
    float qf = (float)q;
    if (!(qf == qf)) return 0;
    return (int)__builtin_rintf(qf);
}
// ... of a value of a wider type: the quotient stays fp32
__device__ __forceinline__ int q40_code_wide(float x, float scale) {
    const float qf = x / scale;
    return (qf == qf) ? (int)__builtin_rintf(qf) : 0;
}

// The same codes without a division per value.  For a group whose scale is a normal finite fp16 number, x * (1 / scale) in
// fp32 lies within 2^-21 (relative) of the quotient and |quotient| < 8, so it rounds to the same code unless it lies that
// close to a point where the code changes; such values (and groups with any other scale) take the division.  A division is
// ~16 instructions of which two run at a quarter of the rate: a weight of 45 M values is 29 us of vector ALU with it, more
// than its bytes cost.
__device__ __forceinline__ bool q40_scale_is_plain(float scale) { return scale >= 6.103515625e-05f && scale <= 65504.0f; }
// fp16 values: the code changes where the fp16 rounding of the quotient does, at midpoints between fp16 numbers - fp32 numbers
// whose low 13 bits are 0x1000 (below 2^-14 the midpoints lie elsewhere, but there every code is 0)
__device__ __forceinline__ int q40_code_near(half_t x, float inv, bool &doubt) {
    const float q = (float)x * inv;
    doubt = ((__builtin_bit_cast(uint32_t, q) + 0x1003u) & 0x1FFFu) <= 6u;
    return (int)(short)__builtin_rintf16((half_t)q);
}
// fp32 quotients: the code changes at n + 1/2.  Adding 1.5 * 2^23 rounds to an integer that stands in the low bits of the sum.  (A NaN
// beside finite values leaves the group's scale plain: it is in doubt too and takes the division, code 0.  fp16 groups take their
// largest magnitude from the bit patterns, so with a NaN their scale is one.)
__device__ __forceinline__ int q40_code_near(float x, float inv, bool &doubt) {
    constexpr float round = 12582912.0f;
    const float t = __builtin_fmaf(x, inv, round), r = t - round;
    doubt = !(fabsf(__builtin_fmaf(x, inv, -r)) <= 0.5f - 7.62939453125e-06f);
    return __builtin_bit_cast(int, t);
}
__device__ __forceinline__ int q40_code_exact(half_t x, float scale) { return q40_code(x, scale); }
__device__ __forceinline__ int q40_code_exact(float x, float scale) { return q40_code_wide(x, scale); }

// The codes of eight values; only the low four bits of each count.
template <typename T>
__device__ __forceinline__ void q40_codes8(const T (&x)[8], float scale, int (&code)[8]) {
    if (q40_scale_is_plain(scale)) {
        const float inv = 1.0f / scale;
        bool doubt[8], any = false;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            code[i] = q40_code_near(x[i], inv, doubt[i]);
            any |= doubt[i];
        }
        if (any) {
#pragma unroll
            for (int i = 0; i < 8; ++i)
                if (doubt[i]) code[i] = q40_code_exact(x[i], scale);
        }
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) code[i] = q40_code_exact(x[i], scale);
    }
}

// eight codes -> value j in bits 4j .. 4j+3
__device__ __forceinline__ uint32_t nibbles8(const int (&c)[8]) {
    uint32_t v = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j) v |= (uint32_t)(c[j] & 15) << (4 * j);
    return v;
}
__device__ __forceinline__ u32x2 pack_codes(uint32_t hi, uint32_t lo) {
    uint32_t b0 = 0, b1 = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        b0 |= ((((hi >> (4 * j)) & 15) << 4) | ((lo >> (4 * j)) & 15)) << (8 * j);
        b1 |= ((((hi >> (4 * j + 16)) & 15) << 4) | ((lo >> (4 * j + 16)) & 15)) << (8 * j);
    }
    return u32x2{b0, b1};
}
// largest value of the 8 lanes that share lane / 8
__device__ __forceinline__ float max8(float v) {
    v = fmaxf(v, dpp_move<DPP_QUAD_XOR1>(v));
    v = fmaxf(v, dpp_move<DPP_QUAD_XOR2>(v));
    return fmaxf(v, dpp_move<DPP_ROW_HALF_MIRROR>(v));
}
__device__ __forceinline__ uint32_t max8(uint32_t v) {       // (bit patterns below 2^31: compared as integers)
    v = max(v, __builtin_bit_cast(uint32_t, dpp_move<DPP_QUAD_XOR1>(__builtin_bit_cast(float, v))));
    v = max(v, __builtin_bit_cast(uint32_t, dpp_move<DPP_QUAD_XOR2>(__builtin_bit_cast(float, v))));
    return max(v, __builtin_bit_cast(uint32_t, dpp_move<DPP_ROW_HALF_MIRROR>(__builtin_bit_cast(float, v))));
}

// Lane layout: 8 lanes per 64-value group (8 values = one 128-bit load each), so a wave covers
// 8 groups = 4 packed rows.  absmax is reduced over the 8 lanes of a group with xor-shuffles.
__global__ __launch_bounds__(256) void q40_quantize_kernel(const u32x4 *__restrict__ in,
                                                           uint8_t *__restrict__ w,
                                                           half_t *__restrict__ s, long groups) {
    long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    long g = t >> 3;
    int c = (int)(t & 7);
    bool live = g < groups;
    u32x4 raw = live ? in[t] : u32x4{0, 0, 0, 0};
    half_t x[8];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        h2 p = as_h2(raw[j]);
        x[2 * j] = p.x;
        x[2 * j + 1] = p.y;
    }
    // |x| as bit patterns: for finite values the integer order is the magnitude order
    uint32_t amax = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        uint32_t a = raw[j] & 0x7FFF7FFFu;
        uint32_t m = max(a & 0xFFFFu, a >> 16);
        amax = max(amax, m);
    }
    amax = max8(amax);
    half_t amax_h = __builtin_bit_cast(half_t, (uint16_t)amax);
    half_t scale_h = (half_t)((float)amax_h / 7.0f);
    float scale = (float)scale_h;
    int code[8];
    q40_codes8(x, scale, code);
    const uint32_t nib = nibbles8(code);
    // the partner group (g ^ 1) sits 8 lanes away; even groups supply high nibbles
    uint32_t other = (uint32_t)__shfl_xor((int)nib, 8, 64);
    if (!live) return;
    if (c == 0) s[g] = scale_h;
    if ((g & 1) == 0) {
        *reinterpret_cast<u32x2 *>(w + (g >> 1) * 64 + c * 8) = pack_codes(nib, other);
    }
}

// The same quantiser for checkpoint weights held in fp32 or bfloat16 (passed widened to fp32, which is exact).  torch's
// arithmetic for those types (fp16_to_int4.py:60-70 run on such a tensor): wmax / 7.0 is rounded to the tensor's own
// type (fp32, or bfloat16) and then to fp16; w / scale promotes to fp32, so the quotient is NOT rounded to fp16 before
// round-half-even; 0 / 0 -> NaN -> code 0.  SRC_BF16 selects the intermediate bfloat16 rounding of the scale.
__device__ __forceinline__ float round_to_bf16(float x) {
    uint32_t u = __builtin_bit_cast(uint32_t, x);
    if ((u & 0x7F800000u) == 0x7F800000u) return x;                  // inf / nan stay
    u += 0x7FFFu + ((u >> 16) & 1u);
    return __builtin_bit_cast(float, u & 0xFFFF0000u);
}
template <bool SRC_BF16>
__global__ __launch_bounds__(256) void q40_quantize_f32_kernel(const f4 *__restrict__ in, uint8_t *__restrict__ w,
                                                               half_t *__restrict__ s, long groups) {
    long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    long g = t >> 3;
    int c = (int)(t & 7);
    bool live = g < groups;
    f4 a = live ? in[2 * t] : f4{0.f, 0.f, 0.f, 0.f}, b = live ? in[2 * t + 1] : f4{0.f, 0.f, 0.f, 0.f};
    const float x[8] = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
    float amax = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) amax = fmaxf(amax, fabsf(x[j]));
    amax = max8(amax);
    float q7 = amax / 7.0f;
    if (SRC_BF16) q7 = round_to_bf16(q7);
    const half_t scale_h = (half_t)q7;
    const float scale = (float)scale_h;
    int code[8];
    q40_codes8(x, scale, code);
    const uint32_t nib = nibbles8(code);
    uint32_t other = (uint32_t)__shfl_xor((int)nib, 8, 64);
    if (!live) return;
    if (c == 0) s[g] = scale_h;
    if ((g & 1) == 0) {
        *reinterpret_cast<u32x2 *>(w + (g >> 1) * 64 + c * 8) = pack_codes(nib, other);
    }
}

// a / 7, correctly rounded, of a magnitude: the quotient by the reciprocal corrected by its remainder.  (Infinities and NaN, and what is so
// large that the remainder might overflow, are left to the division.)
__device__ __forceinline__ float seventh(float a) {
    constexpr float r = 1.0f / 7.0f;
    float q = a * r;
    q = __builtin_fmaf(__builtin_fmaf(-q, 7.0f, a), r, q);
    if (!(a < 3e38f)) q = a / 7.0f;
    return q;
}
// The codes of eight values in the low halves of eight bytes (the high halves hold anything).
// Values of at most 11 significant bits (fp16, bfloat16): the quotient is corrected by its remainder, which gives the division's (corrected_quotient).
// With a doubt about the values next to a tie, as below, most waves divided: a bfloat16 weight has one value in 440 exactly on a tie.
__device__ __forceinline__ u32x2 q40_bytes8(const half_t (&x)[8], float scale) {
    u16x2 code[4];
    if (q40_scale_is_plain(scale)) {
        const float inv = __builtin_amdgcn_rcpf(scale);
#pragma unroll
        for (int i = 0; i < 4; ++i) {                        // rounded to fp16, then added to 1536, whose neighbours are one apart
            const f2 q = {corrected_quotient((float)x[2 * i], scale, inv), corrected_quotient((float)x[2 * i + 1], scale, inv)};
            code[i] = __builtin_bit_cast(u16x2, __builtin_convertvector(q, h2) + h2{(half_t)1536.0f, (half_t)1536.0f});
        }
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) code[i >> 1][i & 1] = (uint16_t)q40_code(x[i], scale);
    }
    auto four = [&](int i) { return __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, code[i + 1]), __builtin_bit_cast(uint32_t, code[i]), 0x06040200u); };
    return u32x2{four(0), four(2)};
}
// (A NaN's low bits are zeros, and so is its code.)
__device__ __forceinline__ u32x2 q40_bytes8_bf16(const float (&x)[8], float scale) {
    uint32_t t[8];
    if (q40_scale_is_plain(scale)) {
        const float inv = __builtin_amdgcn_rcpf(scale);
#pragma unroll
        for (int i = 0; i < 8; ++i) t[i] = __builtin_bit_cast(uint32_t, corrected_quotient(x[i], scale, inv) + 12582912.0f);      // 1.5 x 2^23
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) t[i] = (uint32_t)q40_code_wide(x[i], scale);
    }
    auto four = [&](int i) { return __builtin_amdgcn_perm(t[i + 1], t[i], 0x0c0c0400u) | __builtin_amdgcn_perm(t[i + 3], t[i + 2], 0x04000c0cu); };
    return u32x2{four(0), four(4)};
}
// fp32 values: x / scale + 192.5 has 16 bits below the point, so that bits 16 .. 19 are the quotient rounded.  The sum is within 2^-16 of
// the exact one, and a code is in doubt, and divided for, where the bits below the point say that a whole number is at most as far away: it or its
// neighbours (one value in 20000; a NaN has zeros there or is found as one).  Whether any is: the least of eight distances, two to a register.
__device__ __forceinline__ u32x2 q40_bytes8_f32(const float (&x)[8], float scale) {
    uint32_t t[8];
    bool all = !q40_scale_is_plain(scale);
    const float inv = __builtin_amdgcn_rcpf(scale);
#pragma unroll
    for (int i = 0; i < 8; ++i) t[i] = __builtin_bit_cast(uint32_t, __builtin_fmaf(x[i], inv, 192.5f));
    auto near = [&](int i) { return __builtin_bit_cast(u16x2, pack_lo16(t[i], t[i + 1])) + u16x2{1, 1}; };
    const u16x2 least = __builtin_elementwise_min(__builtin_elementwise_min(near(0), near(2)), __builtin_elementwise_min(near(4), near(6)));
    // (finite values do not add up to a NaN)
    const float sum = ((x[0] + x[1]) + (x[2] + x[3])) + ((x[4] + x[5]) + (x[6] + x[7]));
    if (all || min(least.x, least.y) < 3 || sum != sum) {
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (all || ((t[i] + 1) & 0xFFFFu) < 3 || x[i] != x[i]) t[i] = (uint32_t)q40_code_wide(x[i], scale) << 16;
    }
    auto four = [&](int i) { return __builtin_amdgcn_perm(t[i + 1], t[i], 0x0c0c0602u) | __builtin_amdgcn_perm(t[i + 3], t[i + 2], 0x06020c0cu); };
    return u32x2{four(0), four(4)};
}

// ---- a checkpoint's linear weight [N, K] -> Q4_0 of its transpose, in one pass ------------------------------------------------
// A workgroup takes 128 outputs n x 128 bytes of inputs k.  The tile is read along k (whole cache lines, 16 bytes a lane), turned in LDS
// and quantised along n: eight lanes share input column k (two columns at a time for 16-bit types), lane o holding outputs
// 8 o .. 8 o + 7 of either group of 64, so a lane's codes are 8 consecutive bytes of packed row (k, n / 128).
// Neighbouring blocks of 128 outputs (halves of one 128-byte line of codes, parts of one line of scales) go to one XCD, one
// after the other, so that its L2 joins them; `together` of them at a k (smh_q40_quantize_t).
// Bound by HBM (2 or 4 bytes read, 17/32 written per value); loads alone take 18 us at 11008 x 4096 bfloat16, and the vector ALU, with no steady state
// to hide it in (few tiles a compute unit), most of the rest.  In turn, us, with a division in every wave that has a value next to a tie, fp32 tiles of 256
// bytes and all blocks of outputs at a k, and now: bfloat16 11008 x 4096 28.5 and 27.5 (4.2 TB/s), 8192 x 1024 7.9 and 6.8, 28672 x 8192 136 and 132 (4.5
// TB/s); fp16 4096 x 4096 16.4 and 12.2, 19968 x 2111 40.1 and 29.7; fp32 8192 x 8192 91.4 and 65.1 (4.7 TB/s), 3072 x 3001 13.7 and 11.7.  (Tiles of 256
// bytes: level.  Workgroups that stay and load the next tile under this one: 31 to 44 us at 11008 x 4096, where others wait they wait, too.)
//   SRC 0: fp16, 1: bfloat16, 2: fp32.  P: dwords of an LDS row, odd so that the eight rows a wave reads at a time are 8 P = 8
// (mod 64) banks apart.
constexpr int QT_ROW = 128, QT_THREADS = 2 * QT_ROW;        // bytes of a tile's row; eight lanes to a dword of it
template <int SRC>
__global__ __launch_bounds__(QT_THREADS) void q40_quantize_t_kernel(const uint8_t *__restrict__ in, int N, int K, uint8_t *__restrict__ w,
                                                                    half_t *__restrict__ s, int k_tiles, int together) {
    constexpr int ES = SRC == 2 ? 4 : 2;                     // bytes of a source value
    constexpr int P = QT_ROW / 4 + 1;
    __shared__ uint32_t tile[128 * P];
    const int tid = threadIdx.x;
    const int n_blocks = N / 128;
    const int total = n_blocks * k_tiles, per = (total + 7) / 8;       // (of a grid: below 2^31 - 8)
    constexpr int VEC = 16 / ES;                             // values of a load
    constexpr int LPR = QT_ROW / 16;                         // lanes a row
    constexpr int LOADS = 128 / (QT_THREADS / LPR);
    const int id = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= per || id >= total) return;
    const DivMod of = uniform_divmod(id, together * k_tiles);
    const int nb0 = of.q * together;
    const DivMod at = uniform_divmod(of.r, min(together, n_blocks - nb0));
    const int nb = nb0 + at.r, k0 = at.q * (QT_ROW / ES);
    {
        const int c = tid % LPR, r0 = tid / LPR, k = k0 + c * VEC;
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            const int r = r0 + i * (QT_THREADS / LPR);
            const uint8_t *src = in + ((long)(nb * 128 + r) * K + k) * ES;
            uint32_t v[4] = {0, 0, 0, 0};
            if (k + VEC <= K) {
                __builtin_memcpy(v, src, 16);                // (rows of an odd K start at any multiple of the value's size)
            } else {
#pragma unroll
                for (int e = 0; e < VEC; ++e) {
                    if (k + e >= K) continue;
                    if constexpr (ES == 4) v[e] = *reinterpret_cast<const uint32_t *>(src + 4 * e);
                    else v[e / 2] |= (uint32_t)*reinterpret_cast<const uint16_t *>(src + 2 * e) << (16 * (e & 1));
                }
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) tile[r * P + 4 * c + q] = v[q];
        }
    }
    __syncthreads();
    constexpr int KL = SRC == 2 ? 1 : 2;                     // input columns per LDS dword
    const int o = tid & 7;
    {
        const int kc = tid >> 3;                             // dword column
        uint32_t d[2][8];
#pragma unroll
        for (int g = 0; g < 2; ++g)
#pragma unroll
            for (int i = 0; i < 8; ++i) d[g][i] = tile[(64 * g + 8 * o + i) * P + kc];
#pragma unroll
        for (int h = 0; h < KL; ++h) {
            const int k = k0 + KL * kc + h;
            u32x2 nib[2];                                    // codes in the low halves of the bytes, either group's
            half_t sc[2];
#pragma unroll
            for (int g = 0; g < 2; ++g) {
                if constexpr (SRC == 0) {
                    uint32_t bits[8], abits = 0;             // |x| as a bit pattern: integer order is magnitude order
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        bits[i] = h == 0 ? d[g][i] & 0xFFFFu : d[g][i] >> 16;
                        abits = max(abits, bits[i] & 0x7FFFu);
                    }
                    sc[g] = (half_t)seventh((float)__builtin_bit_cast(half_t, (uint16_t)max8(abits)));
                    half_t x[8];
#pragma unroll
                    for (int i = 0; i < 8; ++i) x[i] = __builtin_bit_cast(half_t, (uint16_t)bits[i]);
                    nib[g] = q40_bytes8(x, (float)sc[g]);
                } else {
                    float x[8], amax = 0.f;
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        if constexpr (SRC == 1) x[i] = __builtin_bit_cast(float, h == 0 ? d[g][i] << 16 : d[g][i] & 0xFFFF0000u);
                        else x[i] = __builtin_bit_cast(float, d[g][i]);
                        amax = fmaxf(amax, fabsf(x[i]));
                    }
                    float q7 = seventh(max8(amax));
                    if constexpr (SRC == 1) q7 = round_to_bf16(q7);
                    sc[g] = (half_t)q7;
                    if constexpr (SRC == 1) nib[g] = q40_bytes8_bf16(x, (float)sc[g]);
                    else nib[g] = q40_bytes8_f32(x, (float)sc[g]);
                }
            }
            if (k >= K) continue;
            const u32x2 both = (nib[0] << 4 & 0xF0F0F0F0u) | (nib[1] & 0x0F0F0F0Fu);
            *reinterpret_cast<u32x2 *>(w + ((long)k * n_blocks + nb) * 64 + 8 * o) = both;
            if (o == 0) *reinterpret_cast<h2 *>(s + ((long)k * n_blocks + nb) * 2) = h2{sc[0], sc[1]};
        }
    }
}

// One thread per output dword of the tiled layout (q40_matmul.hpp): 1024 nibble dwords + 64 scale dwords per tile.
__global__ __launch_bounds__(256) void q40_tile_kernel(const uint8_t *__restrict__ w, const half_t *__restrict__ s,
                                                       int K, int N, uint32_t *__restrict__ tiled, long tiles) {
    const long idx = (long)blockIdx.x * 256 + threadIdx.x;
    constexpr int DW = TILE_BYTES / 4;
    if (idx >= tiles * DW) return;
    const long tile = idx / DW;
    const int d = (int)(idx - tile * DW);
    const long steps = tiled_steps(K);
    const int unit = (int)(tile / steps), step = (int)(tile - (long)unit * steps);
    uint32_t out;
    if (d < TILE_W_BYTES / 4) {
        const int q = d >> 8, lane = (d >> 2) & 63, e = d & 3;         // piece, lane, dword of the lane's 16 bytes
        const int g = lane >> 4, c = lane & 15, blk = q >> 1, B = 2 * (q & 1) + (e >> 1);
        const long col = (long)unit * 128 + 64 * blk + 4 * c + B;       // byte column of the checkpoint row
        const int r0 = 32 * step + 8 * g + ((e & 1) ? 2 : 0);           // x: rows 0,4,1,5; x2: rows 2,6,3,7
        const int rows[4] = {r0, r0 + 4, r0 + 1, r0 + 5};
        out = 0;
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            uint32_t byte = 0;                                           // code 0 | code 0 before the flip
            if (rows[b] < K && col < N / 2) byte = w[(long)rows[b] * (N / 2) + col];
            out |= (byte ^ 0x88u) << (8 * b);
        }
    } else {
        const int e = d - TILE_W_BYTES / 4;                              // [g][group][i / 2]
        const int g = e >> 4, grp = (e >> 2) & 3, i = 2 * (e & 3);
        const long gcol = (long)unit * 4 + grp;
        uint32_t v[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int row = 32 * step + 8 * g + i + h;
            v[h] = (row < K && gcol < N / 64) ? __builtin_bit_cast(uint16_t, s[(long)row * (N / 64) + gcol]) : 0u;
        }
        out = v[0] | (v[1] << 16);
    }
    tiled[idx] = out;
}

}  // namespace smh

extern "C" size_t smh_q40_tiled_bytes(int K, int N) {
    if (K <= 0 || N <= 0) return 0;
    return (size_t)smh::tiled_units(N) * smh::tiled_steps(K) * smh::TILE_BYTES;
}

extern "C" int smh_q40_tile(const void *w, const void *s, int K, int N, void *tiled, size_t tiled_bytes, smh_stream_t stream) {
    using namespace smh;
    SMH_REQUIRE(K > 0 && N > 0 && N % 128 == 0, "smh_q40_tile: K=%d N=%d (N must be a positive multiple of 128)", K, N);
    SMH_REQUIRE(w && s && tiled, "smh_q40_tile: null pointer");
    SMH_REQUIRE(tiled_bytes >= smh_q40_tiled_bytes(K, N), "smh_q40_tile: buffer %zu < %zu bytes", tiled_bytes, smh_q40_tiled_bytes(K, N));
    SMH_REQUIRE(((uintptr_t)tiled & 127) == 0, "smh_q40_tile: the tiled buffer must be 128-byte aligned");
    const long tiles = tiled_units(N) * tiled_steps(K);
    const long threads = tiles * (TILE_BYTES / 4);
    hipLaunchKernelGGL(q40_tile_kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                       (const uint8_t *)w, (const half_t *)s, K, N, (uint32_t *)tiled, tiles);
    return launch_status();
}

extern "C" int smh_q40_dequant(const void *w, const void *s, void *out, long rows, smh_stream_t stream) {
    using namespace smh;
    SMH_REQUIRE(rows >= 0, "smh_q40_dequant: rows=%ld", rows);
    if (rows == 0) return 0;
    SMH_REQUIRE(w && s && out, "smh_q40_dequant: null pointer");
    long threads = rows * 4;
    dim3 grid((unsigned)((threads + 255) / 256));
    hipLaunchKernelGGL(q40_dequant_kernel, grid, dim3(256), 0, (hipStream_t)stream,
                       (const u32x4 *)w, (const uint32_t *)s, (half_t *)out, rows);
    return launch_status();
}

// ---- the block-of-32 flavour (scale = absmax / 8, codes 0..15 with offset 8, elements j and j + 16 share byte j) ----
// one thread per block: 16 bytes + one fp16 scale <-> 32 fp16 values
namespace smh {
__global__ __launch_bounds__(256) void gq40_dequant_kernel(const u32x4 *__restrict__ packed, const half_t *__restrict__ scale,
                                                           half_t *__restrict__ out, long blocks) {
    const long b = (long)blockIdx.x * 256 + threadIdx.x;
    if (b >= blocks) return;
    const u32x4 v = packed[b];
    const half_t sc = scale[b];
    half_t lo[16], hi[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) {
        const uint32_t byte = (v[j >> 2] >> (8 * (j & 3))) & 255u;
        lo[j] = (half_t)(float)((int)(byte & 15u) - 8) * sc;         // exact small integer times the scale: one fp16 rounding
        hi[j] = (half_t)(float)((int)(byte >> 4) - 8) * sc;
    }
    u32x4 *o = reinterpret_cast<u32x4 *>(out + b * 32);
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        o[q] = u32x4{as_u32(h2{lo[8 * q], lo[8 * q + 1]}), as_u32(h2{lo[8 * q + 2], lo[8 * q + 3]}),
                     as_u32(h2{lo[8 * q + 4], lo[8 * q + 5]}), as_u32(h2{lo[8 * q + 6], lo[8 * q + 7]})};
        o[2 + q] = u32x4{as_u32(h2{hi[8 * q], hi[8 * q + 1]}), as_u32(h2{hi[8 * q + 2], hi[8 * q + 3]}),
                         as_u32(h2{hi[8 * q + 4], hi[8 * q + 5]}), as_u32(h2{hi[8 * q + 6], hi[8 * q + 7]})};
    }
}

// rint(fp16(x / scale)) cut to -8 .. 8 while still a float (a scale that underflowed to 0 gives +-inf), NaN (0 / 0) -> 0
__device__ __forceinline__ int gq40_code(half_t x, float scale) {
    const float qf = (float)(half_t)((float)x / scale);
    if (!(qf == qf)) return 0;
    return (int)__builtin_rintf(fminf(fmaxf(qf, -8.0f), 8.0f));
}

__global__ __launch_bounds__(256) void gq40_quantize_kernel(const u32x4 *__restrict__ in, u32x4 *__restrict__ packed,
                                                            half_t *__restrict__ scale, long blocks) {
    const long b = (long)blockIdx.x * 256 + threadIdx.x;
    if (b >= blocks) return;
    half_t x[32];
    uint32_t amax = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const u32x4 r = in[b * 4 + q];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const h2 pr = as_h2(r[j]);
            x[8 * q + 2 * j] = pr.x;
            x[8 * q + 2 * j + 1] = pr.y;
            const uint32_t a = r[j] & 0x7FFF7FFFu;                  // |x| as bit patterns: integer order = magnitude order
            amax = max(amax, max(a & 0xFFFFu, a >> 16));
        }
    }
    const half_t scale_h = (half_t)((float)__builtin_bit_cast(half_t, (uint16_t)amax) / 8.0f);
    const float sf = (float)scale_h;
    uint32_t w[4] = {0, 0, 0, 0};
#pragma unroll
    for (int j = 0; j < 16; ++j) {
        const int ql = min(gq40_code(x[j], sf) + 8, 15), qh = min(gq40_code(x[j + 16], sf) + 8, 15);
        w[j >> 2] |= (uint32_t)(ql | (qh << 4)) << (8 * (j & 3));
    }
    packed[b] = u32x4{w[0], w[1], w[2], w[3]};
    scale[b] = scale_h;
}
}  // namespace smh

extern "C" int smh_gq40_dequant(const void *packed, const void *scale, void *out, long blocks, smh_stream_t stream) {
    using namespace smh;
    SMH_REQUIRE(blocks >= 0, "smh_gq40_dequant: blocks=%ld", blocks);
    if (blocks == 0) return 0;
    SMH_REQUIRE(packed && scale && out && (((uintptr_t)packed | (uintptr_t)out) & 15) == 0, "smh_gq40_dequant: null or misaligned pointer");
    hipLaunchKernelGGL(gq40_dequant_kernel, dim3((unsigned)((blocks + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                       (const u32x4 *)packed, (const half_t *)scale, (half_t *)out, blocks);
    return launch_status();
}

extern "C" int smh_gq40_quantize(const void *in, void *packed, void *scale, long blocks, smh_stream_t stream) {
    using namespace smh;
    SMH_REQUIRE(blocks >= 0, "smh_gq40_quantize: blocks=%ld", blocks);
    if (blocks == 0) return 0;
    SMH_REQUIRE(in && packed && scale && (((uintptr_t)in | (uintptr_t)packed) & 15) == 0, "smh_gq40_quantize: null or misaligned pointer");
    hipLaunchKernelGGL(gq40_quantize_kernel, dim3((unsigned)((blocks + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                       (const u32x4 *)in, (u32x4 *)packed, (half_t *)scale, blocks);
    return launch_status();
}

extern "C" int smh_q40_quantize(const void *in, void *w, void *s, long groups, smh_stream_t stream) {
    using namespace smh;
    SMH_REQUIRE(groups >= 0 && (groups & 1) == 0, "smh_q40_quantize: groups=%ld must be even", groups);
    if (groups == 0) return 0;
    SMH_REQUIRE(in && w && s, "smh_q40_quantize: null pointer");
    long threads = groups * 8;
    dim3 grid((unsigned)((threads + 255) / 256));
    hipLaunchKernelGGL(q40_quantize_kernel, grid, dim3(256), 0, (hipStream_t)stream,
                       (const u32x4 *)in, (uint8_t *)w, (half_t *)s, groups);
    return launch_status();
}

extern "C" int smh_q40_quantize_f32(const void *in, int src_bf16, void *w, void *s, long groups, smh_stream_t stream) {
    using namespace smh;
    SMH_REQUIRE(groups >= 0 && (groups & 1) == 0, "smh_q40_quantize_f32: groups=%ld must be even", groups);
    if (groups == 0) return 0;
    SMH_REQUIRE(in && w && s && ((uintptr_t)in & 15) == 0, "smh_q40_quantize_f32: null or misaligned pointer");
    long threads = groups * 8;
    dim3 grid((unsigned)((threads + 255) / 256));
    if (src_bf16) hipLaunchKernelGGL(q40_quantize_f32_kernel<true>, grid, dim3(256), 0, (hipStream_t)stream, (const f4 *)in, (uint8_t *)w, (half_t *)s, groups);
    else hipLaunchKernelGGL(q40_quantize_f32_kernel<false>, grid, dim3(256), 0, (hipStream_t)stream, (const f4 *)in, (uint8_t *)w, (half_t *)s, groups);
    return launch_status();
}

extern "C" int smh_q40_quantize_t(const void *in, int src_type, int N, int K, void *w, void *s, smh_stream_t stream) {
    using namespace smh;
    SMH_REQUIRE(src_type >= 0 && src_type <= 2, "smh_q40_quantize_t: src_type=%d (0 fp16, 1 bfloat16, 2 fp32)", src_type);
    SMH_REQUIRE(N > 0 && N % 128 == 0 && K > 0, "smh_q40_quantize_t: N=%d (a positive multiple of 128) K=%d", N, K);
    SMH_REQUIRE(in && w && s && ((uintptr_t)in & (src_type == 2 ? 3 : 1)) == 0 && ((uintptr_t)w & 7) == 0 && ((uintptr_t)s & 3) == 0,
                "smh_q40_quantize_t: null or misaligned pointer");
    const int tile_k = QT_ROW / (src_type == 2 ? 4 : 2), k_tiles = (K + tile_k - 1) / tile_k;
    const long blocks = ((long)(N / 128) * k_tiles + 7) / 8 * 8;
    SMH_REQUIRE(blocks < (1L << 31), "smh_q40_quantize_t: N=%d K=%d is too large for one launch", N, K);
    // Two blocks of outputs share a line of codes.  Where an XCD walks all blocks of outputs at one k, and there are more than run at a time, all it reads
    // at a time lies at one offset of many rows, in few memory channels: from 64 on it takes two blocks along k instead.  us, all blocks and two: 11008 x
    // 4096 bfloat16 30.9 and 28.8, 28672 x 8192 136 and 127, 8192 x 8192 fp32 99 and 64, fp16 43.4 and 44.0; below, 4096 x 4096 bfloat16 12.7 and 13.5,
    // 4096 x 8192 fp16 23.3 and 25.6.
    const int together = N / 128 >= 64 ? 2 : N / 128;
    const auto kern = src_type == 0 ? q40_quantize_t_kernel<0> : src_type == 1 ? q40_quantize_t_kernel<1> : q40_quantize_t_kernel<2>;
    hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(QT_THREADS), 0, (hipStream_t)stream, (const uint8_t *)in, N, K, (uint8_t *)w, (half_t *)s, k_tiles, together);
    return launch_status();
}
