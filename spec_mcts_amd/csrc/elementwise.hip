// Small fused kernels around the Q4_0 linears: RMSNorm, SiLU*up, greedy argmax, RoPE (+ Q4_0
// append of the new K/V row) and the branch fork copy.  All are launch- or HBM-bound; the point of
// fusing is to keep a decode step at a handful of launches, not arithmetic.
#include "smh_common.hpp"

namespace smh {

// ---- RMSNorm: fp32 normalise -> fp16 -> * weight -> fp16 ------------------------------------------
// one workgroup per row; dim % 8 == 0
__global__ __launch_bounds__(256) void rmsnorm_kernel(const half_t *__restrict__ x, const half_t *__restrict__ wt,
                                                      half_t *__restrict__ out, int dim, float eps) {
    __shared__ float s_part[4];
    const long row = blockIdx.x;
    const half_t *xr = x + row * dim;
    half_t *orow = out + row * dim;
    float ss = 0.f;
    for (int i = threadIdx.x * 8; i < dim; i += 256 * 8) {
        h8 v = *reinterpret_cast<const h8 *>(xr + i);
#pragma unroll
        for (int j = 0; j < 8; ++j) ss += (float)v[j] * (float)v[j];
    }
    ss = wave_sum(ss);
    if ((threadIdx.x & 63) == 0) s_part[threadIdx.x >> 6] = ss;
    __syncthreads();
    const float total = s_part[0] + s_part[1] + s_part[2] + s_part[3];
    const float r = rms_factor(total, dim, eps);
    for (int i = threadIdx.x * 8; i < dim; i += 256 * 8) {
        h8 v = *reinterpret_cast<const h8 *>(xr + i);
        h8 w = *reinterpret_cast<const h8 *>(wt + i);
        h8 o;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            half_t n = scale_to_half(v[j], r);
            o[j] = n * w[j];
        }
        *reinterpret_cast<h8 *>(orow + i) = o;
    }
}

// ---- SwiGLU gate: fp16(silu(g)) * u ------------------------------------------------------------------
__global__ __launch_bounds__(256) void silu_mul_kernel(const half_t *__restrict__ g, const half_t *__restrict__ u,
                                                       half_t *__restrict__ out, long n) {
    long i = ((long)blockIdx.x * 256 + threadIdx.x) * 8;
    if (i + 8 <= n) {
        h8 a = *reinterpret_cast<const h8 *>(g + i);
        h8 b = *reinterpret_cast<const h8 *>(u + i);
        h8 o;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            float af = (float)a[j];
            half_t sl = (half_t)(af / (1.0f + expf(-af)));
            o[j] = sl * b[j];
        }
        *reinterpret_cast<h8 *>(out + i) = o;
    } else {
        for (; i < n; ++i) {
            float af = (float)g[i];
            half_t sl = (half_t)(af / (1.0f + expf(-af)));
            out[i] = sl * u[i];
        }
    }
}

// ---- greedy pick: largest logit, lowest index on ties --------------------------------------------------
__device__ __forceinline__ void argmax_merge(float &bv, int &bi, float v, int i) {
    if (v > bv || (v == bv && i < bi)) { bv = v; bi = i; }
}
// one workgroup of 1024 threads per row; 128-bit loads, four in flight per thread, when the row allows them
__global__ __launch_bounds__(1024) void argmax_kernel(const half_t *__restrict__ logits, int vocab, long ld,
                                                      int64_t *__restrict__ out) {
    __shared__ float s_v[16];
    __shared__ int s_i[16];
    const half_t *row = logits + (long)blockIdx.x * ld;
    float bv = -INFINITY;
    int bi = 0x7fffffff;
    const bool wide = (ld % 8 == 0) && ((reinterpret_cast<uintptr_t>(logits) & 15) == 0);
    const int chunks = wide ? vocab / 8 : 0;
    for (int c0 = threadIdx.x; c0 < chunks; c0 += 4 * 1024) {
        h8 v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int c = c0 + 1024 * j;
            if (c < chunks) v[j] = *reinterpret_cast<const h8 *>(row + 8 * c);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int c = c0 + 1024 * j;
            if (c < chunks) {
#pragma unroll
                for (int e = 0; e < 8; ++e) argmax_merge(bv, bi, (float)v[j][e], 8 * c + e);
            }
        }
    }
    for (int i = 8 * chunks + threadIdx.x; i < vocab; i += 1024) argmax_merge(bv, bi, (float)row[i], i);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        float ov = __shfl_xor(bv, o, 64);
        int oi = __shfl_xor(bi, o, 64);
        argmax_merge(bv, bi, ov, oi);
    }
    if ((threadIdx.x & 63) == 0) { s_v[threadIdx.x >> 6] = bv; s_i[threadIdx.x >> 6] = bi; }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < 16; ++w) argmax_merge(bv, bi, s_v[w], s_i[w]);
        out[blockIdx.x] = (bi == 0x7fffffff) ? 0 : bi;
    }
}

// ---- RoPE, rotate-half form, three fp16 roundings per element ----------------------------------------
// lane i of a wave owns the pair (i, i + 64) of one 128-wide head vector
__device__ __forceinline__ void rope_pair(half_t &x1, half_t &x2, half_t cs, half_t sn) {
#pragma clang fp contract(off)      // the two products are rounded to fp16 before they are added
    half_t a = x1 * cs, b = (-x2) * sn;     // q*cos, rotate_half(q)*sin for the first half
    half_t c = x2 * cs, d = x1 * sn;        // same for the second half
    x1 = a + b;
    x2 = c + d;
}

// code = rint(fp16(x / scale)), NaN -> 0 (same as the flat quantiser)
__device__ __forceinline__ int kv_code(half_t x, float scale) {
    float qf = (float)(half_t)((float)x / scale);
    if (!(qf == qf)) return 0;
    return (int)__builtin_rintf(qf);
}

// Quantise one 128-wide vector held as (lo = element lane, hi = element lane+64) into one packed row.
__device__ __forceinline__ void kv_store_row(half_t lo, half_t hi, uint8_t *row, half_t *scales, int lane) {
    uint32_t a_lo = (uint32_t)(__builtin_bit_cast(uint16_t, lo) & 0x7FFFu);
    uint32_t a_hi = (uint32_t)(__builtin_bit_cast(uint16_t, hi) & 0x7FFFu);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        a_lo = max(a_lo, (uint32_t)__shfl_xor((int)a_lo, o, 64));
        a_hi = max(a_hi, (uint32_t)__shfl_xor((int)a_hi, o, 64));
    }
    half_t s0 = (half_t)((float)__builtin_bit_cast(half_t, (uint16_t)a_lo) / 7.0f);   // group of elements 0..63
    half_t s1 = (half_t)((float)__builtin_bit_cast(half_t, (uint16_t)a_hi) / 7.0f);   // group of elements 64..127
    int c0 = kv_code(lo, (float)s0), c1 = kv_code(hi, (float)s1);
    row[lane] = (uint8_t)(((c0 & 15) << 4) | (c1 & 15));
    if (lane == 0) { scales[0] = s0; scales[1] = s1; }
}

// decode step: one wave per (branch, head); heads 0..H-1 are queries, H..H+Hkv-1 are key/value heads
__global__ __launch_bounds__(256) void rope_append_kv_kernel(half_t *__restrict__ q, half_t *__restrict__ k,
                                                             const half_t *__restrict__ v, int B, int H, int Hkv,
                                                             const half_t *__restrict__ cos_tab, const half_t *__restrict__ sin_tab,
                                                             const int32_t *__restrict__ pos_dev,
                                                             uint8_t *__restrict__ cache_k, half_t *__restrict__ cache_ks,
                                                             uint8_t *__restrict__ cache_v, half_t *__restrict__ cache_vs,
                                                             int Smax, const int32_t *__restrict__ t_dev) {
    const int lane = threadIdx.x & 63;
    const long item = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int heads = H + Hkv;
    if (item >= (long)B * heads) return;
    const int b = (int)(item / heads);
    const int h = (int)(item % heads);
    const int pos = *pos_dev;
    const half_t cs = cos_tab[(long)pos * 64 + lane];
    const half_t sn = sin_tab[(long)pos * 64 + lane];
    if (h < H) {
        half_t *p = q + ((long)b * H + h) * 128;
        half_t x1 = p[lane], x2 = p[lane + 64];
        rope_pair(x1, x2, cs, sn);
        p[lane] = x1;
        p[lane + 64] = x2;
        return;
    }
    const int hk = h - H;
    half_t *pk = k + ((long)b * Hkv + hk) * 128;
    half_t x1 = pk[lane], x2 = pk[lane + 64];
    rope_pair(x1, x2, cs, sn);
    pk[lane] = x1;
    pk[lane + 64] = x2;
    if (cache_k == nullptr) return;
    const int t = *t_dev;
    if (t < 0 || t >= Smax) return;
    const long row = ((long)b * Smax + t) * Hkv + hk;
    kv_store_row(x1, x2, cache_k + row * 64, cache_ks + row * 2, lane);
    const half_t *pv = v + ((long)b * Hkv + hk) * 128;
    kv_store_row(pv[lane], pv[lane + 64], cache_v + row * 64, cache_vs + row * 2, lane);
}

// prefill: q [S,H,128], k [S,Hkv,128]; token s sits at position pos0 + s.  One thread owns eight rotation pairs (d .. d+7 and
// d+64 ..) of one head: 16-byte loads and stores (with a pair a thread, 2-byte accesses: 19.7 us at 2047 rows of the 7B shape)
__global__ __launch_bounds__(256) void rope_kernel(half_t *__restrict__ q, half_t *__restrict__ k, int S, int H, int Hkv,
                                                   const half_t *__restrict__ cos_tab, const half_t *__restrict__ sin_tab, int pos0) {
    const int s = blockIdx.y, item = blockIdx.x * 256 + threadIdx.x, h = item >> 3, d = 8 * (item & 7);
    if (h >= H + Hkv) return;
    half_t *p = ((h < H) ? q + ((long)s * H + h) * 128 : k + ((long)s * Hkv + (h - H)) * 128) + d;
    h8 cs, sn, lo, hi;                                       // (copies: the tensors may start at any element)
    __builtin_memcpy(&cs, cos_tab + (long)(pos0 + s) * 64 + d, 16);
    __builtin_memcpy(&sn, sin_tab + (long)(pos0 + s) * 64 + d, 16);
    __builtin_memcpy(&lo, p, 16);
    __builtin_memcpy(&hi, p + 64, 16);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        half_t x1 = lo[j], x2 = hi[j];
        rope_pair(x1, x2, cs[j], sn[j]);
        lo[j] = x1;
        hi[j] = x2;
    }
    __builtin_memcpy(p, &lo, 16);
    __builtin_memcpy(p + 64, &hi, 16);
}

// ---- fork: copy one branch's cache row to `forks` other branches ------------------------------------------
__global__ __launch_bounds__(256) void kv_fork_kernel(u32x4 *__restrict__ cache, long row_vec, int origin, int curr) {
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    if (i >= row_vec) return;
    const int dst = curr + blockIdx.y;
    cache[(long)dst * row_vec + i] = cache[(long)origin * row_vec + i];
}

}  // namespace smh

extern "C" int smh_rmsnorm(const void *x, const void *weight, void *out, int rows, int dim, float eps, smh_stream_t stream) {
    using namespace smh;
    SMH_REQUIRE(rows >= 0 && dim > 0 && dim % 8 == 0, "smh_rmsnorm: rows=%d dim=%d (dim must be a multiple of 8)", rows, dim);
    if (rows == 0) return 0;
    SMH_REQUIRE(x && weight && out, "smh_rmsnorm: null pointer");
    hipLaunchKernelGGL(rmsnorm_kernel, dim3(rows), dim3(256), 0, (hipStream_t)stream,
                       (const half_t *)x, (const half_t *)weight, (half_t *)out, dim, eps);
    return launch_status();
}

extern "C" int smh_silu_mul(const void *g, const void *u, void *out, long n, smh_stream_t stream) {
    using namespace smh;
    SMH_REQUIRE(n >= 0, "smh_silu_mul: n=%ld", n);
    if (n == 0) return 0;
    SMH_REQUIRE(g && u && out, "smh_silu_mul: null pointer");
    long blocks = (n + 2047) / 2048;
    hipLaunchKernelGGL(silu_mul_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream,
                       (const half_t *)g, (const half_t *)u, (half_t *)out, n);
    return launch_status();
}

namespace smh {

// ---- temperature / top-k sampling -----------------------------------------------------------------------------
// One 1024-thread workgroup per row.  x = fp16(logit / temperature) (the reference divides fp16 tensors); the k largest
// x, equal values taken lowest index first, are found by the threads' maxima (k above 512 and rows of mostly equal logits: with a
// two-pass radix select, 256-bin histograms in LDS) on an order-preserving 16-bit key, gathered, ordered by (x descending, index ascending) with a rank sort, turned into
// probabilities p = fp16(softmax) as F.softmax on an fp16 tensor returns them, and one candidate is drawn by inverse
// CDF with the caller's uniform number.
constexpr int SAMPLE_MAX_K = 1024;
constexpr int SAMPLE_HOT_MAX = 576;            // threads whose logits are looked at again
// Up to here the bound is guessed from sixteenths of the maxima.  The guess takes k / 14 + 1 steps and saves three rounds.  80 rows of 32016, us, without and with
// one: k = 32 7.2 and 6.8, 65 9.0 and 8.8, 96 9.4 and 9.6.
constexpr int SAMPLE_GUESS_MAX_K = 80;
constexpr int SAMPLE_PICK_MAX_K = 512;         // up to here the candidates are picked by the threads' maxima (above, they would be thousands)

__device__ __forceinline__ uint32_t sample_key(half_t x) {
    const uint32_t b = __builtin_bit_cast(uint16_t, x);
    return (b & 0x8000u) ? (~b & 0xFFFFu) : (b | 0x8000u);       // larger value <=> larger key
}
// ... of two fp16 values in one word
typedef int16_t s16x2 __attribute__((ext_vector_type(2)));
typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t sample_keys2(uint32_t b) {
    const uint32_t neg = __builtin_bit_cast(uint32_t, __builtin_bit_cast(s16x2, b) >> 15);       // 0xFFFF in the halves that are negative
    return b ^ (neg | 0x80008000u);
}
__device__ __forceinline__ half_t sample_unkey(uint32_t k) {
    const uint16_t b = (uint16_t)((k & 0x8000u) ? (k & 0x7FFFu) : (~k & 0xFFFFu));
    return __builtin_bit_cast(half_t, b);
}

// the largest value of a lane's row of sixteen lanes (in all of them), and of the wave
__device__ __forceinline__ uint32_t row16_max_bits(uint32_t v) {
    auto move = [&](auto ctrl) { v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, decltype(ctrl)::value, 0xf, 0xf, false)); };
    move(std::integral_constant<int, DPP_QUAD_XOR1>{});
    move(std::integral_constant<int, DPP_QUAD_XOR2>{});
    move(std::integral_constant<int, DPP_ROW_HALF_MIRROR>{});
    move(std::integral_constant<int, DPP_ROW_ROR8>{});
    return v;
}
__device__ __forceinline__ uint32_t wave_max_bits(uint32_t v) {
    const int r = (int)row16_max_bits(v);
    auto of = [&](int lane) { return (uint32_t)__builtin_amdgcn_readlane(r, lane); };
    return max(max(of(0), of(16)), max(of(32), of(48)));
}

// Inclusive prefix sum over the wave (lane order) without LDS: within rows of sixteen lanes, then a row's last lane to the next row, then lane 31 to the upper half
__device__ __forceinline__ int wave_prefix_sum(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);        // lane i - 1, - 2, - 4, - 8 of the row
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);        // rows 1 and 3
    return v + __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // rows 2 and 3
}

// Inclusive prefix sums over the 1024 threads of the workgroup (thread order): inside a wave by lane shifts, across waves
// through s_w[16]; two barriers.  Every thread of the workgroup must call.
template <class T>
__device__ __forceinline__ T sample_block_scan(T v, T *s_w) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const T t = __shfl_up(v, o, 64);
        if (lane >= o) v += t;
    }
    if (lane == 63) s_w[wave] = v;
    __syncthreads();
    T base = 0;
    for (int w = 0; w < wave; ++w) base += s_w[w];
    __syncthreads();
    return v + base;
}

// bins[t] <- sum of bins[t..255]; then the bin where the count from the top reaches `want` and the count above it
__device__ __forceinline__ void sample_pick_bin(int *bins, int *s_w, int want, int *out_bin, int *out_above) {
    const int t = threadIdx.x;
    const int mine = t < 256 ? bins[255 - t] : 0;                 // thread t holds bin 255 - t: a prefix sum from the top
    const int upto = sample_block_scan(mine, s_w);
    if (t < 256) bins[255 - t] = upto;
    __syncthreads();
    if (t < 256) {
        const int above = t == 255 ? 0 : bins[t + 1];
        if (bins[t] >= want && above < want) { *out_bin = t; *out_above = above; }
    }
    __syncthreads();
}

// counts == nullptr: one draw per row, uniform[row] -> out[row].  Otherwise row r makes counts[r] draws with replacement from
// its candidates, with the uniform numbers (and into the slots of out) that start at counts[0] + ... + counts[r-1].
// Up to 32768 logits (a multiple of 8, rows 16-byte aligned) and k <= 512 the row is read once into registers and the candidates
// are those not below a bound that about k of the threads' maxima reach (a handful more than k): no histogram of the whole row, whose LDS
// atomics pile up on the few bins that logits fall into.  80 rows of 32016, k = 32: 35 us with histograms, 7.2 with the k-th largest maximum, four bits at
// a time, and 6.7 with a bound guessed in one round (k = 1, 16 rows: 6.5 and 5.6; k = 512, 31 and 26, by the ranking's shares).
// Bound by its instructions (sixteen waves on a compute unit: 18 cycles each for all of them) and a chain of barriers.  So keys are made and
// compared two to an instruction, only the few threads whose maximum reaches the bound hand their logits out, one to a thread, instead
// of every wave looking through 32 (12.3 us with that), and what the draws need is on its way from the start.
// Otherwise, and where the maxima leave more than 1024 candidates (ordered or mostly equal logits), two histogram passes: thread
// t owns the contiguous chunk of ceil(vocab / 1024) logits that starts at t times that.
__global__ __launch_bounds__(1024) void sample_topk_kernel(const half_t *__restrict__ logits, int vocab, long ld, float temperature,
                                                           int top_k, const float *__restrict__ uniform, int64_t *__restrict__ out,
                                                           const int32_t *__restrict__ counts, const float *__restrict__ row_temps, int n_draws,
                                                           int keep_ties) {
    // row_temps: a temperature per row, applied in fp32 (a tensor divisor promotes the fp16 logits to fp32 in torch, a
    // Python scalar does not): candidates by the raw logits (division by a positive number keeps their order, and two
    // different fp16 values stay different in fp32), softmax and probabilities in fp32
    // keep_ties: the filter form of top-k (everything below the k-th largest value is masked, so EVERY value equal to it
    // stays a candidate - up to SAMPLE_MAX_K candidates in all), on fp32 logits / temperature
    const bool wide = row_temps != nullptr || keep_ties;
    if (row_temps != nullptr) temperature = row_temps[blockIdx.x];
    // a row temperature that is not positive (a ramp that reaches 0, a NaN) has no softmax: the row draws its largest logit
    // every time (the limit of the distribution as the temperature goes to 0), lowest index first among equals
    const bool greedy_row = row_temps != nullptr && !(temperature > 0.f);
    if (greedy_row) temperature = 1.0f;
    __shared__ int bins[256];
    __shared__ __attribute__((aligned(16))) uint32_t hot_words[SAMPLE_HOT_MAX * 16];
    __shared__ int hot_tid[SAMPLE_HOT_MAX];
    int *const wbins = reinterpret_cast<int *>(hot_words);                 // [256 * 16]
    static_assert(SAMPLE_HOT_MAX >= 256, "the histograms fit");
    __shared__ int s_wi[16];
    __shared__ float s_wf[16];
    __shared__ int s_bin, s_above, s_count, s_hot;
    __shared__ int s_first, s_draws;
    __shared__ float s_uniform[64];
    __shared__ __attribute__((aligned(16))) uint32_t c_key[SAMPLE_MAX_K];
    __shared__ int c_idx[SAMPLE_MAX_K];
    __shared__ uint32_t o_key[SAMPLE_MAX_K];
    __shared__ int o_idx[SAMPLE_MAX_K];
    __shared__ float cdf[SAMPLE_MAX_K];
    const int tid = threadIdx.x;
    const half_t *row = logits + (long)blockIdx.x * ld;
    int k = min(top_k, vocab);
    auto key_of = [&](half_t x) { return sample_key(wide ? x : (half_t)((float)x / temperature)); };
    auto value_of = [&](uint32_t key) { return wide ? (float)sample_unkey(key) / temperature : (float)sample_unkey(key); };
    const int wv = tid >> 6, lane = tid & 63;

    // One wave: which draws are this row's (the counts of the rows before it added up, all loads together) and the uniform numbers of the
    // first 64.  Every sum is cut at n_draws < 2^31 - counts that add up to more than the buffers hold are cut - so none of these
    // unsigned sums wraps.
    float my_uniform = 0.f;                    // (left in s_uniform when it is there: waited for at once, it kept the others at their first barrier)
    auto find_draws = [&]() {
        int first = blockIdx.x, draws = 1;
        if (counts != nullptr) {
            const uint32_t most = (uint32_t)max(n_draws, 0);
            uint32_t sum = 0;
            for (int r = lane; r < (int)blockIdx.x; r += 64) sum = min(sum + (uint32_t)max(counts[r], 0), most);
            const int own = counts[blockIdx.x];
            auto add = [&](auto ctrl) { sum = min(sum + (uint32_t)__builtin_amdgcn_update_dpp(0, (int)sum, decltype(ctrl)::value, 0xf, 0xf, false), most); };
            add(std::integral_constant<int, DPP_QUAD_XOR1>{});
            add(std::integral_constant<int, DPP_QUAD_XOR2>{});
            add(std::integral_constant<int, DPP_ROW_HALF_MIRROR>{});
            add(std::integral_constant<int, DPP_ROW_ROR8>{});
            auto row = [&](int l) { return (uint32_t)__builtin_amdgcn_readlane((int)sum, l); };
            sum = min(min(row(0) + row(16), most) + min(row(32) + row(48), most), most);
            first = (int)sum;
            draws = min(max(own, 0), (int)(most - sum));
        }
        if (lane == 0) { s_first = first; s_draws = draws; }
        if (!greedy_row && lane < draws) my_uniform = uniform[first + lane];
    };

    constexpr int CH = 32;
    const bool in_regs = vocab <= 1024 * CH && vocab % 8 == 0 && (reinterpret_cast<uintptr_t>(row) & 15) == 0;     // (uniform)
    bool found = false;                        // the candidates are in o_key / o_idx, in order
    const bool by_maxima = in_regs && k <= SAMPLE_PICK_MAX_K;
    if (by_maxima) {
        // ---- candidates by the threads' maxima ----
        // At least k logits are not below the k-th largest of the 1024 threads' own maxima, so the k largest are among those
        // that are not (about k + k^2 / 64 of them for unordered logits).  Order and equality are those of the
        // quotients; the quotient is monotonic, so the logits themselves are compared, down to the smallest one with the same
        // quotient.
        uint32_t raw[CH / 2];
        u32x4 from[CH / 8];
#pragma unroll
        for (int q = 0; q < CH / 8; ++q) {
            const int i = 8 * (tid + 1024 * q);
            from[q] = u32x4{0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFFFFFFu};  // key 0: below every number
            if (i < vocab) from[q] = *reinterpret_cast<const u32x4 *>(row + i);
        }
        if (wv == 0) find_draws();
#pragma unroll
        for (int q = 0; q < CH / 8; ++q)
#pragma unroll
            for (int j = 0; j < 4; ++j) raw[4 * q + j] = sample_keys2(from[q][j]);
        u16x2 two = __builtin_bit_cast(u16x2, raw[0]);
#pragma unroll
        for (int j = 1; j < CH / 2; ++j) two = __builtin_elementwise_max(two, __builtin_bit_cast(u16x2, raw[j]));
        const uint32_t mx = max((uint32_t)two[0], (uint32_t)two[1]);
        uint32_t *maxima = hot_words;
        maxima[tid] = mx;
        if (tid == 0) s_count = s_hot = 0;
        __syncthreads();
        uint32_t mine[16];                     // every wave holds all the maxima ...
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const u32x4 v = *reinterpret_cast<const u32x4 *>(&maxima[256 * j + 4 * lane]);
#pragma unroll
            for (int e = 0; e < 4; ++e) mine[4 * j + e] = v[e];
        }
        // A bound that at least k maxima reach: thr, where fewer than k reach over.  It need not be the k-th largest, as long as only a few threads more reach it.
        auto reach = [&](uint32_t t) {
            int n = 0;
#pragma unroll
            for (int j = 0; j < 16; ++j) n += __popcll(__ballot(mine[j] >= t));
            return n;
        };
        const int wave = __builtin_amdgcn_readfirstlane(wv);
        int *slot = bins;
        uint32_t thr = 0;
        if (k <= SAMPLE_GUESS_MAX_K) {
            // Sixteen guesses: each wave's r-th largest of a sixteenth of the maxima, r = k / 14 + 1 (from k = 13 on 1.16 to 2.3 times k / 16), of which k to
            // k + 32 maxima reach one in two or three (unordered logits, 300 rows at each k up to 80: one row needed a further round, at k = 68).
            uint32_t v = maxima[16 * lane + ((wave + (lane >> 2)) & 15)], t = 0, over = 0x10000u;
            for (int r = k / 14; r >= 0; --r) {
                t = wave_max_bits(v);
                if (lane == __builtin_ctzll(__ballot(v == t))) v = 0u;
            }
            const int n = reach(t);
            if (lane == 0) slot[wave] = (int)(t << 11 | (uint32_t)n);
            __syncthreads();
            const uint32_t g = (uint32_t)slot[lane & 15], at = g & 2047u;
            const uint32_t best = __builtin_amdgcn_readfirstlane(row16_max_bits(at >= (uint32_t)k ? g : 0u));         // the highest that k reach
            int reached = 1024;
            if (best != 0) { thr = best >> 11; reached = (int)(best & 2047u); }
            over -= __builtin_amdgcn_readfirstlane(row16_max_bits(at < (uint32_t)k ? 0x10000u - (g >> 11) : 0u));      // the lowest that fewer do
            while (over - thr > 1 && reached > k + 32) {       // every wave counts at one of sixteen values between the two
                slot += 16;
                const uint32_t step = (over - thr + 14) >> 4;
                const int m = reach(min(thr + 1 + (uint32_t)wave * step, over));
                if (lane == 0) slot[wave] = m;
                __syncthreads();
                const int now = slot[lane & 15], most = __popcll(__ballot(now >= k) & 0xFFFFull);      // (the counts fall from wave to wave)
                over = min(thr + 1 + (uint32_t)most * step, over);
                if (most > 0) {
                    reached = __builtin_amdgcn_readlane(now, most - 1);
                    thr += 1 + (uint32_t)(most - 1) * step;
                }
            }
        } else {
#pragma unroll
            for (int shift = 12; shift >= 0; shift -= 4) {     // every wave counts at one value of the next four bits
                const int n = reach(thr | ((uint32_t)wave << shift));
                if (lane == 0) slot[wave] = n;
                __syncthreads();
                // (the counts fall from wave to wave, and the first one's reaches k)
                thr |= (uint32_t)(__popcll(__ballot(slot[lane & 15] >= k) & 0xFFFFull) - 1) << shift;
                slot += 16;
            }
        }
        bool small = true;
        if (!wide) {                           // (one candidate a lane: thr - lane)
            const bool same = key_of(sample_unkey(thr - min((uint32_t)lane, thr))) == key_of(sample_unkey(thr)) && (uint32_t)lane <= thr;
            const int steps = __builtin_ctzll(~(__ballot(same) >> 1));
            thr -= steps;
            small = steps < 63;
        }
        if (wv == 0) s_uniform[lane] = my_uniform;
        const bool real = small && thr > 0;                     // (key 0: also the slots past the row)
        // the threads whose maximum reaches the bound leave their keys, in any order
        const bool hot = real && mx >= thr;
        const uint64_t hots = __ballot(hot);
        if (hots != 0) {                       // (uniform)
            int at = 0;
            if (lane == 0) at = atomicAdd(&s_hot, __popcll(hots));
            at = __builtin_amdgcn_readfirstlane(at) + __popcll(hots & ((1ull << lane) - 1));
            if (hot && at < SAMPLE_HOT_MAX) {
#pragma unroll
                for (int j = 0; j < 4; ++j) *reinterpret_cast<u32x4 *>(&hot_words[16 * at + 4 * j]) = u32x4{raw[4 * j], raw[4 * j + 1], raw[4 * j + 2], raw[4 * j + 3]};
                hot_tid[at] = tid;
            }
        }
        __syncthreads();
        const int n_hot = s_hot;
        if (real && n_hot <= SAMPLE_HOT_MAX) {
            for (int x0 = 0; x0 < 32 * n_hot; x0 += 1024) {
                const int x = x0 + tid;
                uint32_t key = 0;
                if (x < 32 * n_hot) key = reinterpret_cast<const uint16_t *>(hot_words)[x];
                const bool in = key >= thr;
                const uint64_t ins = __ballot(in);
                if (ins != 0) {                // (uniform)
                    int at = 0;
                    if (lane == 0) at = atomicAdd(&s_count, __popcll(ins));
                    at = __builtin_amdgcn_readfirstlane(at) + __popcll(ins & ((1ull << lane) - 1));
                    // key above 32767 - index: one comparison orders by value, then by index
                    const uint32_t j = x & 31, i = 8 * (hot_tid[min(x >> 5, SAMPLE_HOT_MAX - 1)] + 1024 * (j >> 3)) + (j & 7);
                    if (in && at < SAMPLE_MAX_K) c_key[at] = ((wide ? key : key_of(sample_unkey(key))) << 15) | (32767u - i);
                }
            }
            __syncthreads();
            const int count = s_count;
            if (count <= SAMPLE_MAX_K) {
                // rank = number of candidates that come before.  `parts` waves share 64 candidates, each comparing them with every
                // so-many-th quad of the others (the same for all lanes of a wave).
                int part = wave, parts = 16, cand = lane;
                if (count > 64) {
                    const int groups = (__builtin_amdgcn_readfirstlane(count) + 63) >> 6;
                    const int inv = __builtin_amdgcn_readfirstlane((int)(65536.0f * __builtin_amdgcn_rcpf((float)groups))) + 1;
                    part = (wave * inv) >> 16;                 // wave / groups (both at most 16)
                    parts = (16 * inv) >> 16;
                    cand += 64 * (wave - part * groups);
                }
                const uint32_t mine_c = cand < count ? c_key[cand] : 0u;
                if (tid < 1024 - count) c_key[count + tid] = 0u;           // (below every candidate)
                c_idx[tid] = 0;
                __syncthreads();
                int rank = 0;
                for (int j = 4 * part; j < count && part < parts; j += 4 * parts) {
                    const u32x4 v = *reinterpret_cast<const u32x4 *>(&c_key[j]);
#pragma unroll
                    for (int e = 0; e < 4; ++e) rank += v[e] > mine_c;
                }
                if (parts > 1) {
                    if (cand < count && rank > 0) atomicAdd(&c_idx[cand], rank);
                    __syncthreads();
                    rank = c_idx[cand];
                }
                if (part == 0 && cand < count) {
                    o_key[rank] = mine_c >> 15;
                    o_idx[rank] = 32767 - (int)(mine_c & 32767u);
                }
                __syncthreads();
                if (keep_ties) {                               // every value equal to the k-th
                    const uint32_t kth = o_key[k - 1];
                    k += __syncthreads_count(tid >= k && tid < count && o_key[tid] == kth);
                }
                found = true;
            }
        }
    }
    if (!found) {
    // ---- by histograms: many candidates, or rows that cannot be held in registers ----
    __syncthreads();
    const bool hold = in_regs && top_k > SAMPLE_PICK_MAX_K;
    const int chunk = hold ? CH : (vocab + 1023) / 1024;
    const int lo = min(tid * chunk, vocab), hi = min(vocab, lo + chunk);
    uint32_t kr[CH / 2];                       // hold: keys of elements lo + 2 j (low half) and lo + 2 j + 1
    if (hold) {
        u32x4 raw[CH / 8];
#pragma unroll
        for (int q = 0; q < CH / 8; ++q) {
            raw[q] = u32x4{0u, 0u, 0u, 0u};
            if (lo + 8 * q < hi) raw[q] = *reinterpret_cast<const u32x4 *>(row + lo + 8 * q);
        }
#pragma unroll
        for (int j = 0; j < CH / 2; ++j) {
            const uint32_t two = raw[j >> 2][j & 3];
            const uint32_t k0 = key_of(__builtin_bit_cast(half_t, (uint16_t)(two & 0xFFFFu)));
            const uint32_t k1 = key_of(__builtin_bit_cast(half_t, (uint16_t)(two >> 16)));
            kr[j] = k0 | (k1 << 16);
        }
    }
    // f(index, key) for every logit of this thread's chunk, in index order
    auto for_each = [&](auto f) {
        if (hold) {
#pragma unroll
            for (int j = 0; j < CH; ++j)
                if (lo + j < hi) f(lo + j, (kr[j >> 1] >> (16 * (j & 1))) & 0xFFFFu);
        } else {
            for (int i = lo; i < hi; ++i) f(i, key_of(row[i]));
        }
    };

    // ---- the k-th largest key: high byte, then low byte ----
    // Atomics of different waves on one LDS word take turns, and logits crowd into a few high bytes: every wave counts into a
    // histogram of its own (word = bin * 16 + wave, the 16 copies of a bin in 16 banks), which are then added.
    auto fold_bins = [&]() {
        if (tid < 256) {
            int n = 0;
#pragma unroll
            for (int w = 0; w < 16; ++w) n += wbins[tid * 16 + w];
            bins[tid] = n;
        }
        __syncthreads();
    };
    for (int i = tid; i < 256 * 16; i += 1024) wbins[i] = 0;
    if (tid == 0) s_count = 0;
    __syncthreads();
    for_each([&](int, uint32_t key) { atomicAdd(&wbins[(key >> 8) * 16 + wv], 1); });
    __syncthreads();
    fold_bins();
    sample_pick_bin(bins, s_wi, k, &s_bin, &s_above);
    const int b1 = s_bin, above1 = s_above;
    __syncthreads();
    for (int i = tid; i < 256 * 16; i += 1024) wbins[i] = 0;
    __syncthreads();
    for_each([&](int, uint32_t key) {
        if ((int)(key >> 8) == b1) atomicAdd(&wbins[(key & 255u) * 16 + wv], 1);
    });
    __syncthreads();
    fold_bins();
    sample_pick_bin(bins, s_wi, k - above1, &s_bin, &s_above);
    const uint32_t kth = ((uint32_t)b1 << 8) | (uint32_t)s_bin;      // key of the k-th largest value
    int ties_wanted = k - (above1 + s_above);                          // how many of the values equal to it are in
    if (keep_ties) {                                                   // all of them, while the candidate arrays hold them
        ties_wanted = min(bins[s_bin] - s_above, SAMPLE_MAX_K - (above1 + s_above));
        k = above1 + s_above + ties_wanted;
    }
    __syncthreads();

    // ---- gather: everything above the k-th key, and of the ties the lowest indices (the chunks are in index order, so a
    //      prefix sum of the per-thread tie counts gives each tie its rank by index) ----
    int my_ties = 0;
    for_each([&](int, uint32_t key) { my_ties += key == kth; });
    int tie_rank = sample_block_scan(my_ties, s_wi) - my_ties;         // ties at lower indices
    for_each([&](int i, uint32_t key) {
        bool take = key > kth;
        if (key == kth) { take = tie_rank < ties_wanted; ++tie_rank; }
        if (take) {
            const int slot = atomicAdd(&s_count, 1);
            c_key[slot] = key;
            c_idx[slot] = i;
        }
    });
    __syncthreads();

    // ---- order the k candidates: rank = number of candidates that come before (the last wave has none of the first 960) ----
    // (Here its loads are waited for beside the ranking; at the top of the histograms, by the first wave, 16 rows with k = 600 took 81.3 us instead of 79.0.)
    if (!by_maxima && wv == 15) {
        find_draws();
        s_uniform[lane] = my_uniform;
    }
    if (tid < k) {
        const uint32_t mk = c_key[tid];
        const int mi = c_idx[tid];
        int rank = 0;
        for (int j = 0; j < k; ++j) rank += (c_key[j] > mk) || (c_key[j] == mk && c_idx[j] < mi);
        o_key[rank] = mk;
        o_idx[rank] = mi;
    }
    __syncthreads();

    }

    // ---- p = fp16(softmax) (fp32 with a row temperature or the filter form), inverse CDF ----
    const float xmax = value_of(o_key[0]);
    const float e = tid < k ? expf(value_of(o_key[tid]) - xmax) : 0.f;
    const bool one_wave = k <= 64;             // every candidate in the first wave: the same sums without the workgroup's barriers
    auto wave_scan = [&](float v) {
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const float u = __shfl_up(v, o, 64);
            if ((tid & 63) >= o) v += u;
        }
        return v;
    };
    float upto, before, all;                   // cumulative probability with and without candidate tid, and of all
    if (one_wave) {
        if (tid >= 64) return;
        const float total = __shfl(wave_scan(e), k - 1, 64);
        const float pr = tid < k ? (wide ? e / total : (float)(half_t)(e / total)) : 0.f;
        upto = wave_scan(pr);
        all = __shfl(upto, k - 1, 64);
        before = __shfl_up(upto, 1, 64);
        if (tid == 0) before = 0.f;
    } else {
        cdf[tid] = sample_block_scan(e, s_wf);
        __syncthreads();
        const float total = cdf[k - 1];
        __syncthreads();
        const float pr = tid < k ? (wide ? e / total : (float)(half_t)(e / total)) : 0.f;
        cdf[tid] = sample_block_scan(pr, s_wf);
        __syncthreads();
        upto = cdf[tid];
        before = tid == 0 ? 0.f : cdf[tid - 1];
        all = cdf[k - 1];
    }
    const long first = s_first;
    const int draws = s_draws;
    if (greedy_row) {
        for (int j = tid; j < draws; j += one_wave ? 64 : 1024) out[first + j] = o_idx[0];
        return;
    }
    if (tid < k) {
        // first candidate whose cumulative probability exceeds the target (the last one if rounding leaves none)
        auto draw = [&](int j, float target) {
            if ((before <= target && target < upto) || (tid == k - 1 && target >= upto)) out[first + j] = o_idx[tid];
        };
        // (two loops: one load from either address would be a flat one)
        for (int j = 0; j < min(draws, 64); ++j) draw(j, s_uniform[j] * all);
        for (int j = 64; j < draws; ++j) draw(j, uniform[first + j] * all);
    }
}

// The bookkeeping of one step of the tree sampler (mcts.py:127-152) for all branches in one launch, one workgroup.
//   draws   the tokens every live branch drew this step (sample_topk_kernel with counts): branch i owns cnt[i] of them,
//           in branch order
//   per branch i < *curr_b, in order: its distinct tokens in ascending order with their multiplicities (torch.unique,
//           :131); if the branch is alive the smallest stays on row i with its multiplicity (:135-138) and each further
//           distinct token opens a new row while rows are left (:141-150): the new row takes the origin's token
//           history, the token, its multiplicity, and - instead of a copy of K/V rows - the origin's page ids of the
//           suffix rows written so far.  Dead branches change nothing.  Then the step's column of every dead row is
//           zeroed (:160).
//   tok / cnt = output_counts[0] / [1] of the reference; origin[r] = the branch row r was forked from in this step, else -1.
constexpr int TREE_MAX_BATCH = 1024;
// What follows the fork in a step of the search loop (mcts.py:160-175), for the variant that does the whole step in one launch:
// the terminal state machine on the step's column, the lengths and the mask of live rows, the tokens the next forward
// reads, and the two numbers the host needs (branches, ended rows).
struct TreeFinish {
    int32_t *state;              // end_stateMachine [batch_size]
    const int64_t *seq;          // the terminal sequence
    int seq_len;
    int64_t eos;
    int32_t *results_len;        // [batch_size]
    int64_t *next_tokens;        // [batch_size]: column t of results, the next decode step's input
    int32_t *summary;            // [2]: branches after the step, rows that have ended
};
// t_dev != nullptr: the step's column AND the suffix rows written so far are *t_dev (a search step t follows t decode steps),
// read on the device so that one captured launch serves every step.
__global__ __launch_bounds__(256) void tree_fork_kernel(const int64_t *__restrict__ draws, int n_draws, int32_t *__restrict__ tok, int32_t *__restrict__ cnt,
                                                        uint8_t *__restrict__ alive, int32_t *__restrict__ curr_b, int batch_size,
                                                        int64_t *__restrict__ results, long ld, int t,
                                                        int32_t *__restrict__ pages, long pages_stride, int n_rows,
                                                        int32_t *__restrict__ origin, const int32_t *__restrict__ t_dev, TreeFinish fin) {
    if (t_dev != nullptr) {
        t = min(max(*t_dev, 0), (int)ld - 1);                    // (a counter outside the row is cut, never followed)
        n_rows = (int)min((long)t, pages_stride);
    }
    __shared__ uint64_t keys[TREE_MAX_BATCH];      // (branch, token) of every draw, sorted by the whole workgroup
    __shared__ int64_t u_tok[TREE_MAX_BATCH];      // per branch its distinct tokens in ascending order (at the segment's start)
    __shared__ int u_cnt[TREE_MAX_BATCH];          // ... and their multiplicities
    __shared__ int seg_off[TREE_MAX_BATCH + 1];    // first draw of branch i
    __shared__ int seg_uniq[TREE_MAX_BATCH];       // distinct tokens of branch i
    __shared__ int scan[TREE_MAX_BATCH + 1];       // distinct (branch, token) pairs before position i
    __shared__ int start[TREE_MAX_BATCH + 1];      // first position of the u-th distinct pair
    __shared__ int wave_sum[4];
    __shared__ int s_new;                          // branches after the step
    const int tid = threadIdx.x;
    const int c0 = min(max(*curr_b, 0), batch_size);             // (a counter outside the batch is cut, never followed)
    if (tid == 0) {
        int off = 0;
        for (int i = 0; i < c0; ++i) { seg_off[i] = off; off = min(off + min(max(cnt[i], 0), TREE_MAX_BATCH), TREE_MAX_BATCH); }
        seg_off[c0] = off;
    }
    __syncthreads();
    const int total = min(seg_off[c0], min(n_draws, TREE_MAX_BATCH));   // draws the buffer does not hold do not exist
    // key of draw i: its branch (the last one whose segment starts at or before i, found by bisection) above its token;
    // slots past the draws sort to the end
    for (int i = tid; i < TREE_MAX_BATCH; i += 256) {
        uint64_t key = ~0ull;
        if (i < total) {
            int lo = 0, hi = c0 - 1;
            while (lo < hi) {
                const int mid = (lo + hi + 1) >> 1;
                if (seg_off[mid] <= i) lo = mid; else hi = mid - 1;
            }
            key = ((uint64_t)(uint32_t)lo << 32) | (uint64_t)(uint32_t)draws[i];
        }
        keys[i] = key;
    }
    for (int r = tid; r < batch_size; r += 256) origin[r] = -1;
    __syncthreads();
    // bitonic sort of the keys by the whole workgroup, over the smallest power of two that holds the draws (the slots
    // past them hold the largest key and stay behind)
    int n_sort = 2;
    while (n_sort < total) n_sort <<= 1;
    for (int k = 2; k <= n_sort; k <<= 1)
        for (int j = k >> 1; j > 0; j >>= 1) {
            for (int x = tid; x < n_sort / 2; x += 256) {
                const int i = ((x & ~(j - 1)) << 1) | (x & (j - 1));        // the lower index of the pair (i, i + j)
                const uint64_t a = keys[i], b = keys[i + j];
                const bool up = (i & k) == 0;
                if ((a > b) == up) { keys[i] = b; keys[i + j] = a; }
            }
            __syncthreads();
        }
    // run-length encoding by the whole workgroup: a position opens a run when its key differs from its predecessor's
    // (a new branch always does); an exclusive scan numbers the runs, start[u] is where run u begins
    {
        int head[4], local = 0;
        const int base = tid * 4;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int i = base + e;
            head[e] = (i < total && (i == 0 || keys[i] != keys[i - 1])) ? 1 : 0;
            local += head[e];
        }
        int incl = local;                                   // inclusive scan over the 256 threads: wave scan, then wave sums
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int v = __shfl_up(incl, o, 64);
            if ((tid & 63) >= o) incl += v;
        }
        if ((tid & 63) == 63) wave_sum[tid >> 6] = incl;
        __syncthreads();
        int before = incl - local;
        for (int w = 0; w < (tid >> 6); ++w) before += wave_sum[w];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            scan[base + e] = before;
            if (head[e]) start[before] = base + e;
            before += head[e];
        }
        if (tid == 255) { scan[TREE_MAX_BATCH] = before; start[before] = total; }
    }
    __syncthreads();
    const int n_runs = scan[TREE_MAX_BATCH];
    for (int i = tid; i < c0; i += 256) {
        const int lo = min(seg_off[i], total), hi = min(seg_off[i + 1], total);
        seg_uniq[i] = scan[hi] - scan[lo];                  // (scan[total] counts every run: no run opens past the draws)
    }
    for (int u = tid; u < n_runs; u += 256) {
        const int at = start[u];
        const int br = (int)(keys[at] >> 32);
        const int slot = min(seg_off[br], total) + (u - scan[min(seg_off[br], total)]);
        u_tok[slot] = (int64_t)(int32_t)(uint32_t)keys[at];
        u_cnt[slot] = start[u + 1] - at;
    }
    __syncthreads();
    // rows are handed out in branch order (what is left depends on every earlier branch): one thread walks the branches
    if (tid == 0) {
        int cur = c0;
        for (int i = 0; i < c0; ++i) {
            if (!alive[i] || seg_uniq[i] == 0) continue;
            const int lo = seg_off[i];
            tok[i] = (int32_t)u_tok[lo];
            cnt[i] = u_cnt[lo];
            const int forks = min(seg_uniq[i] - 1, batch_size - cur);
            for (int j = 0; j < forks; ++j) {
                origin[cur + j] = i;
                tok[cur + j] = (int32_t)u_tok[lo + 1 + j];
                cnt[cur + j] = u_cnt[lo + 1 + j];
            }
            cur += max(forks, 0);
        }
        s_new = cur;
        *curr_b = cur;
    }
    __syncthreads();
    const int c1 = s_new;
    // token histories and page ids of the new rows, then this step's column
    for (int r = c0; r < c1; ++r) {
        const int o = origin[r];
        for (long j = tid; j < ld; j += 256) results[(long)r * ld + j] = results[(long)o * ld + j];
        if (pages != nullptr)
            for (int j = tid; j < n_rows; j += 256) pages[(long)r * pages_stride + j] = pages[(long)o * pages_stride + j];
    }
    __syncthreads();
    int ended = 0;
    for (int r = tid; r < batch_size; r += 256) {
        int64_t token = results[(long)r * ld + t];
        if (!alive[r]) token = 0;
        else if (r < c1 && (r >= c0 || seg_uniq[r] > 0)) token = tok[r];
        results[(long)r * ld + t] = token;
        if (fin.state != nullptr) {
            // detectTerminal on the step's column (mcts.py:14-28, :162), lengths and mask (:163-164)
            const int32_t st = fin.state[r];
            const int32_t match = (st >= 0 && st < fin.seq_len && fin.seq[st] == token) ? 1 : 0;
            const int32_t nxt = (st + match) * match;
            const bool done = nxt == fin.seq_len || token == fin.eos;
            fin.state[r] = done ? 0 : nxt;
            const bool was = alive[r] != 0;
            fin.results_len[r] += was ? 1 : 0;
            const bool now = was && !done;
            alive[r] = now ? 1 : 0;
            ended += now ? 0 : 1;
            fin.next_tokens[r] = token;
        }
    }
    if (fin.state != nullptr) {
        __syncthreads();                            // (scan[] is free again)
        scan[tid] = ended;
        __syncthreads();
        for (int o = 128; o > 0; o >>= 1) {
            if (tid < o) scan[tid] += scan[tid + o];
            __syncthreads();
        }
        if (tid == 0) { fin.summary[0] = c1; fin.summary[1] = scan[0]; }
    }
}

// The same step for batches and draws of at most 256: a thread is a branch, a draw, a row in turn.  Nothing is walked by one
// thread: a draw finds its rank among its branch's distinct tokens by comparing it with its branch's other draws (one, once the
// tree has its full batch), the rows of the forks come from a prefix sum (a branch's first new row is c0 + the forks of the
// branches before it, cut at the batch), and everything that depends on no other load is requested at the start.  At 80
// branches, us: 28 for tree_fork_kernel (whose first thread reads the counts and the live flags one behind the other), 3.9 where a draw searches for its
// branch and the prefix sums go through LDS, 3.15 where a branch marks its draws and the sums stay in registers (256 branches: 4.2 and 3.5).
constexpr int TREE_SMALL = 256;
__global__ __launch_bounds__(TREE_SMALL) void tree_small_kernel(const int64_t *__restrict__ draws, int n_draws, int32_t *__restrict__ tok, int32_t *__restrict__ cnt,
                                                                uint8_t *__restrict__ alive, int32_t *__restrict__ curr_b, int batch_size,
                                                                int64_t *__restrict__ results, long ld, int t,
                                                                int32_t *__restrict__ pages, long pages_stride, int n_rows,
                                                                int32_t *__restrict__ origin, const int32_t *__restrict__ t_dev, TreeFinish fin) {
    __shared__ uint32_t d_tok[TREE_SMALL];         // token of draw i
    __shared__ uint8_t d_head[TREE_SMALL];         // draw i is the first of its branch with its token
    __shared__ uint8_t d_branch[TREE_SMALL];       // draw i's branch
    __shared__ int seg[TREE_SMALL + 1];            // first draw of branch i
    __shared__ int uniq[TREE_SMALL], row0[TREE_SMALL];
    __shared__ int r_tok[TREE_SMALL], r_cnt[TREE_SMALL], r_origin[TREE_SMALL];
    __shared__ uint8_t r_set[TREE_SMALL], b_alive[TREE_SMALL];
    __shared__ int s_w[4];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    // inclusive prefix sum over the workgroup; every thread calls
    auto block_scan = [&](int v) {
        v = wave_prefix_sum(v);
        if (lane == 63) s_w[wave] = v;
        __syncthreads();
        for (int w = 0; w < wave; ++w) v += s_w[w];
        __syncthreads();
        return v;
    };
    const bool is_row = tid < batch_size;
    const int c0 = min(max(*curr_b, 0), batch_size);             // (a counter outside the batch is cut, never followed)
    if (t_dev != nullptr) t = *t_dev;
    const int my_cnt = is_row ? cnt[tid] : 0;
    const bool was = is_row && alive[tid] != 0;
    const uint32_t my_tok = tid < n_draws ? (uint32_t)draws[tid] : 0u;
    int32_t st = 0, len = 0;
    if (is_row && fin.state != nullptr) { st = fin.state[tid]; len = fin.results_len[tid]; }
    if (t_dev != nullptr) {
        t = min(max(t, 0), (int)ld - 1);                         // (a counter outside the row is cut, never followed)
        n_rows = (int)min((long)t, pages_stride);
    }
    const int64_t old_token = is_row ? results[(long)tid * ld + t] : 0;
    const int64_t seq_token = is_row && fin.state != nullptr && st >= 0 && st < fin.seq_len ? fin.seq[st] : 0;

    d_tok[tid] = my_tok;
    uniq[tid] = 0;
    r_set[tid] = 0;
    r_origin[tid] = -1;
    b_alive[tid] = was ? 1 : 0;
    const int own = tid < c0 ? min(max(my_cnt, 0), TREE_MAX_BATCH) : 0, upto = block_scan(own);
    seg[tid + 1] = upto;
    for (int j = upto - own; j < min(upto, TREE_SMALL); ++j) d_branch[j] = (uint8_t)tid;
    if (tid == 0) seg[0] = 0;
    __syncthreads();
    const int total = min(seg[c0], n_draws);                     // draws the buffer does not hold do not exist
    // ---- this thread's draw: its branch, whether it is the first with its token there, and how many are equal ----
    int br = 0, lo = 0, hi = 0, mult = 0;
    bool head = tid < total;
    if (tid < total) {
        br = d_branch[tid];
        lo = min(seg[br], total);
        hi = min(seg[br + 1], total);
        for (int j = lo; j < hi; ++j) {
            const bool same = d_tok[j] == my_tok;
            mult += same;
            if (same && j < tid) head = false;
        }
    }
    d_head[tid] = head ? 1 : 0;
    if (head) atomicAdd(&uniq[br], 1);
    __syncthreads();
    // ---- rows of the forks, branch by branch ----
    const int forks = (tid < c0 && was && uniq[tid] > 0) ? uniq[tid] - 1 : 0;
    const int end = block_scan(forks);
    row0[tid] = c0 + end - forks;
    if (tid == TREE_SMALL - 1) seg[TREE_SMALL] = end;            // (seg[256] is read only where 256 branches are live: before this scan)
    __syncthreads();
    const int c1 = min(batch_size, c0 + seg[TREE_SMALL]);
    if (head && b_alive[br]) {
        int rank = 0;                                            // distinct tokens of the branch below this one
        for (int j = lo; j < hi; ++j) rank += d_head[j] && d_tok[j] < my_tok;
        const int r = rank == 0 ? br : row0[br] + rank - 1;
        if (r < batch_size) {
            r_tok[r] = (int32_t)my_tok;
            r_cnt[r] = mult;
            r_set[r] = 1;
            if (rank > 0) r_origin[r] = br;
        }
    }
    __syncthreads();
    // token histories (without this step's column) and page ids of the new rows
    {
        const int n_new = c1 - c0, n = n_new * (int)ld;
        for (int i = tid; i < n; i += TREE_SMALL) {
            const int r = c0 + i / (int)ld, j = i - (r - c0) * (int)ld;
            if (j != t) results[(long)r * ld + j] = results[(long)r_origin[r] * ld + j];
        }
        if (pages != nullptr && n_rows > 0)
            for (int i = tid; i < n_new * n_rows; i += TREE_SMALL) {
                const int r = c0 + i / n_rows, j = i - (r - c0) * n_rows;
                pages[(long)r * pages_stride + j] = pages[(long)r_origin[r] * pages_stride + j];
            }
    }
    // ---- this thread's row ----
    int ended = 0;
    if (is_row) {
        const bool set = r_set[tid] != 0;
        if (set) { tok[tid] = r_tok[tid]; cnt[tid] = r_cnt[tid]; }
        origin[tid] = r_origin[tid];
        int64_t token = old_token;
        if (tid >= c0 && tid < c1 && !set) token = 0;            // (never: every new row has been set)
        if (!was) token = 0;
        else if (set) token = (int64_t)r_tok[tid];
        results[(long)tid * ld + t] = token;
        if (fin.state != nullptr) {
            // detectTerminal on the step's column (mcts.py:14-28, :162), lengths and mask (:163-164)
            const int32_t match = (st >= 0 && st < fin.seq_len && seq_token == token) ? 1 : 0;
            const int32_t nxt = (st + match) * match;
            const bool done = nxt == fin.seq_len || token == fin.eos;
            fin.state[tid] = done ? 0 : nxt;
            fin.results_len[tid] = len + (was ? 1 : 0);
            const bool now = was && !done;
            alive[tid] = now ? 1 : 0;
            ended = now ? 0 : 1;
            fin.next_tokens[tid] = token;
        }
    }
    if (tid == 0) *curr_b = c1;
    if (fin.state != nullptr) {
        const int n = __syncthreads_count(ended);
        if (tid == 0) { fin.summary[0] = c1; fin.summary[1] = n; }
    }
}

}  // namespace smh

extern "C" int smh_sample_topk(const void *logits, int rows, int vocab, long ld, float temperature, int top_k,
                               const float *uniform, int64_t *out, smh_stream_t stream) {
    using namespace smh;
    SMH_REQUIRE(rows >= 0 && vocab > 0 && ld >= vocab, "smh_sample_topk: rows=%d vocab=%d ld=%ld", rows, vocab, ld);
    SMH_REQUIRE(top_k >= 1 && top_k <= SAMPLE_MAX_K, "smh_sample_topk: top_k=%d outside [1,%d]", top_k, SAMPLE_MAX_K);
    SMH_REQUIRE(temperature > 0.f, "smh_sample_topk: temperature=%g must be positive (greedy decoding is smh_argmax)", (double)temperature);
    if (rows == 0) return 0;
    SMH_REQUIRE(logits && uniform && out, "smh_sample_topk: null pointer");
    hipLaunchKernelGGL(sample_topk_kernel, dim3(rows), dim3(1024), 0, (hipStream_t)stream, (const half_t *)logits, vocab, ld, temperature,
                       top_k, uniform, out, (const int32_t *)nullptr, (const float *)nullptr, rows, 0);
    return launch_status();
}

extern "C" int smh_sample_topk_filter(const void *logits, int rows, int vocab, long ld, float temperature, int top_k,
                                      const float *uniform, int64_t *out, smh_stream_t stream) {
    using namespace smh;
    SMH_REQUIRE(rows >= 0 && vocab > 0 && ld >= vocab, "smh_sample_topk_filter: rows=%d vocab=%d ld=%ld", rows, vocab, ld);
    SMH_REQUIRE(top_k >= 1 && top_k <= SAMPLE_MAX_K, "smh_sample_topk_filter: top_k=%d outside [1,%d]", top_k, SAMPLE_MAX_K);
    SMH_REQUIRE(temperature > 0.f, "smh_sample_topk_filter: temperature=%g must be positive (greedy decoding is smh_argmax)", (double)temperature);
    if (rows == 0) return 0;
    SMH_REQUIRE(logits && uniform && out, "smh_sample_topk_filter: null pointer");
    hipLaunchKernelGGL(sample_topk_kernel, dim3(rows), dim3(1024), 0, (hipStream_t)stream, (const half_t *)logits, vocab, ld, temperature,
                       top_k, uniform, out, (const int32_t *)nullptr, (const float *)nullptr, rows, 1);
    return launch_status();
}

extern "C" int smh_sample_topk_counts(const void *logits, int rows, int vocab, long ld, float temperature, int top_k,
                                      const float *uniform, const int32_t *counts, int64_t *out, int n_draws, smh_stream_t stream) {
    using namespace smh;
    SMH_REQUIRE(rows >= 0 && rows <= TREE_MAX_BATCH && vocab > 0 && ld >= vocab, "smh_sample_topk_counts: rows=%d (at most %d) vocab=%d ld=%ld", rows, TREE_MAX_BATCH, vocab, ld);
    SMH_REQUIRE(top_k >= 1 && top_k <= SAMPLE_MAX_K, "smh_sample_topk_counts: top_k=%d outside [1,%d]", top_k, SAMPLE_MAX_K);
    SMH_REQUIRE(temperature > 0.f, "smh_sample_topk_counts: temperature=%g must be positive", (double)temperature);
    if (rows == 0) return 0;
    SMH_REQUIRE(logits && uniform && counts && out && n_draws >= 0, "smh_sample_topk_counts: null pointer or n_draws=%d", n_draws);
    hipLaunchKernelGGL(sample_topk_kernel, dim3(rows), dim3(1024), 0, (hipStream_t)stream, (const half_t *)logits, vocab, ld, temperature,
                       top_k, uniform, out, counts, (const float *)nullptr, n_draws, 0);
    return launch_status();
}

extern "C" int smh_sample_topk_rowtemp(const void *logits, int rows, int vocab, long ld, const float *row_temps, int top_k,
                                       const float *uniform, const int32_t *counts, int64_t *out, int n_draws, smh_stream_t stream) {
    using namespace smh;
    SMH_REQUIRE(rows >= 0 && rows <= TREE_MAX_BATCH && vocab > 0 && ld >= vocab, "smh_sample_topk_rowtemp: rows=%d (at most %d) vocab=%d ld=%ld", rows, TREE_MAX_BATCH, vocab, ld);
    SMH_REQUIRE(top_k >= 1 && top_k <= SAMPLE_MAX_K, "smh_sample_topk_rowtemp: top_k=%d outside [1,%d]", top_k, SAMPLE_MAX_K);
    if (rows == 0) return 0;
    SMH_REQUIRE(logits && row_temps && uniform && counts && out && n_draws >= 0, "smh_sample_topk_rowtemp: null pointer or n_draws=%d", n_draws);
    hipLaunchKernelGGL(sample_topk_kernel, dim3(rows), dim3(1024), 0, (hipStream_t)stream, (const half_t *)logits, vocab, ld, 1.0f,
                       top_k, uniform, out, counts, row_temps, n_draws, 0);
    return launch_status();
}

extern "C" int smh_tree_fork(const int64_t *draws, int n_draws, int32_t *tok, int32_t *cnt, const uint8_t *alive, int32_t *curr_b, int batch_size,
                             int64_t *results, long ld, int t, int32_t *pages, long pages_stride, int n_rows, int32_t *origin,
                             smh_stream_t stream) {
    using namespace smh;
    SMH_REQUIRE(batch_size >= 1 && batch_size <= TREE_MAX_BATCH, "smh_tree_fork: batch_size=%d outside [1,%d]", batch_size, TREE_MAX_BATCH);
    SMH_REQUIRE(draws && n_draws >= 0 && tok && cnt && alive && curr_b && results && origin, "smh_tree_fork: null pointer or n_draws=%d", n_draws);
    SMH_REQUIRE(ld >= 1 && t >= 0 && t < ld, "smh_tree_fork: column %d outside the %ld of a row", t, ld);
    SMH_REQUIRE(pages == nullptr || (pages_stride >= n_rows && n_rows >= 0), "smh_tree_fork: n_rows=%d pages_stride=%ld", n_rows, pages_stride);
    const bool small = batch_size <= TREE_SMALL && n_draws <= TREE_SMALL && ld <= (1 << 20);
    hipLaunchKernelGGL(small ? tree_small_kernel : tree_fork_kernel, dim3(1), dim3(256), 0, (hipStream_t)stream, draws, n_draws, tok, cnt,
                       const_cast<uint8_t *>(alive), curr_b, batch_size, results, ld, t, pages, pages_stride, n_rows, origin, (const int32_t *)nullptr, TreeFinish{});
    return launch_status();
}

extern "C" int smh_tree_step(const int64_t *draws, int n_draws, int32_t *tok, int32_t *cnt, uint8_t *alive, int32_t *curr_b, int batch_size,
                             int64_t *results, long ld, const int32_t *t_dev, int32_t *pages, long pages_stride, int32_t *origin,
                             int32_t *state, const int64_t *terminal_seq, int seq_len, int64_t eos, int32_t *results_len,
                             int64_t *next_tokens, int32_t *summary, smh_stream_t stream) {
    using namespace smh;
    SMH_REQUIRE(batch_size >= 1 && batch_size <= TREE_MAX_BATCH, "smh_tree_step: batch_size=%d outside [1,%d]", batch_size, TREE_MAX_BATCH);
    SMH_REQUIRE(draws && n_draws >= 0 && tok && cnt && alive && curr_b && results && origin && t_dev, "smh_tree_step: null pointer or n_draws=%d", n_draws);
    SMH_REQUIRE(ld >= 1 && (pages == nullptr || pages_stride >= 1), "smh_tree_step: ld=%ld pages_stride=%ld", ld, pages_stride);
    SMH_REQUIRE(state && terminal_seq && seq_len >= 1 && results_len && next_tokens && summary, "smh_tree_step: null pointer or seq_len=%d", seq_len);
    TreeFinish fin{state, terminal_seq, seq_len, eos, results_len, next_tokens, summary};
    const bool small = batch_size <= TREE_SMALL && n_draws <= TREE_SMALL && ld <= (1 << 20);      // (row x column products stay in 32 bits)
    hipLaunchKernelGGL(small ? tree_small_kernel : tree_fork_kernel, dim3(1), dim3(256), 0, (hipStream_t)stream, draws, n_draws, tok, cnt, alive, curr_b,
                       batch_size, results, ld, 0, pages, pages_stride, 0, origin, t_dev, fin);
    return launch_status();
}

namespace smh {

// detectTerminal of the tree sampler (mcts.py:14-28), one thread per branch: the state counts how many tokens of the
// terminal sequence the branch has produced in a row; a token that does not continue it sends the state back to 0
// (also when it equals the sequence's first token, as in the reference); the branch ends when the sequence is
// complete or the token is the end-of-sequence id, and an ended branch restarts at state 0.
__global__ __launch_bounds__(256) void detect_terminal_kernel(const int64_t *__restrict__ token, int32_t *__restrict__ state,
                                                             uint8_t *__restrict__ end, const int64_t *__restrict__ seq, int seq_len,
                                                             int64_t eos, int rows) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= rows) return;
    const int64_t tok = token[i];
    const int32_t st = state[i];
    const int32_t match = (st >= 0 && st < seq_len && seq[st] == tok) ? 1 : 0;
    int32_t nxt = (st + match) * match;
    const bool done = nxt == seq_len || tok == eos;
    end[i] = done ? 1 : 0;
    state[i] = done ? 0 : nxt;
}

}  // namespace smh

extern "C" int smh_detect_terminal(const int64_t *token, int32_t *state, uint8_t *end, const int64_t *terminal_seq, int seq_len,
                                   int64_t eos, int rows, smh_stream_t stream) {
    using namespace smh;
    SMH_REQUIRE(rows >= 0 && seq_len >= 1, "smh_detect_terminal: rows=%d seq_len=%d", rows, seq_len);
    if (rows == 0) return 0;
    SMH_REQUIRE(token && state && end && terminal_seq, "smh_detect_terminal: null pointer");
    hipLaunchKernelGGL(detect_terminal_kernel, dim3((rows + 255) / 256), dim3(256), 0, (hipStream_t)stream, token, state, end,
                       terminal_seq, seq_len, eos, rows);
    return launch_status();
}

extern "C" int smh_argmax(const void *logits, int rows, int vocab, long ld, int64_t *out, smh_stream_t stream) {
    using namespace smh;
    SMH_REQUIRE(rows >= 0 && vocab > 0 && ld >= vocab, "smh_argmax: rows=%d vocab=%d ld=%ld", rows, vocab, ld);
    if (rows == 0) return 0;
    SMH_REQUIRE(logits && out, "smh_argmax: null pointer");
    hipLaunchKernelGGL(argmax_kernel, dim3(rows), dim3(1024), 0, (hipStream_t)stream, (const half_t *)logits, vocab, ld, out);
    return launch_status();
}

extern "C" int smh_rope_append_kv(void *q, void *k, const void *v, int B, int H, int Hkv, int D,
                                  const void *cos_tab, const void *sin_tab, const int32_t *pos_dev,
                                  void *cache_k, void *cache_ks, void *cache_v, void *cache_vs,
                                  int Smax, const int32_t *t_dev, smh_stream_t stream) {
    using namespace smh;
    SMH_REQUIRE(D == 128, "smh_rope_append_kv: head dim %d (only 128)", D);
    SMH_REQUIRE(B >= 0 && H > 0 && Hkv > 0, "smh_rope_append_kv: B=%d H=%d Hkv=%d", B, H, Hkv);
    if (B == 0) return 0;
    SMH_REQUIRE(q && k && cos_tab && sin_tab && pos_dev, "smh_rope_append_kv: null pointer");
    SMH_REQUIRE(!cache_k || (v && cache_ks && cache_v && cache_vs && t_dev && Smax > 0), "smh_rope_append_kv: cache arguments incomplete");
    long items = (long)B * (H + Hkv);
    hipLaunchKernelGGL(rope_append_kv_kernel, dim3((unsigned)((items + 3) / 4)), dim3(256), 0, (hipStream_t)stream,
                       (half_t *)q, (half_t *)k, (const half_t *)v, B, H, Hkv, (const half_t *)cos_tab, (const half_t *)sin_tab,
                       pos_dev, (uint8_t *)cache_k, (half_t *)cache_ks, (uint8_t *)cache_v, (half_t *)cache_vs, Smax, t_dev);
    return launch_status();
}

extern "C" int smh_rope(void *q, void *k, int S, int H, int Hkv, int D, const void *cos_tab, const void *sin_tab,
                        int pos0, smh_stream_t stream) {
    using namespace smh;
    SMH_REQUIRE(D == 128, "smh_rope: head dim %d (only 128)", D);
    SMH_REQUIRE(S >= 0 && H > 0 && Hkv > 0 && pos0 >= 0, "smh_rope: S=%d H=%d Hkv=%d pos0=%d", S, H, Hkv, pos0);
    if (S == 0) return 0;
    SMH_REQUIRE(q && k && cos_tab && sin_tab, "smh_rope: null pointer");
    for (int s0 = 0; s0 < S; s0 += 65535) {                  // (rows of a launch: the grid's second dimension)
        const int n = S - s0 < 65535 ? S - s0 : 65535;
        hipLaunchKernelGGL(rope_kernel, dim3((unsigned)(((H + Hkv) * 8 + 255) / 256), (unsigned)n), dim3(256), 0, (hipStream_t)stream,
                           (half_t *)q + (long)s0 * H * 128, (half_t *)k + (long)s0 * Hkv * 128, n, H, Hkv, (const half_t *)cos_tab,
                           (const half_t *)sin_tab, pos0 + s0);
        if (const int st = launch_status()) return st;
    }
    return 0;
}

namespace smh {
__global__ void set_step_kernel(int32_t *state, int pos, int t) {
    state[0] = pos;
    state[1] = t;
}
}  // namespace smh

extern "C" int smh_set_step(int32_t *state, int pos, int t, smh_stream_t stream) {
    SMH_REQUIRE(state != nullptr && pos >= 0 && t >= 0, "smh_set_step: state=%p pos=%d t=%d", (void *)state, pos, t);
    hipLaunchKernelGGL(smh::set_step_kernel, dim3(1), dim3(1), 0, (hipStream_t)stream, state, pos, t);
    return smh::launch_status();
}

extern "C" int smh_kv_fork(void *cache, void *cache_s, int Bmax, long row_bytes, long row_scales,
                           int origin, int curr, int forks, smh_stream_t stream) {
    using namespace smh;
    SMH_REQUIRE(forks >= 0 && origin >= 0 && origin < Bmax && curr >= 0 && curr + forks <= Bmax,
                "smh_kv_fork: origin=%d curr=%d forks=%d Bmax=%d", origin, curr, forks, Bmax);
    SMH_REQUIRE(origin < curr || origin >= curr + forks, "smh_kv_fork: origin inside the destination range");
    SMH_REQUIRE(row_bytes % 16 == 0 && (row_scales * 2) % 16 == 0, "smh_kv_fork: rows must be multiples of 16 bytes");
    if (forks == 0) return 0;
    SMH_REQUIRE(cache && cache_s, "smh_kv_fork: null pointer");
    long v1 = row_bytes / 16, v2 = row_scales * 2 / 16;
    hipLaunchKernelGGL(kv_fork_kernel, dim3((unsigned)((v1 + 255) / 256), forks), dim3(256), 0, (hipStream_t)stream,
                       (u32x4 *)cache, v1, origin, curr);
    hipLaunchKernelGGL(kv_fork_kernel, dim3((unsigned)((v2 + 255) / 256), forks), dim3(256), 0, (hipStream_t)stream,
                       (u32x4 *)cache_s, v2, origin, curr);
    return launch_status();
}
