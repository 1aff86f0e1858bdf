// Consumers of the Q4_0 matmul's K-slice slabs.
//
// The matmul kernels leave `ksplit` slabs partial[s][m][n] (fp32);
// every kernel here first forms acc = sum_s partial[s][m][n] in fp32 (slice order, so the result does not depend on scheduling), rounds
// it ONCE to fp16 - the value the reference's matmul_q40 returns - and then applies the operator
// that follows the linear in the model:
//   partial_reduce_kernel      c = fp16(acc) (+ fp16 residual add)
//   partial_rmsnorm_kernel     h = h_in + fp16(acc);  xn = RMSNorm(h) * weight
//   partial_silu_mul_kernel    out = fp16(silu(fp16(acc_gate))) * fp16(acc_up)
//   partial_rope_append_kernel q,k,v = fp16(acc); RoPE(q,k); Q4_0 append of k,v to the suffix cache
// so a decode layer is 4 weight-streaming launches plus these small ones, and no kernel ever waits
// for another workgroup.
#include <climits>

#include "q40_warm.hpp"
#include "rope_kv.hpp"
#include "slab_sum.hpp"

namespace smh {

// ---- plain reduce (+ residual) ------------------------------------------------------------------
// RES: a residual of this alignment (elements a load; 0: none)
template <int KS, int RES>
__global__ __launch_bounds__(256) void partial_reduce_kernel(const void *__restrict__ partial, int ks, int M, int m0, int n_total, int col0, int N,
                                                             half_t *__restrict__ c, long ldc, const half_t *__restrict__ resid, long ldr) {
    // grid (quads of a row, rows): no division to find the row (a 64-bit one, 150 instructions, was most of the launch)
    args_ahead<96>();
    const int m = m0 + (int)blockIdx.y, n = (int)(blockIdx.x * blockDim.x + threadIdx.x) * 4;
    if (n >= N) return;
    f4 v[KS];
    slab_load(partial, (long)m * n_total + col0 + n, (long)M * n_total, ks, v);
    h4 r;
    if constexpr (RES == 4) r = *reinterpret_cast<const h4 *>(resid + (long)m * ldr + n);
    if constexpr (RES == 1) {
#pragma unroll
        for (int j = 0; j < 4; ++j) r[j] = resid[(long)m * ldr + n + j];
    }
    const f4 acc = slab_add(v, ks);
    h4 out;
#pragma unroll
    for (int j = 0; j < 4; ++j) out[j] = RES == 0 ? (half_t)acc[j] : (half_t)((float)r[j] + (float)(half_t)acc[j]);
    *reinterpret_cast<h4 *>(c + (long)m * ldc + n) = out;
}

// ---- residual add + RMSNorm ---------------------------------------------------------------------
// one workgroup of 1024 threads per row; h_out = h_in + fp16(acc) (fp16 add), xn = fp16(fp16(h*r)*w)
// A chain of trips to memory bounds it, so everything is requested before the first sum: KS slabs (0: none), PASSES passes of four
// columns a thread, the residual and the norm's weights.  Up to 64 registers two workgroups share a compute unit.
// Grid (rows, 1); Ask = WarmWeights: (rows, 1 and as many times more as make next.workgroups, which ask for the next launch's weights: q40_warm.hpp).
// (A kernel of its own, as the others have fewer arguments and a shorter way to their first load: one more, be it empty, makes 68 bytes of them
// in the place of one line, and 100 rows of 4096 behind four slabs 3.34 us and not 3.27)
template <int PASSES, int KS, class... Ask>
__global__ __launch_bounds__(1024, PASSES * KS <= 8 ? 8 : 4) void partial_rmsnorm_kernel(const void *__restrict__ partial, int ks, int M, int N,
                                                               const half_t *__restrict__ h_in, const half_t *__restrict__ wt,
                                                               float eps, half_t *__restrict__ h_out, half_t *__restrict__ xn_out,
                                                               Ask... next) {
    __shared__ float s_part[16];
    const int m = blockIdx.x;
    if constexpr (sizeof...(Ask) > 0) {
        if (__builtin_expect(blockIdx.y > 0, 0)) {                 // (known without an argument: a row's workgroup asks for all of them at once)
            const int e = ((int)blockIdx.y - 1) * M + m;
            return warm_weights(next..., (M + e) & 7, e >> 3, threadIdx.x, 1024);
        }
    }
    const long slab = (long)M * N;
    float ss = 0.f;
    // each thread owns columns 4t, 4t+1, 4t+2, 4t+3 (+ 4096 per pass); values kept for the second pass
    constexpr int AHEAD = PASSES * KS <= 16 ? PASSES : 1;      // passes whose slabs are on their way together
    h4 hv[PASSES], wv[PASSES];
    f4 v[AHEAD][KS > 0 ? KS : 1];
    const half_t *from = h_in != nullptr ? h_in + (long)m * N : wt;          // (without a residual: read, not used)
#pragma unroll
    for (int ps = 0; ps < PASSES; ++ps) {
        const int n = (ps * 1024 + threadIdx.x) * 4;
        if (n < N) {
            if constexpr (KS > 0 && AHEAD == PASSES) slab_load(partial, (long)m * N + n, slab, ks, v[ps % AHEAD]);
            hv[ps] = *reinterpret_cast<const h4 *>(from + n);
            wv[ps] = *reinterpret_cast<const h4 *>(wt + n);
        }
    }
#pragma unroll
    for (int ps = 0; ps < PASSES; ++ps) {
        const int n = (ps * 1024 + threadIdx.x) * 4;
        if (n < N) {
            h4 &h = hv[ps];
            if constexpr (KS > 0) {
                if constexpr (AHEAD < PASSES) slab_load(partial, (long)m * N + n, slab, ks, v[0]);
                const f4 acc = slab_add(v[ps % AHEAD], ks);
#pragma unroll
                for (int j = 0; j < 4; ++j) h[j] = h_in != nullptr ? (half_t)((float)h[j] + (float)(half_t)acc[j]) : (half_t)acc[j];
            }
            if (h_out != nullptr) *reinterpret_cast<h4 *>(h_out + (long)m * N + n) = h;
#pragma unroll
            for (int j = 0; j < 4; ++j) ss = sumsq_add(ss, (float)h[j]);
        }
    }
    ss = wave_sum(ss);
    if ((threadIdx.x & 63) == 0) s_part[threadIdx.x >> 6] = ss;
    __syncthreads();
    float total = 0.f;
#pragma unroll
    for (int w = 0; w < 16; ++w) total += s_part[w];
    const float r = rms_factor(total, N, eps);
#pragma unroll
    for (int ps = 0; ps < PASSES; ++ps) {
        const int n = (ps * 1024 + threadIdx.x) * 4;
        if (n < N) {
            const h4 w = wv[ps];
            h4 o;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                half_t nv = scale_to_half(hv[ps][j], r);
                o[j] = nv * w[j];
            }
            *reinterpret_cast<h4 *>(xn_out + (long)m * N + n) = o;
        }
    }
}

// RMSNorm of rows that are already fp16: one workgroup of 256 threads a row, eight elements a load, the row kept in registers
// (CH loads a thread).  2047 rows of 4096: 7.2 us; 1024 threads of four elements 16.5.
template <int CH>
__global__ __launch_bounds__(256) void rmsnorm_rows_kernel(const half_t *__restrict__ h, const half_t *__restrict__ wt, int N, float eps,
                                                           half_t *__restrict__ xn_out) {
    __shared__ float s_part[4];
    const half_t *row = h + (long)blockIdx.x * N;
    h8 hv[CH], wv[CH];
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < CH; ++i) {
        const int n = (i * 256 + threadIdx.x) * 8;
        if (n < N) {
            hv[i] = *reinterpret_cast<const h8 *>(row + n);
            wv[i] = *reinterpret_cast<const h8 *>(wt + n);
        }
    }
#pragma unroll
    for (int i = 0; i < CH; ++i)
        if ((i * 256 + (int)threadIdx.x) * 8 < N) {
#pragma unroll
            for (int j = 0; j < 8; ++j) ss = sumsq_add(ss, (float)hv[i][j]);
        }
    ss = wave_sum(ss);
    if ((threadIdx.x & 63) == 0) s_part[threadIdx.x >> 6] = ss;
    __syncthreads();
    const float r = rms_factor(s_part[0] + s_part[1] + s_part[2] + s_part[3], N, eps);
#pragma unroll
    for (int i = 0; i < CH; ++i) {
        const int n = (i * 256 + threadIdx.x) * 8;
        if (n < N) {
            h8 o;
#pragma unroll
            for (int j = 0; j < 8; ++j) o[j] = scale_to_half(hv[i][j], r) * wv[i][j];
            *reinterpret_cast<h8 *>(xn_out + (long)blockIdx.x * N + n) = o;
        }
    }
}

// ---- residual add + sums of squares (the first half of partial_rmsnorm_kernel, spread over 16 workgroups a row) ----
// grid (16, M), one wave each: wave w of a row is wave w of partial_rmsnorm_kernel's workgroup (same columns per
// thread, same order of additions), so sums[m][0..15] added in index order give that kernel's sum of squares bit
// for bit.  The consumer (the matmul that follows, q40_gemv_kernel LAYOUT 3, 4 and 5) normalises what it multiplies.
template <int PASSES, int KS>
__global__ __launch_bounds__(64) void partial_residual_sumsq_kernel(const void *__restrict__ partial, int ks, int M, int N,
                                                                    const half_t *__restrict__ h_in, half_t *__restrict__ h_out,
                                                                    float *__restrict__ sums) {
    const int m = blockIdx.y;
    const int vt = blockIdx.x * 64 + threadIdx.x;      // thread index inside partial_rmsnorm_kernel's workgroup
    const long slab = (long)M * N;
    f4 acc[PASSES][KS];
    h4 res[PASSES];
#pragma unroll
    for (int ps = 0; ps < PASSES; ++ps) {
        const int n = (ps * 1024 + vt) * 4;
        if (n < N) {
            slab_load(partial, (long)m * N + n, slab, ks, acc[ps]);
            if (h_in != nullptr) res[ps] = *reinterpret_cast<const h4 *>(h_in + (long)m * N + n);
        }
    }
    float ss = 0.f;
#pragma unroll
    for (int ps = 0; ps < PASSES; ++ps) {
        const int n = (ps * 1024 + vt) * 4;
        if (n < N) {
            const f4 sum = slab_add(acc[ps], ks);
            h4 v;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                v[j] = (half_t)sum[j];
                if (h_in != nullptr) v[j] = (half_t)((float)res[ps][j] + (float)v[j]);
            }
            *reinterpret_cast<h4 *>(h_out + (long)m * N + n) = v;
#pragma unroll
            for (int j = 0; j < 4; ++j) ss = sumsq_add(ss, (float)v[j]);
        }
    }
    ss = wave_sum(ss);
    if (threadIdx.x == 0) sums[(long)m * SMH_NORM_SUMS + blockIdx.x] = ss;
}

// ---- SwiGLU gate ------------------------------------------------------------------------------------
// slabs hold [gate | up] (2 * n_half columns)
template <int KS>
__global__ __launch_bounds__(256) void partial_silu_mul_kernel(const void *__restrict__ partial, int ks, int M, int n_half,
                                                               half_t *__restrict__ out) {
    // grid (quads of a row, rows): no division to find the row (a 64-bit one costs more than the rest of the arithmetic)
    const int m = blockIdx.y, n = (blockIdx.x * 256 + threadIdx.x) * 4;
    if (n >= n_half) return;
    const long slab = (long)M * 2 * n_half;
    f4 gv[KS], uv[KS];
    slab_load(partial, (long)m * 2 * n_half + n, slab, ks, gv);
    slab_load(partial, (long)m * 2 * n_half + n_half + n, slab, ks, uv);
    const f4 ga = slab_add(gv, ks), ua = slab_add(uv, ks);
    h4 o;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const float gf = (float)(half_t)ga[j];
        const half_t sl = (half_t)(gf / (1.0f + expf(-gf)));
        o[j] = sl * (half_t)ua[j];
    }
    *reinterpret_cast<h4 *>(out + (long)m * n_half + n) = o;
}

// one wave per (branch, head); heads 0..H-1 queries, H..H+Hkv-1 keys, H+Hkv.. values.
// slab columns: [q (H*128) | k (Hkv*128) | v (Hkv*128)]
template <int KS>
__global__ __launch_bounds__(256) void partial_rope_append_kernel(const void *__restrict__ partial, int ks, int B, int H, int Hkv,
                                                                  half_t *__restrict__ q, half_t *__restrict__ k, half_t *__restrict__ v,
                                                                  const half_t *__restrict__ cos_tab, const half_t *__restrict__ sin_tab,
                                                                  const int32_t *__restrict__ pos_dev,
                                                                  uint8_t *__restrict__ cache_k, half_t *__restrict__ cache_ks,
                                                                  uint8_t *__restrict__ cache_v, half_t *__restrict__ cache_vs,
                                                                  int Smax, const int32_t *__restrict__ t_dev) {
    __shared__ float s_row[4][128];
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    // grid (groups of four heads, branches)
    const int heads = H + 2 * Hkv;
    const int hh = blockIdx.x * 4 + wave;
    const bool live = hh < heads;
    const int b = blockIdx.y;
    const int h = live ? hh : 0;
    const int n_total = heads * 128;
    // the slabs are read two adjacent columns per lane; the rotation pairs column i with i + 64, so the sums
    // change lanes through LDS
    // the slabs first: the position, and behind it the rotation factors, travel under them
    f2 parts[KS];
    slab_load(partial, (long)b * n_total + (long)h * 128 + 2 * lane, (long)B * n_total, ks, parts);
    const int t = (t_dev != nullptr) ? *t_dev : -1;
    const int pos = *pos_dev;
    const half_t cos_l = cos_tab[(long)pos * 64 + lane], sin_l = sin_tab[(long)pos * 64 + lane];
    if (live) {
        const f2 sum = slab_add(parts, ks);
        *reinterpret_cast<f2 *>(&s_row[wave][2 * lane]) = sum;
    }
    __syncthreads();
    if (!live) return;
    half_t x1 = (half_t)s_row[wave][lane];
    half_t x2 = (half_t)s_row[wave][lane + 64];
    if (h >= H + Hkv) {                                      // value head: store, append
        const int hk = h - H - Hkv;
        half_t *pv = v + ((long)b * Hkv + hk) * 128;
        pv[lane] = x1;
        pv[lane + 64] = x2;
        if (cache_v != nullptr && t >= 0 && t < Smax) {
            const long row = ((long)b * Smax + t) * Hkv + hk;
            kv_store_row2(x1, x2, cache_v + row * 64, cache_vs + row * 2, lane);
        }
        return;
    }
    rope_pair2(x1, x2, cos_l, sin_l);
    if (h < H) {
        half_t *pq = q + ((long)b * H + h) * 128;
        pq[lane] = x1;
        pq[lane + 64] = x2;
        return;
    }
    const int hk = h - H;
    half_t *pk = k + ((long)b * Hkv + hk) * 128;
    pk[lane] = x1;
    pk[lane + 64] = x2;
    if (cache_k != nullptr && t >= 0 && t < Smax) {
        const long row = ((long)b * Smax + t) * Hkv + hk;
        kv_store_row2(x1, x2, cache_k + row * 64, cache_ks + row * 2, lane);
    }
}

// A prefill's q|k|v product -> q, and k, v as rows of the prompt cache (fp16): sums, one rounding, RoPE of q and k at position
// row + pos0.  One thread owns four rotation pairs (d .. d+3, d+64 ..) of one head.
template <int KS>
__global__ __launch_bounds__(256) void partial_rope_rows_kernel(const void *__restrict__ partial, int ks, int S, int H, int Hkv,
                                                                half_t *__restrict__ q, half_t *__restrict__ k, half_t *__restrict__ v,
                                                                const half_t *__restrict__ cos_tab, const half_t *__restrict__ sin_tab, int pos0) {
    const int heads = H + 2 * Hkv, s = blockIdx.y;
    const int item = blockIdx.x * 256 + threadIdx.x, h = item >> 4, d = 4 * (item & 15);
    if (h >= heads) return;
    const int n_total = heads * 128;
    const long at = (long)s * n_total + h * 128 + d, slab = (long)S * n_total;
    f4 lo_v[KS], hi_v[KS];
    slab_load(partial, at, slab, ks, lo_v);
    slab_load(partial, at + 64, slab, ks, hi_v);
    const f4 lo = slab_add(lo_v, ks), hi = slab_add(hi_v, ks);
    h4 x1, x2;
#pragma unroll
    for (int j = 0; j < 4; ++j) { x1[j] = (half_t)lo[j]; x2[j] = (half_t)hi[j]; }
    if (h < H + Hkv) {
        const h4 cs = *reinterpret_cast<const h4 *>(cos_tab + (long)(pos0 + s) * 64 + d), sn = *reinterpret_cast<const h4 *>(sin_tab + (long)(pos0 + s) * 64 + d);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            half_t a = x1[j], b = x2[j];
            rope_pair2(a, b, cs[j], sn[j]);
            x1[j] = a; x2[j] = b;
        }
    }
    half_t *dst = h < H ? q + ((long)s * H + h) * 128 : h < H + Hkv ? k + ((long)s * Hkv + h - H) * 128 : v + ((long)s * Hkv + h - H - Hkv) * 128;
    *reinterpret_cast<h4 *>(dst + d) = x1;
    *reinterpret_cast<h4 *>(dst + 64 + d) = x2;
}

}  // namespace smh

using namespace smh;

// kernels by the number of slabs (least_slabs)
static_assert(SMH_MAX_KSPLIT == 16, "tables");
#define BY_SLABS(k, ...) {__VA_ARGS__, k(1), k(2), k(3), k(4), k(5), k(6), k(8), k(8), k(10), k(10), k(12), k(12), k(16), k(16), k(16), k(16)}
typedef void (*reduce_kernel_t)(const void *, int, int, int, int, int, int, half_t *, long, const half_t *, long);
typedef void (*rmsnorm_kernel_t)(const void *, int, int, int, const half_t *, const half_t *, float, half_t *, half_t *);
typedef void (*rmsnorm_ask_t)(const void *, int, int, int, const half_t *, const half_t *, float, half_t *, half_t *, WarmWeights);
typedef void (*sumsq_kernel_t)(const void *, int, int, int, const half_t *, half_t *, float *);
#define K_OF(n) partial_reduce_kernel<n, RES>
template <int RES> static const reduce_kernel_t REDUCE_KERNELS[17] = BY_SLABS(K_OF, nullptr);
#undef K_OF
#define K_OF(n) partial_rmsnorm_kernel<PASSES, n>
template <int PASSES> static const rmsnorm_kernel_t RMSNORM_KERNELS[17] = BY_SLABS(K_OF, K_OF(0));
#undef K_OF
#define K_OF(n) partial_rmsnorm_kernel<1, n, WarmWeights>
static const rmsnorm_ask_t RMSNORM_ASK_KERNELS[17] = BY_SLABS(K_OF, nullptr);
#undef K_OF
#define K_OF(n) partial_residual_sumsq_kernel<PASSES, n>
template <int PASSES> static const sumsq_kernel_t SUMSQ_KERNELS[17] = BY_SLABS(K_OF, nullptr);
#undef K_OF
#define K_OF(n) partial_silu_mul_kernel<n>
static const decltype(&partial_silu_mul_kernel<1>) SILU_KERNELS[17] = BY_SLABS(K_OF, nullptr);
#undef K_OF
#define K_OF(n) partial_rope_append_kernel<n>
static const decltype(&partial_rope_append_kernel<1>) ROPE_APPEND_KERNELS[17] = BY_SLABS(K_OF, nullptr);
#undef K_OF
#define K_OF(n) partial_rope_rows_kernel<n>
static const decltype(&partial_rope_rows_kernel<1>) ROPE_ROWS_KERNELS[17] = BY_SLABS(K_OF, nullptr);
#undef K_OF
#undef BY_SLABS

// ---- host side: plan, produce, consume ----------------------------------------------------------------
static int fill_params(MatmulParams &p, const void *a, int M, int K, long lda, int nseg, const void *const *w,
                       const void *const *s, const int *n, const char *who, bool tiled = false, bool gemm = false) {
    SMH_REQUIRE(M >= 0, "%s: M=%d", who, M);
    SMH_REQUIRE(K > 0 && K % 8 == 0, "%s: K=%d must be a positive multiple of 8", who, K);
    SMH_REQUIRE(nseg >= 1 && nseg <= SMH_MAX_SEGMENTS && n != nullptr, "%s: nseg=%d outside [1,%d]", who, nseg, SMH_MAX_SEGMENTS);
    SMH_REQUIRE(lda >= K && lda % 8 == 0, "%s: lda=%ld must be >= K and a multiple of 8 (128-bit loads)", who, lda);
    p = MatmulParams{};
    p.a = (const half_t *)a;
    p.M = M; p.K = K; p.lda = lda; p.nseg = nseg;
    for (int i = 0; i < nseg; ++i) {
        SMH_REQUIRE(n[i] > 0 && n[i] % 128 == 0, "%s: N=%d must be a positive multiple of 128", who, n[i]);
        p.seg[i].w = w ? (const uint8_t *)w[i] : nullptr;
        p.seg[i].s = s ? (const half_t *)s[i] : nullptr;
        p.seg[i].N = n[i];
    }
    p.tiled = tiled ? 1 : 0;                   // (the plan above 16 rows depends on the layout)
    if (M <= SMH_GEMV_MAX_M && !gemm) gemv_fill_plan(p); else gemm_fill_plan(p);
    return 0;
}

extern "C" int smh_q40_matmul_plan(int M, int K, int nseg, const int *n) {
    MatmulParams p;
    if (M <= 0) return 1;
    int st = fill_params(p, nullptr, M, K, (K + 7) / 8 * 8, nseg, nullptr, nullptr, n, "smh_q40_matmul_plan");
    return st < 0 ? st : p.ksplit;
}

extern "C" int smh_q40_matmul_columns(int M, int K, int N) {
    MatmulParams p, b;
    if (M <= SMH_GEMV_MAX_M) return 0;
    const int st = fill_params(p, nullptr, M, K, (K + 7) / 8 * 8, 1, nullptr, nullptr, &N, "smh_q40_matmul_columns");
    return st < 0 ? st : p.kgroups == 2 || (p.ksplit > 1 && gemm_blocks_fit(p, b)) ? 128 : 256;
}

extern "C" int smh_q40_swiglu_fits(int M, int K, int n_half) {
    return (M > 32 && smh::gemm_swiglu_fits(M, K, n_half, true)) ? 1 : 0;
}

int smh::matmul_tiled_swiglu(const void *a, int M, int K, long lda, const void *tiled_gate, const void *tiled_up, int n_half, void *out, long ldo,
                             const WarmWeights &next, smh_stream_t stream) {
    const char *who = "smh_q40_matmul_tiled_swiglu";
    SMH_REQUIRE(gemm_swiglu_fits(M, K, n_half, false),
                "%s: M=%d (17 .. 128) K=%d (a multiple of 64) n_half=%d (a multiple of 128, at most 16384); or M above 128 and K a multiple of 32", who, M, K, n_half);
    SMH_REQUIRE(a && tiled_gate && tiled_up && out, "%s: null pointer", who);
    SMH_REQUIRE(lda >= K && lda % 8 == 0 && ldo >= n_half && ldo % (M > 128 ? 4 : 2) == 0, "%s: lda=%ld (>= K, a multiple of 8) ldo=%ld (>= n_half, even; above 128 rows a multiple of 4)", who, lda, ldo);
    SMH_REQUIRE(((uintptr_t)a & 15) == 0 && ((uintptr_t)out & (M > 128 ? 7 : 3)) == 0 && ((uintptr_t)tiled_gate & 127) == 0 && ((uintptr_t)tiled_up & 127) == 0,
                "%s: misaligned pointer", who);
    MatmulParams p = MatmulParams{};
    p.a = (const half_t *)a; p.M = M; p.K = K; p.lda = lda; p.nseg = 2;
    p.seg[0].w = (const uint8_t *)tiled_gate; p.seg[0].N = n_half;
    p.seg[1].w = (const uint8_t *)tiled_up; p.seg[1].N = n_half;
    p.c = p.seg[0].c = (half_t *)out; p.ldc = p.seg[0].ldc = ldo; p.tiled = 1;
    return M > 128 ? gemm_swiglu_rows_launch(p, (hipStream_t)stream) : gemm_swiglu_launch(p, next, (hipStream_t)stream);
}
extern "C" int smh_q40_matmul_tiled_swiglu(const void *a, int M, int K, long lda, const void *tiled_gate, const void *tiled_up, int n_half,
                                           void *out, long ldo, smh_stream_t stream) {
    SMH_REQUIRE(M > SMH_GEMV_MAX_M, "smh_q40_matmul_tiled_swiglu: M=%d (17 .. 128, or above 128)", M);
    return matmul_tiled_swiglu(a, M, K, lda, tiled_gate, tiled_up, n_half, out, ldo, WarmWeights{}, stream);
}

WarmWeights smh::q40_warm(int M, int K, int nseg, const void *const *tiled, const int *n, bool swiglu, int stages, int workgroups) {
    WarmWeights w = WarmWeights{};
    MatmulParams p;
    if (M < 1 || M > 128 || K % 64 != 0 || stages < 1) return w;
    if (swiglu ? nseg != 2 || n[0] != n[1] || !gemm_swiglu_fits(M, K, n[0], false)
               : fill_params(p, nullptr, M, K, K, nseg, nullptr, nullptr, n, "q40_warm", true, true) != 0 || p.kgroups != 2) return w;
    for (int i = 0; i < nseg; ++i)
        if (tiled[i] == nullptr || ((uintptr_t)tiled[i] & 127) != 0) return w;
    for (int i = 0; i < SMH_MAX_SEGMENTS; ++i) {
        w.w[i] = (const uint8_t *)tiled[min(i, nseg - 1)];
        w.unit0[i] = swiglu || i >= nseg ? INT_MAX : p.seg[i].unit0;
    }
    w.units = swiglu ? n[0] / 128 : p.units;
    w.units_pad = swiglu ? 0 : p.units_pad;
    w.slices = swiglu ? 1 : p.ksplit;
    w.steps = K / 32;
    w.steps_per_slice = swiglu ? w.steps : p.steps_per_slice;
    w.stages = stages;
    w.swiglu = swiglu;
    w.workgroups = min(workgroups, (warm_blocks(w) + 7) / 8 * 8);
    return w;
}

extern "C" int smh_q40_warm_span(int M, int K, int nseg, const int *n, int form, int stages, long *lines, long *first, long *end) {
    SMH_REQUIRE(nseg >= 1 && nseg <= SMH_MAX_SEGMENTS && n && lines && first && end, "smh_q40_warm_span: nseg=%d or a null pointer", nseg);
    const void *const some[SMH_MAX_SEGMENTS] = {(const void *)128, (const void *)128, (const void *)128};
    const WarmWeights w = M > SMH_GEMV_MAX_M || (form & 2) ? q40_warm(M, K, nseg, some, n, form & 1, stages, 8) : WarmWeights{};
    for (int i = 0; i < nseg; ++i) { lines[i] = first[i] = end[i] = 0; }
    for (int at = 0; w.workgroups > 0 && at < warm_blocks(w); ++at) {
        WarmBlock b;
        if (!warm_block(w, at, b)) continue;
        for (int i = 0; i < min(w.stages, b.stages) * warm_lines(w); ++i) {
            int sg;
            const long off = warm_line(w, b, i, sg);
            if (sg < 0 || sg >= nseg) { set_error("smh_q40_warm_span: weight %d of %d", sg, nseg); return -1; }
            if (lines[sg] == 0 || off < first[sg]) first[sg] = off;
            if (off + 128 > end[sg]) end[sg] = off + 128;
            ++lines[sg];
        }
    }
    return w.workgroups > 0 ? 1 : 0;
}

extern "C" int smh_q40_matmul_tiled_direct_fits(int M, int K, int nseg, const int *n) {
    MatmulParams p;
    if (M <= 128) return 0;
    const int st = fill_params(p, nullptr, M, K, (K + 7) / 8 * 8, nseg, nullptr, nullptr, n, "smh_q40_matmul_tiled_direct_fits", true);
    return st < 0 ? st : (gemm_direct_fits(p) ? 1 : 0);
}

extern "C" int smh_q40_matmul_tiled_direct_columns(int M, int K, int nseg, const int *n) {
    MatmulParams p;
    if (smh_q40_matmul_tiled_direct_fits(M, K, nseg, n) != 1) return 0;
    const int st = fill_params(p, nullptr, M, K, (K + 7) / 8 * 8, nseg, nullptr, nullptr, n, "smh_q40_matmul_tiled_direct_columns", true);
    return st < 0 ? st : gemm_direct_columns(p);
}

static int swiglu_plan(int M, int K, int n_half, int (*ask)(MatmulParams)) {
    if (M <= SMH_GEMV_MAX_M || !gemm_swiglu_fits(M, K, n_half, false)) return 0;
    MatmulParams p = MatmulParams{};
    p.M = M; p.K = K; p.nseg = 2;
    p.seg[0].N = p.seg[1].N = n_half;
    return ask(p);
}
extern "C" int smh_q40_swiglu_columns(int M, int K, int n_half) { return swiglu_plan(M, K, n_half, gemm_swiglu_columns); }
extern "C" int smh_q40_swiglu_first_columns(int M, int K, int n_half) { return swiglu_plan(M, K, n_half, gemm_swiglu_first_columns); }

static int tiled_direct(const char *who, const void *a, int M, int K, long lda, int nseg, const void *const *tiled, const int *n, void *const *out,
                        const void *residual, long ldr, int rope_heads, const void *cos_tab, const void *sin_tab, smh_stream_t stream) {
    MatmulParams p;
    const int st = fill_params(p, a, M, K, lda, nseg, tiled, nullptr, n, who, true);
    if (st) return st;
    SMH_REQUIRE(gemm_direct_fits(p), "%s: M=%d (above 128) K=%d (a multiple of 32) nseg=%d: ask smh_q40_matmul_tiled_direct_fits first", who, M, K, nseg);
    SMH_REQUIRE(a && tiled && out && ((uintptr_t)a & 15) == 0, "%s: null or misaligned pointer", who);
    for (int i = 0; i < nseg; ++i) {
        SMH_REQUIRE(tiled[i] && ((uintptr_t)tiled[i] & 127) == 0 && out[i] && ((uintptr_t)out[i] & 15) == 0, "%s: weight or output %d is null or misaligned", who, i);
        p.seg[i].c = (half_t *)out[i];
        p.seg[i].ldc = n[i];
    }
    SMH_REQUIRE(residual == nullptr || (nseg == 1 && ldr >= n[0]), "%s: a residual goes with one weight, ldr=%ld", who, ldr);
    p.direct = 1;
    p.epilogue = residual ? SMH_EPI_RESIDUAL : SMH_EPI_NONE;
    p.resid = (const half_t *)residual;
    p.ldr = ldr;
    if (rope_heads > 0) {
        p.rope_cols = 128 * rope_heads;
        p.rope_cos = (const half_t *)cos_tab;
        p.rope_sin = (const half_t *)sin_tab;
    }
    return gemm_launch(p, (hipStream_t)stream);
}
extern "C" int smh_q40_matmul_tiled_direct(const void *a, int M, int K, long lda, int nseg, const void *const *tiled, const int *n, void *const *out,
                                           const void *residual, long ldr, smh_stream_t stream) {
    return tiled_direct("smh_q40_matmul_tiled_direct", a, M, K, lda, nseg, tiled, n, out, residual, ldr, 0, nullptr, nullptr, stream);
}
extern "C" int smh_q40_matmul_tiled_direct_rope(const void *a, int M, int K, long lda, int nseg, const void *const *tiled, const int *n, void *const *out,
                                                int rope_heads, const void *cos_tab, const void *sin_tab, smh_stream_t stream) {
    const char *who = "smh_q40_matmul_tiled_direct_rope";
    long heads = 0;
    SMH_REQUIRE(nseg >= 1 && nseg <= SMH_MAX_SEGMENTS && n, "%s: nseg=%d outside [1,%d]", who, nseg, SMH_MAX_SEGMENTS);
    for (int i = 0; i < nseg; ++i) heads += n[i] / 128;
    SMH_REQUIRE(rope_heads >= 1 && rope_heads <= heads && cos_tab && sin_tab && (((uintptr_t)cos_tab | (uintptr_t)sin_tab) & 15) == 0,
                "%s: rope_heads=%d of %ld, or a null or misaligned table", who, rope_heads, heads);
    SMH_REQUIRE(M < 1 << 24, "%s: M=%d (32-bit offsets of the tables)", who, M);
    return tiled_direct(who, a, M, K, lda, nseg, tiled, n, out, nullptr, 0, rope_heads, cos_tab, sin_tab, stream);
}

extern "C" int smh_q40_matmul_plan_tiled(int M, int K, int nseg, const int *n) {
    MatmulParams p;
    if (M <= 0) return 1;
    int st = fill_params(p, nullptr, M, K, (K + 7) / 8 * 8, nseg, nullptr, nullptr, n, "smh_q40_matmul_plan_tiled", true);
    return st < 0 ? st : p.ksplit;
}

extern "C" size_t smh_q40_matmul_workspace_bytes(int max_m, int max_n) {
    // K is split only while (column units x row blocks) <= 512, so the slabs never exceed
    // 512 tiles of 128 x 256 floats for the GEMM, or SMH_MAX_KSPLIT x 16 x N floats for the GEMV
    size_t n = (size_t)(max_n < 128 ? 128 : max_n);
    size_t m = (size_t)(max_m < 1 ? 1 : (max_m > SMH_GEMV_MAX_M ? SMH_GEMV_MAX_M : max_m));
    size_t floats = n * m * SMH_MAX_KSPLIT;
    if (max_m > SMH_GEMV_MAX_M && floats < (size_t)512 * 128 * 256) floats = (size_t)512 * 128 * 256;
    return floats * sizeof(float) + 256;
}

extern "C" int smh_q40_matmul_partial(const void *a, int M, int K, long lda, int nseg, const void *const *w,
                                      const void *const *s, const int *n, void *partial, size_t partial_bytes,
                                      smh_stream_t stream) {
    MatmulParams p;
    int st = fill_params(p, a, M, K, lda, nseg, w, s, n, "smh_q40_matmul_partial");
    if (st) return st;
    if (M == 0) return 0;
    SMH_REQUIRE(a && w && s && partial, "smh_q40_matmul_partial: null pointer");
    for (int i = 0; i < nseg; ++i) SMH_REQUIRE(w[i] && s[i], "smh_q40_matmul_partial: null weight %d", i);
    size_t need = (size_t)p.ksplit * M * p.n_total * sizeof(float);
    SMH_REQUIRE(partial_bytes >= need, "smh_q40_matmul_partial: partial buffer %zu < %zu bytes", partial_bytes, need);
    p.partial = (float *)partial;
    p.direct = 0;
    return M <= SMH_GEMV_MAX_M ? gemv_launch(p, (hipStream_t)stream) : gemm_launch(p, (hipStream_t)stream);
}

int smh::blocks_plan(int M, int K, int nseg, const int *n) {
    MatmulParams p;
    return fill_params(p, nullptr, M, K, (K + 7) / 8 * 8, nseg, nullptr, nullptr, n, "blocks_plan", true, true) == 0 && p.kgroups == 2 ? p.ksplit : 0;
}
extern "C" int smh_q40_matmul_partial_tiled(const void *a, int M, int K, long lda, int nseg, const void *const *tiled,
                                            const int *n, void *partial, size_t partial_bytes, smh_stream_t stream) {
    return matmul_partial_tiled(a, M, K, lda, nseg, tiled, n, partial, partial_bytes, false, stream);
}
int smh::matmul_partial_tiled(const void *a, int M, int K, long lda, int nseg, const void *const *tiled, const int *n, void *partial, size_t partial_bytes,
                              bool blocks, smh_stream_t stream) {
    MatmulParams p;
    int st = fill_params(p, a, M, K, lda, nseg, tiled, nullptr, n, "smh_q40_matmul_partial_tiled", true, blocks);
    if (st) return st;
    if (M == 0) return 0;
    SMH_REQUIRE(a && tiled && partial, "smh_q40_matmul_partial_tiled: null pointer");
    for (int i = 0; i < nseg; ++i)
        SMH_REQUIRE(tiled[i] && ((uintptr_t)tiled[i] & 127) == 0, "smh_q40_matmul_partial_tiled: weight %d is null or not 128-byte aligned", i);
    size_t need = (size_t)p.ksplit * M * p.n_total * sizeof(float);
    SMH_REQUIRE(partial_bytes >= need, "smh_q40_matmul_partial_tiled: partial buffer %zu < %zu bytes", partial_bytes, need);
    p.partial = (float *)partial;
    p.direct = 0;
    p.tiled = 1;
    return M <= SMH_GEMV_MAX_M && !blocks ? gemv_launch(p, (hipStream_t)stream) : gemm_launch(p, (hipStream_t)stream);
}

extern "C" int smh_q40_matmul_partial_tiled_silu(const void *gate_up_partial, int gate_up_ksplit, int M, int K, int nseg,
                                                 const void *const *tiled, const int *n, void *partial, size_t partial_bytes,
                                                 smh_stream_t stream) {
    MatmulParams p;
    int st = fill_params(p, nullptr, M, K, (K + 7) / 8 * 8, nseg, tiled, nullptr, n, "smh_q40_matmul_partial_tiled_silu", true);
    if (st) return st;
    if (M == 0) return 0;
    SMH_REQUIRE(M <= SMH_SILU_IN_MAX_M, "smh_q40_matmul_partial_tiled_silu: M=%d (at most %d rows; use smh_partial_silu_mul above)", M, SMH_SILU_IN_MAX_M);
    SMH_REQUIRE(K % 32 == 0, "smh_q40_matmul_partial_tiled_silu: K=%d must be a multiple of 32", K);
    SMH_REQUIRE(gate_up_partial && tiled && partial, "smh_q40_matmul_partial_tiled_silu: null pointer");
    SMH_REQUIRE(gate_up_ksplit >= 1 && gate_up_ksplit <= SMH_MAX_KSPLIT, "smh_q40_matmul_partial_tiled_silu: ksplit=%d", gate_up_ksplit);
    for (int i = 0; i < nseg; ++i)
        SMH_REQUIRE(tiled[i] && ((uintptr_t)tiled[i] & 127) == 0, "smh_q40_matmul_partial_tiled_silu: weight %d is null or not 128-byte aligned", i);
    size_t need = (size_t)p.ksplit * M * p.n_total * sizeof(float);
    SMH_REQUIRE(partial_bytes >= need, "smh_q40_matmul_partial_tiled_silu: partial buffer %zu < %zu bytes", partial_bytes, need);
    SMH_REQUIRE(partial != gate_up_partial, "smh_q40_matmul_partial_tiled_silu: the product cannot overwrite the slabs it is made from");
    p.partial = (float *)partial;
    p.direct = 0;
    p.tiled = 1;
    p.gu_partial = (const float *)gate_up_partial;
    p.gu_ksplit = gate_up_ksplit;
    return gemv_launch(p, (hipStream_t)stream);
}

extern "C" int smh_q40_norm_in_fits(int M, int K, int nseg, const int *n) {
    MatmulParams p;
    if (M <= 0 || M > SMH_GEMV_MAX_M || K % 32 != 0) return 0;
    int st = fill_params(p, nullptr, M, K, (K + 7) / 8 * 8, nseg, nullptr, nullptr, n, "smh_q40_norm_in_fits", true);
    return st < 0 ? st : (gemv_norm_in_fits(p) ? 1 : 0);
}

extern "C" int smh_decode_norm_in_fits(int M, int K, int nseg, const int *n) {
    MatmulParams p;
    if (M <= 0 || M > SMH_GEMV_MAX_M || K % 32 != 0) return 0;
    int st = fill_params(p, nullptr, M, K, K, nseg, nullptr, nullptr, n, "smh_decode_norm_in_fits", true);
    return st < 0 ? st : (gemv_norm_in_fits(p) || gemv_norm_step_fits(p) ? 1 : 0);
}

namespace smh {
int matmul_partial_tiled_norm(const void *h, long ldh, const void *sums, const void *norm_weight, float eps, int M, int K, int nseg, const void *const *tiled,
                              const int *n, void *partial, size_t partial_bytes, bool steps, smh_stream_t stream) {
    const char *who = "smh_q40_matmul_partial_tiled_norm";
    MatmulParams p;
    int st = fill_params(p, h, M, K, ldh, nseg, tiled, nullptr, n, who, true);
    if (st) return st;
    if (M == 0) return 0;
    SMH_REQUIRE(M <= SMH_GEMV_MAX_M, "%s: M=%d (at most %d rows; use smh_partial_rmsnorm above)", who, M, SMH_GEMV_MAX_M);
    SMH_REQUIRE(K % 32 == 0 && ldh % 8 == 0, "%s: K=%d must be a multiple of 32, ldh=%ld of 8", who, K, ldh);
    SMH_REQUIRE(h && sums && norm_weight && tiled && partial, "%s: null pointer", who);
    SMH_REQUIRE(((uintptr_t)h & 15) == 0 && ((uintptr_t)norm_weight & 15) == 0 && ((uintptr_t)sums & 15) == 0, "%s: h, norm_weight and sums must be 16-byte aligned", who);
    for (int i = 0; i < nseg; ++i)
        SMH_REQUIRE(tiled[i] && ((uintptr_t)tiled[i] & 127) == 0, "%s: weight %d is null or not 128-byte aligned", who, i);
    SMH_REQUIRE(gemv_norm_in_fits(p) || (steps && gemv_norm_step_fits(p)), "%s: %d rows x K-slices of %d rows exceed %d bytes (ask smh_q40_norm_in_fits first)", who, M,
                p.steps_per_slice * 32, SMH_NORM_IN_MAX_XS_BYTES);
    size_t need = (size_t)p.ksplit * M * p.n_total * sizeof(float);
    SMH_REQUIRE(partial_bytes >= need, "%s: partial buffer %zu < %zu bytes", who, partial_bytes, need);
    p.partial = (float *)partial;
    p.direct = 0;
    p.tiled = 1;
    p.norm_w = (const half_t *)norm_weight;
    p.norm_ss = (const float *)sums;
    p.norm_eps = eps;
    return gemv_launch(p, (hipStream_t)stream);
}
}  // namespace smh

extern "C" int smh_q40_matmul_partial_tiled_norm(const void *h, long ldh, const void *sums, const void *norm_weight, float eps,
                                                 int M, int K, int nseg, const void *const *tiled, const int *n,
                                                 void *partial, size_t partial_bytes, smh_stream_t stream) {
    return matmul_partial_tiled_norm(h, ldh, sums, norm_weight, eps, M, K, nseg, tiled, n, partial, partial_bytes, false, stream);
}

static int reduce_launch(const void *partial, int ksplit, int M, int n_total, int col0, int N, void *c, long ldc,
                         int epilogue, const void *residual, long ldr, hipStream_t stream) {
    const int quads = N / 4, threads = min(256, (quads + 63) / 64 * 64);       // of a row
    const bool aligned = ldr % 4 == 0 && (uintptr_t)residual % 8 == 0;
    const auto kern = (epilogue != SMH_EPI_RESIDUAL ? REDUCE_KERNELS<0> : aligned ? REDUCE_KERNELS<4> : REDUCE_KERNELS<1>)[ksplit];
    for (int m0 = 0; m0 < M; m0 += 65535)                    // (a grid has at most 65535 rows)
        hipLaunchKernelGGL(kern, dim3((unsigned)((quads + threads - 1) / threads), (unsigned)min(M - m0, 65535)), dim3(threads), 0, stream, partial, ksplit, M, m0,
                           n_total, col0, N, (half_t *)c, ldc, (const half_t *)residual, ldr);
    return launch_status();
}

extern "C" int smh_partial_reduce(const void *partial, int ksplit, int M, int n_total, int col0, int N, void *c, long ldc,
                                  int epilogue, const void *residual, long ldr, smh_stream_t stream) {
    SMH_REQUIRE(ksplit >= 1 && ksplit <= SMH_MAX_KSPLIT, "smh_partial_reduce: ksplit=%d outside [1,%d]", ksplit, SMH_MAX_KSPLIT);
    SMH_REQUIRE(M >= 0 && N > 0 && N % 4 == 0 && col0 >= 0 && col0 % 4 == 0 && col0 + N <= n_total && n_total % 4 == 0,
                "smh_partial_reduce: M=%d N=%d col0=%d n_total=%d", M, N, col0, n_total);
    SMH_REQUIRE(epilogue == SMH_EPI_NONE || epilogue == SMH_EPI_RESIDUAL, "smh_partial_reduce: epilogue=%d", epilogue);
    if (M == 0) return 0;
    SMH_REQUIRE(partial && c && ldc >= N && ldc % 4 == 0, "smh_partial_reduce: bad output");
    SMH_REQUIRE(epilogue != SMH_EPI_RESIDUAL || (residual && ldr >= N), "smh_partial_reduce: residual missing");
    return reduce_launch(partial, ksplit, M, n_total, col0, N, c, ldc, epilogue, residual, ldr, (hipStream_t)stream);
}

static int matmul_fp16(const void *a, int M, int K, long lda, const void *b_w, const void *b_s, int N, void *c, long ldc,
                       int epilogue, const void *residual, long ldr, void *workspace, size_t workspace_bytes,
                       smh_stream_t stream, const char *who, int force) {
    SMH_REQUIRE(force != 1 || M <= SMH_GEMV_MAX_M, "%s: M=%d outside [0,%d]", who, M, SMH_GEMV_MAX_M);
    SMH_REQUIRE(epilogue == SMH_EPI_NONE || epilogue == SMH_EPI_RESIDUAL, "%s: epilogue=%d", who, epilogue);
    SMH_REQUIRE(ldc >= N, "%s: ldc=%ld too small", who, ldc);
    MatmulParams p;
    const void *ws[1] = {b_w};
    const void *ss[1] = {b_s};
    int st = fill_params(p, a, M, K, lda, 1, ws, ss, &N, who);
    if (st) return st;
    if (M == 0) return 0;
    SMH_REQUIRE(a && b_w && b_s && c, "%s: null pointer", who);
    SMH_REQUIRE(epilogue != SMH_EPI_RESIDUAL || (residual && ldr >= N), "%s: residual missing", who);
    if (force == 2 && M <= SMH_GEMV_MAX_M) gemm_fill_plan(p);        // smh_q40_gemm on a small batch
    const bool gemm = (force == 2) || M > SMH_GEMV_MAX_M;
    p.c = p.seg[0].c = (half_t *)c; p.ldc = p.seg[0].ldc = ldc; p.resid = (const half_t *)residual; p.ldr = ldr; p.epilogue = epilogue;
    if (p.ksplit == 1) {
        p.direct = 1;
        SMH_REQUIRE(!gemm || ldc % 8 == 0, "%s: ldc=%ld must be a multiple of 8 for M > 16", who, ldc);
        return gemm ? gemm_launch(p, (hipStream_t)stream) : gemv_launch(p, (hipStream_t)stream);
    }
    size_t need = (size_t)p.ksplit * M * N * sizeof(float);          // (what smh_q40_matmul_plan says; fewer slabs where gemm_blocks_fit has a form)
    SMH_REQUIRE(workspace && workspace_bytes >= need, "%s: workspace %zu < %zu bytes", who, workspace_bytes, need);
    p.partial = (float *)workspace;
    p.direct = 0;
    MatmulParams b;
    if (gemm && gemm_blocks_fit(p, b)) {
        p = b;
        // (a result written over its own activations needs the second launch that p's slabs would have given it)
        const char *a0 = (const char *)a, *c0 = (const char *)c;
        const bool apart = c0 + ((long)(M - 1) * ldc + N) * sizeof(half_t) <= a0 || a0 + ((long)(M - 1) * lda + K) * sizeof(half_t) <= c0;
        p.direct = p.ksplit == 1 && ldc % 4 == 0 && apart ? 1 : 0;
        if (p.direct) return gemm_launch(p, (hipStream_t)stream);
    }
    st = gemm ? gemm_launch(p, (hipStream_t)stream) : gemv_launch(p, (hipStream_t)stream);
    if (st) return st;
    SMH_REQUIRE(ldc % 4 == 0, "%s: ldc=%ld must be a multiple of 4", who, ldc);
    return reduce_launch(p.partial, p.ksplit, M, N, 0, N, c, ldc, epilogue, residual, ldr, (hipStream_t)stream);
}

extern "C" int smh_q40_gemv(const void *a, int M, int K, long lda, const void *b_w, const void *b_s, int N, void *c, long ldc,
                            int epilogue, const void *residual, long ldr, void *workspace, size_t workspace_bytes, smh_stream_t stream) {
    return matmul_fp16(a, M, K, lda, b_w, b_s, N, c, ldc, epilogue, residual, ldr, workspace, workspace_bytes, stream, "smh_q40_gemv", 1);
}
extern "C" int smh_q40_gemm(const void *a, int M, int K, long lda, const void *b_w, const void *b_s, int N, void *c, long ldc,
                            int epilogue, const void *residual, long ldr, void *workspace, size_t workspace_bytes, smh_stream_t stream) {
    return matmul_fp16(a, M, K, lda, b_w, b_s, N, c, ldc, epilogue, residual, ldr, workspace, workspace_bytes, stream, "smh_q40_gemm", 2);
}
extern "C" int smh_q40_matmul(const void *a, int M, int K, long lda, const void *b_w, const void *b_s, int N, void *c, long ldc,
                              int epilogue, const void *residual, long ldr, void *workspace, size_t workspace_bytes, smh_stream_t stream) {
    return matmul_fp16(a, M, K, lda, b_w, b_s, N, c, ldc, epilogue, residual, ldr, workspace, workspace_bytes, stream, "smh_q40_matmul", 0);
}

int smh::partial_rmsnorm(const void *partial, int ksplit, int M, int N, const void *h_in, const void *weight, float eps, void *h_out, void *xn_out,
                         const WarmWeights &next, smh_stream_t stream) {
    SMH_REQUIRE(partial == nullptr || (ksplit >= 1 && ksplit <= SMH_MAX_KSPLIT), "smh_partial_rmsnorm: ksplit=%d", ksplit);
    SMH_REQUIRE(M >= 0 && N > 0 && N % 4 == 0 && N <= 16384, "smh_partial_rmsnorm: M=%d N=%d (N must be a multiple of 4, <= 16384)", M, N);
    SMH_REQUIRE(partial != nullptr || h_in != nullptr, "smh_partial_rmsnorm: no input");
    if (M == 0) return 0;
    SMH_REQUIRE(weight && xn_out, "smh_partial_rmsnorm: null pointer");
    if (partial == nullptr && h_out == nullptr && N % 8 == 0 && (((uintptr_t)h_in | (uintptr_t)weight | (uintptr_t)xn_out) & 15) == 0) {
        const auto kern = N <= 4096 ? rmsnorm_rows_kernel<2> : N <= 8192 ? rmsnorm_rows_kernel<4> : rmsnorm_rows_kernel<8>;
        hipLaunchKernelGGL(kern, dim3(M), dim3(256), 0, (hipStream_t)stream, (const half_t *)h_in, (const half_t *)weight, N, eps, (half_t *)xn_out);
        return launch_status();
    }
    const int ks = partial == nullptr ? 0 : ksplit;
    const auto kern = N <= 4096 ? RMSNORM_KERNELS<1>[ks] : N <= 8192 ? RMSNORM_KERNELS<2>[ks] : RMSNORM_KERNELS<4>[ks];
    if (next.workgroups > 0 && ks > 0 && N <= 4096) {
        hipLaunchKernelGGL(RMSNORM_ASK_KERNELS[ks], dim3(M, 1 + (next.workgroups + M - 1) / M), dim3(1024), 0, (hipStream_t)stream, partial, ks, M, N, (const half_t *)h_in,
                           (const half_t *)weight, eps, (half_t *)h_out, (half_t *)xn_out, next);
        return launch_status();
    }
    hipLaunchKernelGGL(kern, dim3(M), dim3(1024), 0, (hipStream_t)stream, partial, ks, M, N, (const half_t *)h_in, (const half_t *)weight, eps, (half_t *)h_out,
                       (half_t *)xn_out);
    return launch_status();
}
extern "C" int smh_partial_rmsnorm(const void *partial, int ksplit, int M, int N, const void *h_in, const void *weight, float eps,
                                   void *h_out, void *xn_out, smh_stream_t stream) {
    return partial_rmsnorm(partial, ksplit, M, N, h_in, weight, eps, h_out, xn_out, WarmWeights{}, stream);
}

extern "C" int smh_partial_residual_sumsq(const void *partial, int ksplit, int M, int N, const void *h_in, void *h_out, void *sums,
                                          smh_stream_t stream) {
    SMH_REQUIRE(partial != nullptr && ksplit >= 1 && ksplit <= SMH_MAX_KSPLIT, "smh_partial_residual_sumsq: partial=%p ksplit=%d", partial, ksplit);
    SMH_REQUIRE(M >= 0 && N > 0 && N % 4 == 0 && N <= 16384, "smh_partial_residual_sumsq: M=%d N=%d (N must be a multiple of 4, <= 16384)", M, N);
    if (M == 0) return 0;
    SMH_REQUIRE(h_out && sums, "smh_partial_residual_sumsq: null pointer");
    const auto kern = N <= 4096 ? SUMSQ_KERNELS<1>[ksplit] : N <= 8192 ? SUMSQ_KERNELS<2>[ksplit] : SUMSQ_KERNELS<4>[ksplit];
    hipLaunchKernelGGL(kern, dim3(SMH_NORM_SUMS, M), dim3(64), 0, (hipStream_t)stream, partial, ksplit, M, N, (const half_t *)h_in, (half_t *)h_out, (float *)sums);
    return launch_status();
}

extern "C" int smh_partial_silu_mul(const void *partial, int ksplit, int M, int n_half, void *out, smh_stream_t stream) {
    SMH_REQUIRE(ksplit >= 1 && ksplit <= SMH_MAX_KSPLIT, "smh_partial_silu_mul: ksplit=%d", ksplit);
    SMH_REQUIRE(M >= 0 && n_half > 0 && n_half % 4 == 0, "smh_partial_silu_mul: M=%d n_half=%d", M, n_half);
    if (M == 0) return 0;
    SMH_REQUIRE(partial && out, "smh_partial_silu_mul: null pointer");
    SMH_REQUIRE(M <= 65535, "smh_partial_silu_mul: M=%d (at most 65535 rows per launch)", M);
    hipLaunchKernelGGL(SILU_KERNELS[ksplit], dim3((unsigned)((n_half / 4 + 255) / 256), (unsigned)M), dim3(256), 0, (hipStream_t)stream,
                       partial, ksplit, M, n_half, (half_t *)out);
    return launch_status();
}

extern "C" int smh_partial_rope_append_kv(const void *partial, int ksplit, int B, int H, int Hkv, int D, void *q, void *k, void *v,
                                          const void *cos_tab, const void *sin_tab, const int32_t *pos_dev,
                                          void *cache_k, void *cache_ks, void *cache_v, void *cache_vs, int Smax,
                                          const int32_t *t_dev, smh_stream_t stream) {
    SMH_REQUIRE(D == 128, "smh_partial_rope_append_kv: head dim %d (only 128)", D);
    SMH_REQUIRE(ksplit >= 1 && ksplit <= SMH_MAX_KSPLIT, "smh_partial_rope_append_kv: ksplit=%d", ksplit);
    SMH_REQUIRE(B >= 0 && H > 0 && Hkv > 0, "smh_partial_rope_append_kv: B=%d H=%d Hkv=%d", B, H, Hkv);
    if (B == 0) return 0;
    SMH_REQUIRE(partial && q && k && v && cos_tab && sin_tab && pos_dev, "smh_partial_rope_append_kv: null pointer");
    SMH_REQUIRE(!cache_k || (cache_ks && cache_v && cache_vs && t_dev && Smax > 0), "smh_partial_rope_append_kv: cache arguments incomplete");
    SMH_REQUIRE(B <= 65535, "smh_partial_rope_append_kv: B=%d (at most 65535 branches per launch)", B);
    hipLaunchKernelGGL(ROPE_APPEND_KERNELS[ksplit], dim3((unsigned)((H + 2 * Hkv + 3) / 4), (unsigned)B), dim3(256), 0, (hipStream_t)stream,
                       partial, ksplit, B, H, Hkv, (half_t *)q, (half_t *)k, (half_t *)v,
                       (const half_t *)cos_tab, (const half_t *)sin_tab, pos_dev, (uint8_t *)cache_k, (half_t *)cache_ks,
                       (uint8_t *)cache_v, (half_t *)cache_vs, Smax, t_dev);
    return launch_status();
}

extern "C" int smh_partial_rope_rows(const void *partial, int ksplit, int S, int H, int Hkv, int D, void *q, void *k, void *v, const void *cos_tab,
                                     const void *sin_tab, int pos0, smh_stream_t stream) {
    SMH_REQUIRE(D == 128, "smh_partial_rope_rows: head dim %d (only 128)", D);
    SMH_REQUIRE(ksplit >= 1 && ksplit <= SMH_MAX_KSPLIT, "smh_partial_rope_rows: ksplit=%d", ksplit);
    SMH_REQUIRE(S >= 0 && S <= 65535 && H > 0 && Hkv > 0 && pos0 >= 0, "smh_partial_rope_rows: S=%d (at most 65535) H=%d Hkv=%d pos0=%d", S, H, Hkv, pos0);
    if (S == 0) return 0;
    SMH_REQUIRE(partial && q && k && v && cos_tab && sin_tab, "smh_partial_rope_rows: null pointer");
    hipLaunchKernelGGL(ROPE_ROWS_KERNELS[ksplit], dim3((unsigned)(((H + 2 * Hkv) * 16 + 255) / 256), (unsigned)S), dim3(256), 0, (hipStream_t)stream, partial, ksplit,
                       S, H, Hkv, (half_t *)q, (half_t *)k, (half_t *)v, (const half_t *)cos_tab, (const half_t *)sin_tab, pos0);
    return launch_status();
}
