// Shared-prefix decode attention: one query per (branch, head) over
//   [ prefix K/V (P rows, fp16, shared by all branches) || that branch's suffix (fp16 or Q4_0 rows)
//     || the new token's exact fp16 K/V ].
//
// Two kernels.
//  1. attn_prefix_kernel, grid (splits, kv heads, query groups): a workgroup stages one slice of the
//     prefix for one kv head in LDS ONCE (K row-major, V transposed) and the branches' queries for
//     that head are multiplied against it on the matrix cores: the queries are the N dimension of
//     S^T = K . Q^T and of O^T = V^T . P^T, so the prefix is read from HBM once per head instead of
//     once per branch (with many queries a slice's query tiles are dealt to a few workgroups, which
//     re-read it from the cache).  Each (slice, query) leaves an un-normalised partial (max, sum, o[128]).
//  2. attn_suffix_kernel, one wave per (branch, query head): streams the branch's own suffix rows
//     (HBM-bound; Q4_0 rows are decoded in registers), keeps an online softmax per 16-lane group,
//     folds in the prefix partials and the new token, normalises and writes fp16.
// With fp16 suffixes the slices and the walks are one launch and a merge follows (attn_parts_kernel); fp16 pages that neighbouring
// branches share go through attn_page_tile_kernel before the walk.
// Scores and softmax are fp32 throughout (exp2 of log2(e)-scaled scores); probabilities are rounded to fp16 only as the operand of
// the P.V matrix product of a shared prefix and of a prefill (walks and shared pages hold all their bits, attn_tile_kernel's prefix 22).
//
// Algorithmic HBM traffic: prefix 2*P*Hkv*D*2 B once + per branch its suffix rows
// (512 B fp16 or 136 B Q4_0 per row and kv head) + q/out.
#include <mutex>
#include <type_traits>

#include "attn_rows.hpp"
#include "attn_tiles.hpp"
#include "q40_warm.hpp"
#include "rope_kv.hpp"

namespace smh {

constexpr int ATT_D = 128;
constexpr int ATT_TW_MAX = 128;            // prefix rows per workgroup
constexpr int ATT_KPITCH = 136;            // halves per LDS row of K (272 B: 16 rows hit distinct banks)
constexpr float LOG2E = 1.4426950408889634f;
constexpr int ATT_ONE_TW = 64;             // prefix rows per workgroup of the one-launch kernel: two workgroups fit a compute unit
constexpr int ATT_FUSED_MAX_Q = 128;       // queries per kv head (branches x query heads per kv head) of the fused variant

struct AttnParams {
    const half_t *q;
    half_t *out;
    const half_t *prefix_k, *prefix_v;
    const void *suffix_k, *suffix_v;
    const half_t *suffix_ks, *suffix_vs;
    const int32_t *lens;
    const half_t *cur_k, *cur_v;
    float *part_o;           // [splits][Hkv][Bq][128]
    float *part_ml;          // [splits][Hkv][Bq][2]
    long suffix_batch_stride_rows;   // rows (tokens) between consecutive branches of the suffix
    // paged suffix: row j of branch b is pool row pages[b * pages_stride + j] instead of b * suffix_batch_stride_rows + j
    // (page ids of page_bytes = 2, 4 or 8 bytes each); pages == nullptr: contiguous rows per branch
    const void *pages;
    long pages_stride;
    int page_bytes;
    long pool_rows;          // rows of the pool the page ids point into: an id outside 0 .. pool_rows-1 reads the nearest row, never past the pool
    // element strides of the fp16 K/V tensors: between consecutive rows (tokens) and between kv heads.  Token-major
    // [rows, Hkv, 128] is (Hkv * 128, 128); a head-major pool [Hkv, rows, 128] is (128, rows * 128).  Q4_0 rows are token-major.
    long pfx_row_stride, pfx_head_stride;
    long sfx_row_stride, sfx_head_stride;
    int B, H, Hkv, n_rep, Bq;        // Bq = B * n_rep queries per kv head
    int suffix_waves;                // waves that share one query's suffix rows (1, 2 or 4)
    int P, tw, splits;
    int suffix_format, lens_stride;
    float scale_log2;                // log2(e) / sqrt(D)
    // FUSED kernels: q, the new token's k and v come straight from the fp32 K-slice slabs of the wq|wk|wv product
    // ([qkv_ks][B][(H + 2 Hkv) * 128]); RoPE, the fp16 rounding points and the Q4_0 append of k, v are those of
    // partial_rope_append_kernel (q / cur_k / cur_v above are not read)
    const float *qkv;
    int qkv_ks;
    const half_t *cos_tab, *sin_tab;
    const int32_t *pos_dev;
    uint8_t *app_k, *app_v;          // the branches' suffix caches (row *app_t of every branch is written); may be null
    half_t *app_ks, *app_vs;
    const int32_t *app_t;
    int app_smax;
    uint32_t *counters;              // one-launch variant: arrivals per kv head (zero between launches)
    uint8_t *tile_done;              // [Hkv][query tiles][splits]: 1 where attn_page_tile_kernel has left the partials of a slice
};

// x / n_rep and x % n_rep for the query heads per kv head; 1 (multi-head attention) needs no division
__device__ __forceinline__ int div_rep(const AttnParams &p, int x) { return p.n_rep == 1 ? x : x / p.n_rep; }
__device__ __forceinline__ int mod_rep(const AttnParams &p, int x) { return p.n_rep == 1 ? 0 : x % p.n_rep; }

// Columns `col` .. (T: float or f4) of branch b in the fused q|k|v product, requested and then added in slice order; at most QKS slabs.  No
// condition on a load (past the last slab: that one again, counted as zero): behind one the compiler waited for what it had before it
// requested the rest.
template <typename T, int QKS>
__device__ __forceinline__ void qkv_request(const AttnParams &p, int b, int col, T (&v)[QKS]) {
    const int cols = (p.H + 2 * p.Hkv) * ATT_D;
    const float *src = p.qkv + (long)b * cols + col;
    const long slab = (long)p.B * cols;
#pragma unroll
    for (int s_ = 0; s_ < QKS; ++s_) v[s_] = *reinterpret_cast<const T *>(src + min(s_, p.qkv_ks - 1) * slab);
}
template <typename T, int QKS>
__device__ __forceinline__ T qkv_sum(const AttnParams &p, const T (&v)[QKS]) {
    T tot = T{};
#pragma unroll
    for (int s_ = 0; s_ < QKS; ++s_) tot += s_ < p.qkv_ks ? v[s_] : T{};
    return tot;
}

// position of prefix row t (0..tw-1) inside an LDS row of V^T: within each block of 32 rows the
// order is chosen so that the 8 probabilities a lane holds after two S^T tiles (rows 4g+r of tile 2j
// and of tile 2j+1) are 8 consecutive halves.
// dims 4cc..4cc+3 (lo) and 64+4cc.. (hi) of the rotated query of head h, branch b: the rotation pairs d and d + 64
// sit in the same lane
template <int QKS>
__device__ __forceinline__ void qkv_query(const AttnParams &p, int b, int h, int pos, int cc, h4 &lo, h4 &hi) {
    f4 lo_v[QKS], hi_v[QKS];
    qkv_request(p, b, h * ATT_D + 4 * cc, lo_v);
    qkv_request(p, b, h * ATT_D + 64 + 4 * cc, hi_v);
    const h4 cs = *reinterpret_cast<const h4 *>(p.cos_tab + (long)pos * 64 + 4 * cc);
    const h4 sn = *reinterpret_cast<const h4 *>(p.sin_tab + (long)pos * 64 + 4 * cc);
    const f4 lo_s = qkv_sum(p, lo_v), hi_s = qkv_sum(p, hi_v);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        half_t x1 = (half_t)lo_s[j], x2 = (half_t)hi_s[j];
        rope_pair2(x1, x2, cs[j], sn[j]);
        lo[j] = x1; hi[j] = x2;
    }
}

__device__ __forceinline__ int vt_pos(int t) {
    const int blk = t & ~31, w = t & 31;
    const int j2 = w >> 4, g = (w >> 2) & 3, r = w & 3;
    return blk + 8 * g + 4 * j2 + r;
}

// COHERENT: the partials are read by another workgroup of the same launch (device-scope stores)
// TWM: most prefix rows a workgroup takes (p.tw <= TWM), which sizes its LDS
// qg, n_qg: this workgroup takes the query tiles of rounds qg, qg + n_qg, ... (a round = one tile per wave)
// QKS: most slabs of the q|k|v product (FUSED)
template <bool FUSED, bool COHERENT, int TWM, int QKS = 16>
__device__ __forceinline__ void attn_prefix_body(const AttnParams &p, int split, int hk, int qg = 0, int n_qg = 1) {
    __shared__ __attribute__((aligned(16))) half_t ks[TWM][ATT_KPITCH];
    __shared__ __attribute__((aligned(16))) half_t vt[ATT_D][TWM + 8];
    __shared__ __attribute__((aligned(16))) half_t qs[FUSED ? ATT_FUSED_MAX_Q : 1][ATT_D + 8];      // FUSED: the rotated queries of this kv head

    const int tid = threadIdx.x;
    const int wave = tid >> 6, lane = tid & 63, c = lane & 15, g = lane >> 4;
    const int t0 = split * p.tw;
    const int cnt = min(p.tw, p.P - t0);
    const int tw32 = (cnt + 31) & ~31;          // rows actually touched by the matrix ops

    // the B operand of S^T = K . Q^T for query tile qt: dims 32*k4 + 8g .. +7 of query row c
    const int q_tiles = (p.Bq + 15) / 16;
    auto load_q = [&](int qt, h8 (&qb)[4]) {
        const int qr = min(qt * 16 + c, p.Bq - 1);
        if (!FUSED) {
            const int b = div_rep(p, qr), r_ = mod_rep(p, qr);
            const half_t *qp = p.q + ((long)b * p.H + hk * p.n_rep + r_) * ATT_D + 8 * g;
#pragma unroll
            for (int k4 = 0; k4 < 4; ++k4) qb[k4] = *reinterpret_cast<const h8 *>(qp + 32 * k4);
        } else {
#pragma unroll
            for (int k4 = 0; k4 < 4; ++k4) qb[k4] = *reinterpret_cast<const h8 *>(&qs[qr][32 * k4 + 8 * g]);
        }
    };
    // un-fused: the first tile's query is requested before the prefix slice is staged
    h8 qb_first[4];
    const int qt_first = wave + 4 * qg;
    if (!FUSED && qt_first < q_tiles) load_q(qt_first, qb_first);

    // ---- stage K (row-major) and V (transposed) ----
    // A thread moves piece ch (8 dims) of FOUR consecutive rows 4 kg .. 4 kg + 3: their V values sit side by side in a
    // row of vt (vt_pos), so V goes out as 8-byte stores instead of 2-byte ones.
    const int ch = tid & 15;
    auto stage_load4 = [&](int kg, u32x4 (&kv)[4], u32x4 (&vv)[4]) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int t = 4 * kg + e;
            kv[e] = u32x4{0, 0, 0, 0}; vv[e] = u32x4{0, 0, 0, 0};
            if (t < cnt) {
                const long off = (long)(t0 + t) * p.pfx_row_stride + (long)hk * p.pfx_head_stride + ch * 8;
                kv[e] = *reinterpret_cast<const u32x4 *>(p.prefix_k + off);
                vv[e] = *reinterpret_cast<const u32x4 *>(p.prefix_v + off);
            }
        }
    };
    auto stage_store4 = [&](int kg, const u32x4 (&kv)[4], const u32x4 (&vv)[4]) {
#pragma unroll
        for (int e = 0; e < 4; ++e) *reinterpret_cast<u32x4 *>(&ks[4 * kg + e][ch * 8]) = kv[e];
        const int pos = vt_pos(4 * kg);
        const h8 v0 = __builtin_bit_cast(h8, vv[0]), v1 = __builtin_bit_cast(h8, vv[1]);
        const h8 v2 = __builtin_bit_cast(h8, vv[2]), v3 = __builtin_bit_cast(h8, vv[3]);
#pragma unroll
        for (int j = 0; j < 8; ++j) *reinterpret_cast<h4 *>(&vt[ch * 8 + j][pos]) = h4{v0[j], v1[j], v2[j], v3[j]};
    };
    auto build_queries = [&]() {
        const int cc = tid & 15;
        const int pos = *p.pos_dev;
        for (int qr = tid >> 4; qr < p.Bq; qr += 16) {
            h4 lo, hi;
            qkv_query<QKS>(p, div_rep(p, qr), hk * p.n_rep + mod_rep(p, qr), pos, cc, lo, hi);
            *reinterpret_cast<h4 *>(&qs[qr][4 * cc]) = lo;
            *reinterpret_cast<h4 *>(&qs[qr][64 + 4 * cc]) = hi;
        }
    };
    if (FUSED && TWM <= 64) {
        // every load of the workgroup is requested before anything waits: the K / V slice into registers, then
        // the slabs from which all 256 threads build the rotated queries of this kv head (8 dims each)
        static_assert(!FUSED || TWM > 64 || TWM == 64, "one group of four rows per thread");
        u32x4 kv[4], vv[4];
        const int kg = tid >> 4;
        if (4 * kg < tw32) stage_load4(kg, kv, vv);
        build_queries();
        if (4 * kg < tw32) stage_store4(kg, kv, vv);
    } else {
        if (FUSED) build_queries();
        for (int kg = tid >> 4; 4 * kg < tw32; kg += 16) {
            u32x4 kv[4], vv[4];
            stage_load4(kg, kv, vv);
            stage_store4(kg, kv, vv);
        }
    }
    __syncthreads();

    const int t_tiles = tw32 / 16;
    for (int qt = qt_first; qt < q_tiles; qt += 4 * n_qg) {
        h8 qb[4];
        if (!FUSED && qt == qt_first) {
#pragma unroll
            for (int k4 = 0; k4 < 4; ++k4) qb[k4] = qb_first[k4];
        } else {
            load_q(qt, qb);
        }
        // S^T tiles: element r of st[j] is row t = 16j + 4g + r, column (query) c
        f4 st[TWM / 16];
        float mx = -INFINITY;
#pragma unroll
        for (int j = 0; j < TWM / 16; ++j) {
            st[j] = f4{0.f, 0.f, 0.f, 0.f};
            if (j < t_tiles) {
#pragma unroll
                for (int k4 = 0; k4 < 4; ++k4) {
                    h8 ka = *reinterpret_cast<const h8 *>(&ks[16 * j + c][32 * k4 + 8 * g]);
                    st[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ka, qb[k4], st[j], 0, 0, 0);
                }
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int t = 16 * j + 4 * g + r;
                    const float sv = (t < cnt) ? st[j][r] * p.scale_log2 : -INFINITY;
                    st[j][r] = sv;
                    mx = fmaxf(mx, sv);
                }
            }
        }
        mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        float sum = 0.f;
#pragma unroll
        for (int j = 0; j < TWM / 16; ++j) {
            if (j < t_tiles) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float e = exp2f(st[j][r] - mx);      // masked rows: exp2(-inf) = 0
                    st[j][r] = e;
                    sum += e;
                }
            }
        }
        sum += __shfl_xor(sum, 16, 64);
        sum += __shfl_xor(sum, 32, 64);

        // O^T tiles: element r of ot[dt] is row d = 16dt + 4g + r, column (query) c
        f4 ot[8];
#pragma unroll
        for (int dt = 0; dt < 8; ++dt) ot[dt] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int jj = 0; jj < TWM / 32; ++jj) {
            if (2 * jj < t_tiles) {
                h8 pb;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    pb[r] = (half_t)st[2 * jj][r];
                    pb[4 + r] = (half_t)st[2 * jj + 1][r];
                }
#pragma unroll
                for (int dt = 0; dt < 8; ++dt) {
                    h8 va = *reinterpret_cast<const h8 *>(&vt[16 * dt + c][32 * jj + 8 * g]);
                    ot[dt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(va, pb, ot[dt], 0, 0, 0);
                }
            }
        }
        const int qrow = qt * 16 + c;
        if (qrow < p.Bq) {
            const long base = ((long)split * p.Hkv + hk) * p.Bq + qrow;
            float *po = p.part_o + base * ATT_D;
#pragma unroll
            for (int dt = 0; dt < 8; ++dt) {
                if (COHERENT) st_f4(po + 16 * dt + 4 * g, ot[dt]);
                else *reinterpret_cast<f4 *>(po + 16 * dt + 4 * g) = ot[dt];
            }
            if (g == 0) {
                if (COHERENT) { st_f32(p.part_ml + base * 2, partial_max(mx, sum)); st_f32(p.part_ml + base * 2 + 1, sum); }
                else { p.part_ml[base * 2] = partial_max(mx, sum); p.part_ml[base * 2 + 1] = sum; }
            }
        }
    }
}

template <bool FUSED>
__global__ __launch_bounds__(256) void attn_prefix_kernel(AttnParams p) {
    args_ahead<sizeof(AttnParams)>();
    attn_prefix_body<FUSED, false, ATT_TW_MAX>(p, blockIdx.x, blockIdx.y, blockIdx.z, gridDim.z);
}

// ---- pages that the branches of a query tile share ---------------------------------------------------------------
// Branches of a tree share their ancestors' pages, so the same page stands at the same position of many rows of the table
// (the prompt's in all of them).  Workgroup (kv head, slice of 64 positions, tile of 16 queries): where the tile's branches
// have the same ids throughout the slice, its rows are staged in LDS once for the 16 queries and multiplied on the matrix
// cores - wave w scores positions 16 w .. + 15 and then makes dims 32 w .. + 31 of the outputs - and a partial (max, sum,
// o[128]) is left per query; tile_done says so and attn_suffix_kernel skips the slice.  Where they differ, or a staged value
// is infinite or NaN, the slice is left to attn_suffix_kernel.  Probabilities enter the product as three fp16 terms of 2^15 p (the
// second 2^11 times what the first leaves over, the third 2^11 times what the second does), in three accumulators: all 24 bits of
// the fp32 probability down to 2^-38 of the slice's largest, 2^-62 of it absolutely below, so nothing of it is rounded away.
// A workgroup has PT_TILES tiles, one after the other, and stages rows again only where the ids differ from the last tile's.
// Bound by the walk of what is not shared.  32 heads, 512 positions, half of them a prompt: 99 branches 150 -> 100 us a call, 50: 80 -> 60,
// 27: 45 -> 37, 8: 32 -> 20; 460 shared positions and 99 branches: 111 -> 39 us (error against 64 bits 2.1e-4 before and after: the
// output's fp16).  Where nothing is shared the pass costs its 3 us (100 positions, 99 branches: 29.7 -> 26.5 with the walk's gain).
// Two tiles a workgroup where one a workgroup would be more than the 768 that run at a time (three a compute unit): 32 heads, 99 branches,
// 512 positions, 256 of them a prompt 83.1 -> 80.7 us a call (this pass 16.3 -> 14.3), 460 of them 33.2 -> 30.9, 768 with a prompt of 600 68.2 -> 64.6;
// 100 positions, 448 workgroups of one tile, 22.6 and 23.3 with two.  Three and four tiles: no faster, seven: slower.
// The grid runs over the tiles first and the slices last: the first slices are the likely ones, and their workgroups start together (13.8 us before, 12.8).
constexpr int PT_TW = 64;
constexpr long PT_ROUND = 768;
constexpr int PT_MAX_SLICES = 64;          // one bit a slice in the suffix kernel's mask
// Waits for a wave's loads where a loop that keeps a batch on its way begins.  With the first batch still on its way there, the compiler, which
// counts loads, waits in every pass for as much as the first one needs: for the next batch, too.
__device__ __forceinline__ void wait_loads() { __builtin_amdgcn_s_waitcnt(0x0f70); }       // vmcnt(0)

// PB: bytes of a page id, 0 without a page table; PB_ANY: what the parameters say.  Kernels that walk know it when they are compiled: a load
// behind a branch on the width was waited for with everything else on its way, rows of the next batch among them.
constexpr int PB_ANY = -1;
template <int PB> using page_id_t = std::conditional_t<PB == 2 || PB == 4 || PB == 0, int, long>;
template <int PB>
__device__ __forceinline__ page_id_t<PB> page_at(const AttnParams &p, long i) {
    if constexpr (PB == 4) return reinterpret_cast<const int32_t *>(p.pages)[i];
    if constexpr (PB == 2) return reinterpret_cast<const int16_t *>(p.pages)[i];
    if constexpr (PB == 8) return reinterpret_cast<const int64_t *>(p.pages)[i];
    if (p.page_bytes == 4) return reinterpret_cast<const int32_t *>(p.pages)[i];
    if (p.page_bytes == 2) return reinterpret_cast<const int16_t *>(p.pages)[i];
    return reinterpret_cast<const int64_t *>(p.pages)[i];
}
// the pool row of a page id (ids outside the pool are cut at its ends)
template <int PB>
__device__ __forceinline__ long page_row(const AttnParams &p, page_id_t<PB> id) {
    if constexpr (PB == 2 || PB == 4) return min(max(id, 0), (int)min(p.pool_rows - 1, 0x7fffffffL));
    return min(max((long)id, 0L), p.pool_rows - 1);
}
template <int PB, int PT_TILES>
__global__ __launch_bounds__(256) void attn_page_tile_kernel(AttnParams p) {
    args_ahead<sizeof(AttnParams)>();
    __shared__ __attribute__((aligned(16))) half_t ks[PT_TW][ATT_KPITCH];
    __shared__ __attribute__((aligned(16))) half_t vt[ATT_D][PT_TW + 8];
    __shared__ __attribute__((aligned(16))) half_t ps[3][16][PT_TW + 8];      // probabilities of the 16 queries, the three terms, in vt_pos order
    __shared__ long s_row[PT_TILES][PT_TW];        // rows of the tiles' first branches
    __shared__ float s_max[4][16], s_sum[4][16];
    __shared__ uint32_t s_bits[4];
    const int hk = blockIdx.x, split = blockIdx.z, tiles = (p.Bq + 15) / 16, tile0 = blockIdx.y * PT_TILES, n_tiles = min(PT_TILES, tiles - tile0);
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, c = lane & 15, g = lane >> 4;
    const int t0 = split * PT_TW, cnt = min(PT_TW, (int)p.suffix_batch_stride_rows - t0);
    // a tile's queries (B operand of S^T)
    auto queries = [&](int i, h8 (&qb)[4]) {
        const int qr = min((tile0 + i) * 16 + c, p.Bq - 1);
        const half_t *qp = p.q + ((long)div_rep(p, qr) * p.H + hk * p.n_rep + mod_rep(p, qr)) * ATT_D + 8 * g;
#pragma unroll
        for (int k4 = 0; k4 < 4; ++k4) qb[k4] = *reinterpret_cast<const h8 *>(qp + 32 * k4);
    };
    // ---- bit i: every branch of tile i has the first one's ids; bit 8 + i: which are those of tile i - 1's first ----
    uint32_t bits = 0;
    h8 qn[4];
    {
        const int pos = t0 + min(lane, cnt - 1);
        page_id_t<PB> id[PT_TILES][5];             // a tile's first branch's, and those of every fourth other one (past the last: again)
#pragma unroll
        for (int i = 0; i < PT_TILES; ++i) {
            const int b_lo = div_rep(p, min((tile0 + i) * 16, p.Bq - 1)), b_hi = div_rep(p, min((tile0 + i) * 16 + 15, p.Bq - 1));
#pragma unroll
            for (int j = 0; j < 5; ++j) id[i][j] = page_at<PB>(p, (long)(j == 0 ? b_lo : min(b_lo + 1 + wave + 4 * (j - 1), b_hi)) * p.pages_stride + pos);
        }
        queries(0, qn);
#pragma unroll
        for (int i = 0; i < PT_TILES; ++i) {
            bool same = true;
#pragma unroll
            for (int j = 1; j < 5; ++j) same &= id[i][j] == id[i][0];
            if (__all(same)) bits |= 1u << i;
            if (i > 0 && __all(id[i][0] == id[i - 1][0])) bits |= 256u << i;
            if (wave == i % 4) s_row[i][lane] = page_row<PB>(p, id[i][0]);
        }
    }
    if (lane == 0) s_bits[wave] = bits;
    __syncthreads();
    bits = (uint32_t)__builtin_amdgcn_readfirstlane((int)(s_bits[0] & s_bits[1] & s_bits[2] & s_bits[3]));
    bool staged = false, finite = false;           // rows in LDS: those of the tile in hand; whose values are finite
#pragma unroll 1
    for (int n = 0; n < n_tiles; ++n) {
        uint8_t *done = p.tile_done + ((long)hk * tiles + tile0 + n) * p.splits + split;
        const int qrow = (tile0 + n) * 16 + c;
        staged = staged && ((bits >> (8 + n)) & 1) != 0;
        h8 qb[4];
#pragma unroll
        for (int k4 = 0; k4 < 4; ++k4) qb[k4] = qn[k4];
        if (n + 1 < n_tiles) queries(n + 1, qn);
        if (((bits >> n) & 1) == 0) {
            if (tid == 0) *done = 0;
            continue;
        }
        if (!staged) {
            if (n > 0) __syncthreads();                    // (the tile before has been multiplied)
            // ---- the rows: K row-major, V transposed, as in attn_prefix_body ----
            uint32_t bad = 0;
            {
                const int ch = tid & 15, kg = tid >> 4;
                u32x4 kv[4], vv[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const long off = s_row[n][4 * kg + e] * p.sfx_row_stride + (long)hk * p.sfx_head_stride + ch * 8;
                    const half_t *kp = (const half_t *)p.suffix_k + off, *vp = (const half_t *)p.suffix_v + off;
                    // (8-byte loads: a pool's rows are only that much aligned)
                    const u32x2 k0 = *reinterpret_cast<const u32x2 *>(kp), k1 = *reinterpret_cast<const u32x2 *>(kp + 4);
                    const u32x2 v0 = *reinterpret_cast<const u32x2 *>(vp), v1 = *reinterpret_cast<const u32x2 *>(vp + 4);
                    kv[e] = u32x4{k0[0], k0[1], k1[0], k1[1]};
                    vv[e] = u32x4{v0[0], v0[1], v1[0], v1[1]};
                }
#pragma unroll
                for (int e = 0; e < 4; ++e) {
#pragma unroll
                    for (int w = 0; w < 4; ++w) {          // (an exponent of all ones carries into the sign bit)
                        bad |= (kv[e][w] & 0x7fff7fffu) + 0x04000400u;
                        bad |= (vv[e][w] & 0x7fff7fffu) + 0x04000400u;
                    }
                    *reinterpret_cast<u32x4 *>(&ks[4 * kg + e][ch * 8]) = kv[e];
                }
                const int pos = vt_pos(4 * kg);
                const h8 v0 = __builtin_bit_cast(h8, vv[0]), v1 = __builtin_bit_cast(h8, vv[1]);
                const h8 v2 = __builtin_bit_cast(h8, vv[2]), v3 = __builtin_bit_cast(h8, vv[3]);
#pragma unroll
                for (int j = 0; j < 8; ++j) *reinterpret_cast<h4 *>(&vt[ch * 8 + j][pos]) = h4{v0[j], v1[j], v2[j], v3[j]};
            }
            finite = !__syncthreads_or((bad & 0x80008000u) != 0);
            staged = true;
        }
        if (tid == 0) *done = finite ? 1 : 0;
        if (!finite) continue;
        // ---- scores: element r of st is position 16 wave + 4 g + r (past the end: a repeated row, masked), column (query) c ----
        f4 st = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k4 = 0; k4 < 4; ++k4)
            st = __builtin_amdgcn_mfma_f32_16x16x32_f16(*reinterpret_cast<const h8 *>(&ks[16 * wave + c][32 * k4 + 8 * g]), qb[k4], st, 0, 0, 0);
        float mx = -INFINITY;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            st[r] = 16 * wave + 4 * g + r < cnt ? st[r] * p.scale_log2 : -INFINITY;
            mx = fmaxf(mx, st[r]);
        }
        mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        if (g == 0) s_max[wave][c] = mx;
        __syncthreads();
        mx = fmaxf(fmaxf(s_max[0][c], s_max[1][c]), fmaxf(s_max[2][c], s_max[3][c]));
        float sum = 0.f;
        h4 term[3];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float e = exp2f(st[r] - mx);
            sum += e;
            float left = e * 32768.f;
#pragma unroll
            for (int i = 0; i < 3; ++i) {              // (the differences and the powers of two are exact)
                term[i][r] = (half_t)left;
                left = (left - (float)term[i][r]) * 2048.f;
            }
        }
#pragma unroll
        for (int i = 0; i < 3; ++i) *reinterpret_cast<h4 *>(&ps[i][c][32 * (wave >> 1) + 8 * g + 4 * (wave & 1)]) = term[i];
        sum += __shfl_xor(sum, 16, 64);
        sum += __shfl_xor(sum, 32, 64);
        if (g == 0) s_sum[wave][c] = sum;
        __syncthreads();
        // ---- O^T: element r of o[i] is dim 32 wave + 16 i + 4 g + r, column (query) c ----
        f4 ot[3][2];                                   // by term
#pragma unroll
        for (int k = 0; k < 3; ++k)
#pragma unroll
            for (int i = 0; i < 2; ++i) ot[k][i] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int jj = 0; jj < PT_TW / 32; ++jj) {
            const h8 va[2] = {*reinterpret_cast<const h8 *>(&vt[32 * wave + c][32 * jj + 8 * g]), *reinterpret_cast<const h8 *>(&vt[32 * wave + 16 + c][32 * jj + 8 * g])};
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const h8 pb = *reinterpret_cast<const h8 *>(&ps[k][c][32 * jj + 8 * g]);
#pragma unroll
                for (int i = 0; i < 2; ++i) ot[k][i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(va[i], pb, ot[k][i], 0, 0, 0);
            }
        }
        if (qrow < p.Bq) {
            const long base = ((long)split * p.Hkv + hk) * p.Bq + qrow;
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                f4 o;
#pragma unroll
                for (int r = 0; r < 4; ++r) o[r] = (ot[0][i][r] + (ot[1][i][r] + ot[2][i][r] * 0x1p-11f) * 0x1p-11f) * 0x1p-15f;
                *reinterpret_cast<f4 *>(p.part_o + base * ATT_D + 32 * wave + 16 * i + 4 * g) = o;
            }
            if (wave == 0 && g == 0) {
                sum = s_sum[0][c] + s_sum[1][c] + s_sum[2][c] + s_sum[3][c];
                p.part_ml[base * 2] = partial_max(mx, sum);
                p.part_ml[base * 2 + 1] = sum;
            }
        }
    }
}

// ---- causal attention of a prefill on the matrix cores ----------------------------------------------------------
// A workgroup owns 32 QG consecutive query positions of one head; its 2 QG waves are QG groups of 32 queries x two key groups
// that take alternate key tiles (a wave alone on a SIMD waits for its own chain of products, exponentials and LDS reads; two
// keep the matrix cores twice as busy and halve the longest walk).  A wave's 32 queries are the columns of
// S^T = K . Q^T and of O^T += V^T . P^T, both in 32 x 32 x 16 products (an operand read from LDS feeds twice the multiply-adds
// of a 16-column tile: with 16 queries a wave the LDS reads alone took twice the matrix time).  It walks key tiles of 64 up to
// the diagonal with an online softmax; running maximum, sum and O^T stay in registers until the key groups are merged.  The accumulator of S^T
// holds keys 8 i + 4 hi + j of query lane % 32 (hi = lane / 32), so a lane's eight probabilities of 16 keys are a B operand of
// the second product if V^T lists its keys in that order (pv_slot).
//   * K tiles go global -> LDS by DMA, 16-byte chunks XOR-swizzled by the row; V goes through registers into its transposed
//     tile, swizzled so that neither the 8-byte stores nor the 16-byte reads pile up on a few banks.  Two buffers: the next
//     tile is on its way while one is multiplied, one barrier a tile.
//   * O^T is rescaled only when a maximum has grown by more than 2^4 (the probabilities are then at most 16, and the factor
//     cancels in the end): the rescale would be a quarter of the vector instructions of a tile.
//   * The longest walks are dispatched first.
// Bound by the vector ALU (exponentials) and the matrix cores together.  2047 rows x 32 heads: 187 us with 16 queries a wave and
// two barriers a tile, 68 with 32 queries and one key group, 56 (614 TFLOP/s) like this; 512 rows: 22.5 -> 13 us.
// (The two chains of S^T products interleaved, 32-bit row offsets, a higher wave priority for one key group: no gain.)
// q [S,H,128], k, v [S,Hkv,128], out [S,H,128].
constexpr int PF_TW = 64;                                  // keys of a tile
constexpr int PF_BUFFER_WORD3 = 4 << 15;                   // last word of an untyped buffer's descriptor: data format "32"
typedef float f16v __attribute__((ext_vector_type(16)));
typedef const __attribute__((address_space(1))) void *att_gptr_t;
typedef __attribute__((address_space(3))) void *att_lptr_t;
struct PrefillParams {
    const half_t *q, *k, *v;
    half_t *out;
    int S, H, Hkv, n_rep;
    float scale_log2;
};
// half-word slot of key t (0 .. 63) of dim d in V^T's row d
__device__ __forceinline__ int pv_slot(int t, int d) {
    const int chunk = 2 * (t >> 4) + ((t >> 2) & 1);       // sixteen keys are two chunks: hi = 0, hi = 1
    return ((chunk ^ (d & 7) ^ ((d >> 3) & 7)) << 3) + ((t >> 3) & 1) * 4 + (t & 3);
}

template <int QG>
__global__ __launch_bounds__(128 * QG, 1) void attn_prefill_kernel(PrefillParams p) {
    constexpr int NW = 2 * QG;
    constexpr int TILE = PF_TW * ATT_D;                    // halves of a K or V tile
    extern __shared__ __attribute__((aligned(16))) half_t pf_lds[];       // [buffer 2][key group 2][K | V] tiles
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, c = lane & 31, hi = lane >> 5;
    const int qg = wave % QG, kg = wave / QG;
    const int n_qb = (p.S + 32 * QG - 1) / (32 * QG);
    const int qb = n_qb - 1 - blockIdx.x / p.H, h = blockIdx.x % p.H, hk = h / p.n_rep;
    const int q_lo = 32 * (QG * qb + qg);                  // this wave's first query position
    const int my_q = q_lo + c;                             // this lane's query
    const int last_key = min(32 * QG * (qb + 1), p.S) - 1; // the workgroup's diagonal
    const int n_iter = last_key / (2 * PF_TW) + 1;         // pairs of tiles
    auto k_tile = [&](int buf, int g) { return pf_lds + (2 * (2 * buf + g)) * TILE; };
    auto v_tile = [&](int buf, int g) { return pf_lds + (2 * (2 * buf + g) + 1) * TILE; };

    h8 qop[8];                                             // B operand of S^T: dims 16 k + 8 hi .. of query c
    {
        const half_t *qp = p.q + ((long)min(my_q, p.S - 1) * p.H + h) * ATT_D + 8 * hi;
#pragma unroll
        for (int k = 0; k < 8; ++k) qop[k] = *reinterpret_cast<const h8 *>(qp + 16 * k);
    }
    const half_t *kbase = p.k + (long)hk * ATT_D, *vbase = p.v + (long)hk * ATT_D;
    const long row_stride = (long)p.Hkv * ATT_D;
    // K: instruction i of this wave moves four rows of the pair of tiles, lane -> (row lane / 16, slot lane % 16)
    auto k_fetch = [&](int it, int buf) {
#pragma unroll
        for (int i = 0; i < 32 / NW; ++i) {
            const int r4 = (32 / NW) * wave + i, r = 4 * r4 + (lane >> 4);             // row inside the pair
            const int row = min(it * 2 * PF_TW + r, p.S - 1);
            __builtin_amdgcn_global_load_lds((att_gptr_t)(kbase + (row * row_stride + 8 * ((lane & 15) ^ (r & 15)))),
                                             (att_lptr_t)(k_tile(buf, r4 >> 4) + (r4 & 15) * 4 * ATT_D), 16, 0, 0);
        }
    };
    // V: a thread moves 8 dims of FOUR consecutive keys, which sit side by side in a row of V^T
    constexpr int VG = 8 / NW;                             // groups of four keys per thread
    u32x4 vreg[VG][4];
    const int ch = tid & 15;
    auto v_fetch = [&](int it) {
        // Buffer loads over the rows of this pair of tiles that there are: past them they read zeros.  (A repeated last row would be
        // infinite where that row is, and its weight of 0 makes a NaN of it.)
        const int left = min(p.S - it * 2 * PF_TW, 2 * PF_TW), pitch = (int)row_stride * 2;
        const __amdgpu_buffer_rsrc_t rows = __builtin_amdgcn_make_buffer_rsrc(const_cast<half_t *>(vbase) + (long)it * 2 * PF_TW * row_stride, 0,
                                                                              (left - 1) * pitch + 2 * ATT_D, PF_BUFFER_WORD3);
#pragma unroll
        for (int g = 0; g < VG; ++g)
#pragma unroll
            for (int i = 0; i < 4; ++i) vreg[g][i] = __builtin_amdgcn_raw_buffer_load_b128(rows, (4 * ((tid >> 4) + 4 * NW * g) + i) * pitch + 16 * ch, 0, 0);
    };
    auto v_store = [&](int buf) {
#pragma unroll
        for (int g = 0; g < VG; ++g) {
            const int t = 4 * ((tid >> 4) + 4 * NW * g);
            half_t *vt = v_tile(buf, t / PF_TW);
            const h8 v0 = __builtin_bit_cast(h8, vreg[g][0]), v1 = __builtin_bit_cast(h8, vreg[g][1]);
            const h8 v2 = __builtin_bit_cast(h8, vreg[g][2]), v3 = __builtin_bit_cast(h8, vreg[g][3]);
#pragma unroll
            for (int j = 0; j < 8; ++j) *reinterpret_cast<h4 *>(&vt[(8 * ch + j) * PF_TW + pv_slot(t % PF_TW, 8 * ch + j)]) = h4{v0[j], v1[j], v2[j], v3[j]};
        }
    };

    float m_run = -INFINITY, l_run = 0.f;                  // maximum of query c's raw scores (both lanes of the query); sum over this lane's keys
    f16v ot[4];                                            // O^T: element r of ot[d] is dim 32 d + 8 (r / 4) + 4 hi + r % 4 of query c
#pragma unroll
    for (int d = 0; d < 4; ++d)
#pragma unroll
        for (int r = 0; r < 16; ++r) ot[d][r] = 0.f;

    k_fetch(0, 0);
    v_fetch(0);
    v_store(0);
    __syncthreads();                                       // (waits for the DMA too)
    for (int it = 0; it < n_iter; ++it) {
        const int buf = it & 1, k_lo = (2 * it + kg) * PF_TW;
        if (it + 1 < n_iter) {
            k_fetch(it + 1, buf ^ 1);
            v_fetch(it + 1);
        }
        if (k_lo <= q_lo + 31) {                           // (uniform over the wave) else every key lies after this wave's queries
            const half_t *ks = k_tile(buf, kg), *vt = v_tile(buf, kg);
            f16v st[2];
#pragma unroll
            for (int j = 0; j < 2; ++j) {
#pragma unroll
                for (int r = 0; r < 16; ++r) st[j][r] = 0.f;
                const int r = 32 * j + c;
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    const h8 ka = *reinterpret_cast<const h8 *>(&ks[r * ATT_D + 8 * ((2 * k + hi) ^ (r & 15))]);
                    st[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ka, qop[k], st[j], 0, 0, 0);
                }
            }
            if (k_lo + PF_TW - 1 > q_lo) {                 // the diagonal runs through this tile
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        const int key = k_lo + 32 * j + 8 * (r >> 2) + 4 * hi + (r & 3);
                        st[j][r] = key <= my_q ? st[j][r] : -INFINITY;
                    }
            }
            float mx = fmaxf(st[0][0], st[1][0]);
#pragma unroll
            for (int r = 1; r < 16; ++r) mx = fmaxf(fmaxf(st[0][r], st[1][r]), mx);
            mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
            const bool grown = (mx - m_run) * p.scale_log2 > 4.0f;       // (true at the first key, false while there is none: NaN)
            if (__any(grown)) {
                const float m_new = fmaxf(m_run, mx);
                const float alpha = m_run == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f((m_run - m_new) * p.scale_log2);
                m_run = m_new;
                l_run *= alpha;
#pragma unroll
                for (int d = 0; d < 4; ++d)
#pragma unroll
                    for (int r = 0; r < 16; ++r) ot[d][r] *= alpha;
            }
            const float m_scaled = m_run == -INFINITY ? 0.0f : m_run * p.scale_log2;
            h8 pb[4];
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const float e = __builtin_amdgcn_exp2f(__builtin_fmaf(st[j][r], p.scale_log2, -m_scaled));     // masked keys: exp2(-inf) = 0
                    l_run += e;
                    pb[2 * j + (r >> 3)][r & 7] = (half_t)e;
                }
#pragma unroll
            for (int b = 0; b < 4; ++b) {                  // sixteen keys at a time
                // (the second half of a tile that begins at this wave's first query: its keys weigh 0, but 0 times an infinite or NaN
                // value is NaN, so it stays out of the product)
                if (b == 2 && k_lo == q_lo) break;
#pragma unroll
                for (int d = 0; d < 4; ++d) {
                    const int row = 32 * d + c;
                    const h8 va = *reinterpret_cast<const h8 *>(&vt[row * PF_TW + (((2 * b + hi) ^ (row & 7) ^ ((row >> 3) & 7)) << 3)]);
                    ot[d] = __builtin_amdgcn_mfma_f32_32x32x16_f16(va, pb[b], ot[d], 0, 0, 0);
                }
            }
        }
        if (it + 1 < n_iter) v_store(buf ^ 1);
        __syncthreads();
    }
    // ---- the second key group's state through LDS (the tiles are no longer needed) ----
    float *part = reinterpret_cast<float *>(pf_lds) + (long)qg * (66 * 64) + lane;
    if (kg == 1) {
        part[0] = m_run;
        part[64] = l_run;
#pragma unroll
        for (int d = 0; d < 4; ++d)
#pragma unroll
            for (int r = 0; r < 16; ++r) part[(2 + 16 * d + r) * 64] = ot[d][r];
    }
    __syncthreads();
    if (kg == 1) return;
    const float m2 = part[0], m_new = fmaxf(m_run, m2);    // (finite: key 0 is in the first group's first tile)
    const float a1 = __builtin_amdgcn_exp2f((m_run - m_new) * p.scale_log2), a2 = __builtin_amdgcn_exp2f((m2 - m_new) * p.scale_log2);
    l_run = l_run * a1 + part[64] * a2;
    l_run += __shfl_xor(l_run, 32, 64);
    if (my_q < p.S) {
        const float inv = l_run > 0.f ? 1.0f / l_run : 0.f;
        half_t *op = p.out + ((long)my_q * p.H + h) * ATT_D + 4 * hi;
#pragma unroll
        for (int d = 0; d < 4; ++d)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                h4 o;
#pragma unroll
                for (int j = 0; j < 4; ++j) o[j] = (half_t)((ot[d][4 * i + j] * a1 + part[(2 + 16 * d + 4 * i + j) * 64] * a2) * inv);
                *reinterpret_cast<h4 *>(op + 32 * d + 8 * i) = o;
            }
    }
}
constexpr int PF_LDS = 8 * PF_TW * ATT_D * 2;              // 128 KB: one workgroup a compute unit

// One wave per (branch b, query head h): the query heads of one kv head walk the same suffix rows in different
// waves (the rows come from the cache after the first), so a wave's chain of memory round trips does not grow with
// the number of query heads per kv head.  PARTIAL: the pass over the suffix and the new token leaves an un-normalised
// partial (split index p.splits) for the workgroup that merges, instead of folding in the prefix partials itself.
// sub, nsub: nsub consecutive waves of the workgroup share the query; wave `sub` of them walks every
// nsub-th group of four rows, so that a long suffix is a single batch of loads per wave instead of a chain of
// batches; the waves' results are folded through LDS (every wave of the workgroup must then make this call; a wave
// without a query of its own passes a valid (b, h) and live = false, and writes nothing).
// WALK: the rows' format where it is known - a kernel that holds both walks needs registers for the larger one.  WALK_TILES:
// fp16, the slices that tile_done marks are skipped, and only their partials are folded in.
enum { WALK_ANY, WALK_Q40, WALK_F16, WALK_TILES };
template <bool FUSED, bool PARTIAL, int WALK = WALK_ANY, int PB = PB_ANY, int QKS = 16>
__device__ __forceinline__ void attn_suffix_body(const AttnParams &p, int b, int h, int sub = 0, int nsub = 1, bool live = true) {
    constexpr bool TILES = WALK == WALK_TILES;
    const int hk = div_rep(p, h);
    __shared__ __attribute__((aligned(16))) half_t s_kv[FUSED ? 4 : 1][3][ATT_D];     // FUSED: this wave's new k and v rows, its query
    __shared__ float s_fold[4][16][10];                                                 // nsub > 1: the waves' states (m, l, o[8])
    // Lane = 16 g + Q4_LPR rl + e.  In the Q4_0 walk below a row belongs to the Q4_LPR lanes (g, rl, 0..Q4_LPR-1), lane e
    // holding bytes (64 / Q4_LPR) e .. of it; everywhere else the 16 lanes of group g share a row in eight-dim pieces, lane
    // (rl, e) taking piece c = Q4_DW e + rl - a piece whose dims are among those the lane holds in the walk, so that the
    // walk's result needs no exchange between lanes with different e.
    // Measured (64 branches x 32 heads, ragged suffixes of 0..256 rows / 100 branches at ~55 rows): 8 lanes a row and 2 passes a
    // chunk 22.1 / 14.2 us; 4 lanes 23.6 / 16.2 (more registers, 64 lane exchanges at the end); 16 lanes 26.6 / 14.3; 4 passes
    // a chunk 23.9 / 15.8, 1 pass 23.7 / 13.8.  Before (16 lanes, 4 rows a batch, no request ahead): 28.6 / 14.8 us.
    constexpr int Q4_LPR = 8;                              // lanes per row (4, 8 or 16)
    constexpr int Q4_DW = 16 / Q4_LPR;                     // dwords of a row's 64 bytes per lane = row slots per group
    constexpr int Q4_ROWS = 4 * Q4_DW;                     // rows per pass of the wave
    constexpr int Q4_CH = 2;                               // passes per chunk
    const int lane = threadIdx.x & 63, g = lane >> 4, e = lane & (Q4_LPR - 1), rl = (lane & 15) / Q4_LPR, c = Q4_DW * e + rl;
    const int wave = threadIdx.x >> 6;
    int len = 0;
    // a length beyond the branch's rows (a device counter that ran past the cache) is cut at the cache's end
    // (no lengths: every branch has all its rows)
    if (p.suffix_format != SMH_KV_NONE) len = p.lens == nullptr ? (int)p.suffix_batch_stride_rows : min(p.lens[(long)b * p.lens_stride], (int)p.suffix_batch_stride_rows);
    const int gg = g + 4 * sub, gstride = 4 * nsub;      // this group's first row and the distance to its next one
    const long row0 = (long)b * p.suffix_batch_stride_rows;     // first suffix row of this branch
    // page id of suffix position t of this branch, as it comes from memory, and the pool row that it means
    typedef page_id_t<PB> id_t;
    auto id_of = [&](int t) -> id_t {
        if constexpr (PB == PB_ANY) {
            if (p.pages == nullptr) return row0 + t;
            return page_row<PB>(p, page_at<PB>(p, (long)b * p.pages_stride + t));
        } else {
            if constexpr (PB == 0) return t;
            else return page_at<PB>(p, (long)b * p.pages_stride + t);
        }
    };
    auto row_of = [&](id_t id) -> long {
        if constexpr (PB == PB_ANY) return id;
        else if constexpr (PB == 0) return row0 + id;
        else return page_row<PB>(p, id);
    };
    // ---- Q4_0 suffix rows: a wave takes Q4_ROWS rows per pass (row slot Q4_DW g + rl) and Q4_CH passes per chunk; wave
    // `sub` of the nsub that share a query takes every nsub-th pass.  All loads of a chunk are requested together, and
    // the next chunk's before this one is used: the time of this walk is its dependent trips to memory (page id -> row)
    // and its instructions, not its bytes. ----
    typedef uint32_t q4_dw_t __attribute__((ext_vector_type(Q4_DW > 1 ? Q4_DW : 2)));
    struct Q4One { uint32_t x; __device__ uint32_t operator[](int) const { return x; } };
    typedef std::conditional_t<Q4_DW == 1, Q4One, q4_dw_t> q4_reg_t;
    struct Q4Chunk { q4_reg_t k[Q4_CH], v[Q4_CH]; uint32_t ks[Q4_CH], vs[Q4_CH]; };
    const int q4_passes = p.suffix_format == SMH_KV_Q40 ? (len + Q4_ROWS - 1) / Q4_ROWS : 0;     // passes over all waves of the query
    const int q4_mine = q4_passes > sub ? (q4_passes - sub + nsub - 1) / nsub : 0;                // passes of this wave
    const int q4_chunks = (q4_mine + Q4_CH - 1) / Q4_CH;
    auto q4_pos = [&](int n, int u) { return Q4_ROWS * (sub + nsub * (Q4_CH * n + u)) + Q4_DW * g + rl; };  // suffix position of this lane's row
    auto q4_ids = [&](int n, id_t (&id)[Q4_CH]) {
#pragma unroll
        for (int u = 0; u < Q4_CH; ++u) id[u] = id_of(min(q4_pos(n, u), len - 1));                // rows past the end repeat the last one
    };
    auto q4_rows = [&](const id_t (&id)[Q4_CH], Q4Chunk &ck) {
#pragma unroll
        for (int u = 0; u < Q4_CH; ++u) {
            const long row = row_of(id[u]) * p.Hkv + hk;
            ck.k[u] = *reinterpret_cast<const q4_reg_t *>((const uint8_t *)p.suffix_k + row * 64 + 4 * Q4_DW * e);
            ck.v[u] = *reinterpret_cast<const q4_reg_t *>((const uint8_t *)p.suffix_v + row * 64 + 4 * Q4_DW * e);
            ck.ks[u] = *reinterpret_cast<const uint32_t *>(p.suffix_ks + row * 2);
            ck.vs[u] = *reinterpret_cast<const uint32_t *>(p.suffix_vs + row * 2);
        }
    };
    Q4Chunk q4_first;                                       // chunk 0, requested as early as the length is known
    id_t q4_next_id[Q4_CH];                                 // page ids of the chunk after the one in flight
    auto q4_prime = [&]() {
        if (q4_chunks > 0) {
            q4_ids(0, q4_next_id);
            q4_rows(q4_next_id, q4_first);
            if (q4_chunks > 1) q4_ids(1, q4_next_id);
        }
    };
    RowRegs q_first;
    int pos = 0;
    if (FUSED) {
        // Two round trips to memory, not more: first everything that depends on no other load - the suffix length
        // (requested above), the position, the suffix index and the slabs of q, k and v (lane owns the rotation pair
        // (lane, lane + 64) of each: 2 x ksplit loads of 4 bytes; read in the row layout, 8 dims a lane, q's slabs
        // alone take 128 registers and the requests leave one after the other) - then what depends on the length
        // (the first batch of rows) and on the position (the rotation factors).  q changes to the row layout
        // through LDS; k is rotated, k and v are appended to the branch's suffix cache as Q4_0 and left in LDS as
        // exact fp16 for the pass below.
        pos = *p.pos_dev;
        int t = -1;
        float cq1[QKS], cq2[QKS], ck1[QKS], ck2[QKS], cv1[QKS], cv2[QKS];
        qkv_request(p, b, h * ATT_D + lane, cq1);
        qkv_request(p, b, h * ATT_D + lane + 64, cq2);
        if (sub == 0) {                                            // the wave that owns the new token
            t = p.app_k != nullptr ? *p.app_t : -1;
            const int kcol = (p.H + hk) * ATT_D, vcol = (p.H + p.Hkv + hk) * ATT_D;
            qkv_request(p, b, kcol + lane, ck1); qkv_request(p, b, kcol + lane + 64, ck2);
            qkv_request(p, b, vcol + lane, cv1); qkv_request(p, b, vcol + lane + 64, cv2);
        }
        q4_prime();
        const half_t cos_l = p.cos_tab[(long)pos * 64 + lane], sin_l = p.sin_tab[(long)pos * 64 + lane];
        half_t q1 = (half_t)qkv_sum(p, cq1), q2 = (half_t)qkv_sum(p, cq2);
        half_t k1 = q1, k2 = q1, v1 = q1, v2 = q1;
        if (sub == 0) { k1 = (half_t)qkv_sum(p, ck1); k2 = (half_t)qkv_sum(p, ck2); v1 = (half_t)qkv_sum(p, cv1); v2 = (half_t)qkv_sum(p, cv2); }
        rope_pair2(q1, q2, cos_l, sin_l);
        s_kv[wave][2][lane] = q1; s_kv[wave][2][lane + 64] = q2;
        asm volatile("" ::: "memory");                              // the reads below are of another type: keep them behind the writes
        q_first = row_from_fp16(&s_kv[wave][2][0], c);             // same wave writes and reads: LDS operations complete in order
        if (sub == 0) {
            rope_pair2(k1, k2, cos_l, sin_l);
            if (live && h == hk * p.n_rep && t >= 0 && t < p.app_smax) {     // the first query head of a kv head appends the rows
                const long row = ((long)b * p.app_smax + t) * p.Hkv + hk;
                kv_store_row2(k1, k2, p.app_k + row * 64, p.app_ks + row * 2, lane);
                kv_store_row2(v1, v2, p.app_v + row * 64, p.app_vs + row * 2, lane);
            }
            s_kv[wave][0][lane] = k1; s_kv[wave][0][lane + 64] = k2;
            s_kv[wave][1][lane] = v1; s_kv[wave][1][lane + 64] = v2;
            asm volatile("" ::: "memory");
            // same wave writes and reads: LDS operations of a wave complete in order
        }
    }

    {
        // Not FUSED: the query (in the walk over Q4_0 rows its dims this lane holds of a row, pieces Q4_DW e + j, c among them) and the new
        // token's rows are requested here and used behind the first rows of the walk.
        constexpr bool Q4_ONLY = WALK == WALK_Q40;
        constexpr int NQ = Q4_ONLY ? Q4_DW : 1;
        const half_t *q_ptr = FUSED ? nullptr : p.q + ((long)b * p.H + h) * ATT_D;
        RawRow q_raw[NQ], cur_raw[2];
        if constexpr (!FUSED) {
#pragma unroll
            for (int j = 0; j < NQ; ++j) q_raw[j] = raw_row(q_ptr, Q4_ONLY ? Q4_DW * e + j : c);
            if constexpr (WALK < WALK_F16) {                // (the fp16 walk needs the registers)
                const long off = ((long)b * p.Hkv + hk) * ATT_D;
                cur_raw[0] = raw_row(p.cur_k != nullptr ? p.cur_k + off : q_ptr, c);
                cur_raw[1] = raw_row(p.cur_k != nullptr ? p.cur_v + off : q_ptr, c);
            }
        }
        SoftState st;
        st.m = -INFINITY;
        st.l = 0.f;
#pragma unroll
        for (int j = 0; j < 8; ++j) st.o[j] = 0.f;

        // Every load below is issued before its first use, a batch at a time: a wave has few rows to visit
        // (tens, a quarter each per group), so its time is the number of memory round trips it makes in a row.
        // ---- loads for the end of the pass: the new token's exact K/V, the first two prefix partials ----
        const int qrow = b * p.n_rep + (h - hk * p.n_rep);
        const bool has_cur = (FUSED || p.cur_k != nullptr) && g == 0 && sub == 0;
        constexpr int PRE = WALK < WALK_F16 ? 2 : 0;
        f4 pre_lo[PRE + 1], pre_hi[PRE + 1];
        float pre_m[PRE + 1], pre_l[PRE + 1];
#pragma unroll
        for (int i = 0; i < PRE; ++i) {
            const int sp = gg + gstride * i;
            if (!PARTIAL && sp < p.splits) {
                const long base = ((long)sp * p.Hkv + hk) * p.Bq + qrow;
                pre_lo[i] = *reinterpret_cast<const f4 *>(p.part_o + base * ATT_D + 4 * c);
                pre_hi[i] = *reinterpret_cast<const f4 *>(p.part_o + base * ATT_D + 64 + 4 * c);
                pre_m[i] = p.part_ml[base * 2];
                pre_l[i] = p.part_ml[base * 2 + 1];
            }
        }
        // ---- this branch's suffix: group g takes rows g, g+4, ... in batches ----
        uint64_t tiles = 0;                                 // bit s: slice s is done
        constexpr int TILE_PARTS = TILES ? 2 : 0;           // partials of a group that are folded in before the walk
        if (WALK == WALK_F16 || TILES || (WALK == WALK_ANY && p.suffix_format == SMH_KV_FP16)) {
            // Batches of U rows per group, the next one (and the ids of the one after it) on its way while this one is used; one
            // maximum and one rescale a batch.
            constexpr int U = 4;
            static_assert(PT_TW % (4 * 4 * U) == 0, "a batch of the waves of a query lies in one slice");
            const int span = gstride * U, n_batches = (len + span - 1) / span;
            auto next = [&](int i) {
                ++i;
                if (TILES) while (i < n_batches && ((tiles >> (i * span / PT_TW)) & 1) != 0) ++i;
                return i;
            };
            struct Batch { u32x2 kl[U], kh[U], vl[U], vh[U]; };
            std::conditional_t<PB == PB_ANY, int, id_t> id[U];         // (rows of 256 bytes and more: their number fits)
            auto ids = [&](int i) {
#pragma unroll
                for (int u = 0; u < U; ++u) id[u] = id_of(min(span * i + gg + gstride * u, len - 1));             // past the end: the last row again
            };
            auto rows = [&](Batch &r) {
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const long off = row_of(id[u]) * p.sfx_row_stride + (long)hk * p.sfx_head_stride + 4 * c;
                    r.kl[u] = *reinterpret_cast<const u32x2 *>((const half_t *)p.suffix_k + off);
                    r.kh[u] = *reinterpret_cast<const u32x2 *>((const half_t *)p.suffix_k + off + 64);
                    r.vl[u] = *reinterpret_cast<const u32x2 *>((const half_t *)p.suffix_v + off);
                    r.vh[u] = *reinterpret_cast<const u32x2 *>((const half_t *)p.suffix_v + off + 64);
                }
            };
            // dims (0,1), (2,3)
            u32x2 ql, qh;
            if constexpr (FUSED) {
                ql = u32x2{pack_lo16(as_u32(q_first.a02), as_u32(q_first.a13)), pack_hi16(as_u32(q_first.a02), as_u32(q_first.a13))};
                qh = u32x2{pack_lo16(as_u32(q_first.b02), as_u32(q_first.b13)), pack_hi16(as_u32(q_first.b02), as_u32(q_first.b13))};
            } else {
                ql = q_raw[0].lo;
                qh = q_raw[0].hi;
            }
            // What the walk begins with comes in as few trips as there are dependent loads: the first ids (of no use where the first slice is done) with the
            // marks, the slices' partials with the first rows and not behind the last (us, in turn, the grid of attn_page_tile_kernel included: 32 heads,
            // 99 branches, 512 positions, 256 of them a prompt 87.3 -> 84.8, 62 branches, 273 positions, 95 of them 37.3 -> 34.6, 4 branches, 683
            // positions 16.0 -> 15.0; nothing shared over a slice, 2 to 99 branches, 96 to 512 positions: 0.98 .. 1.09 times as fast, the least with 64-bit ids).
            if constexpr (TILES) {
                const uint8_t mark = p.tile_done[((long)hk * ((p.Bq + 15) / 16) + (qrow >> 4)) * p.splits + min(lane, p.splits - 1)];
                ids(0);
                tiles = __ballot(lane < p.splits && mark != 0);
            }
            int i0 = next(-1), i1 = n_batches;
            Batch cur;
            if (i0 < n_batches) {
                if (!TILES || i0 > 0) ids(i0);
                rows(cur);
                i1 = next(i0);
                if (i1 < n_batches) ids(i1);
            }
            f4 part_lo[TILE_PARTS + 1], part_hi[TILE_PARTS + 1];
            float part_m[TILE_PARTS + 1], part_l[TILE_PARTS + 1];
#pragma unroll
            for (int i = 0; i < TILE_PARTS; ++i) {
                const int sp = gg + gstride * i;
                if (sp < p.splits && ((tiles >> sp) & 1) != 0) {
                    const long base = ((long)sp * p.Hkv + hk) * p.Bq + qrow;
                    part_lo[i] = *reinterpret_cast<const f4 *>(p.part_o + base * ATT_D + 4 * c);
                    part_hi[i] = *reinterpret_cast<const f4 *>(p.part_o + base * ATT_D + 64 + 4 * c);
                    part_m[i] = p.part_ml[base * 2];
                    part_l[i] = p.part_ml[base * 2 + 1];
                }
            }
            wait_loads();
#pragma unroll
            for (int i = 0; i < TILE_PARTS; ++i) {
                const int sp = gg + gstride * i;
                if (sp < p.splits && ((tiles >> sp) & 1) != 0) {
                    const float o2[8] = {part_lo[i][0], part_lo[i][2], part_lo[i][1], part_lo[i][3], part_hi[i][0], part_hi[i][2], part_hi[i][1], part_hi[i][3]};
                    soft_merge(st, part_m[i], part_l[i], o2);
                }
            }
            while (i0 < n_batches) {
                Batch nxt;
                int i2 = n_batches;
                if (i1 < n_batches) {
                    rows(nxt);
                    i2 = next(i1);
                    if (i2 < n_batches) ids(i2);
                }
                float sc[U];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    float d = __builtin_amdgcn_fdot2(as_h2(cur.kl[u][0]), as_h2(ql[0]), 0.f, false);
                    d = __builtin_amdgcn_fdot2(as_h2(cur.kl[u][1]), as_h2(ql[1]), d, false);
                    d = __builtin_amdgcn_fdot2(as_h2(cur.kh[u][0]), as_h2(qh[0]), d, false);
                    d = __builtin_amdgcn_fdot2(as_h2(cur.kh[u][1]), as_h2(qh[1]), d, false);
                    sc[u] = row16_sum(d) * p.scale_log2;
                }
                if (span * (i0 + 1) > len) {                // (uniform) the last batch: a repeated row weighs nothing, also where it is infinite
#pragma unroll
                    for (int u = 0; u < U; ++u)
                        if (span * i0 + gg + gstride * u >= len) {
                            sc[u] = -INFINITY;
                            cur.vl[u] = u32x2{0, 0};
                            cur.vh[u] = u32x2{0, 0};
                        }
                }
                float mx = sc[0];
#pragma unroll
                for (int u = 1; u < U; ++u) mx = fmaxf(mx, sc[u]);
                const float m_new = fmaxf(st.m, mx), m_ref = m_new == -INFINITY ? 0.f : m_new;
                const float corr = __builtin_amdgcn_exp2f(st.m - m_ref);
                st.m = m_new;
                st.l *= corr;
#pragma unroll
                for (int k = 0; k < 8; ++k) st.o[k] *= corr;
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const float pr = __builtin_amdgcn_exp2f(sc[u] - m_ref);
                    st.l += pr;
                    const h2 v01 = as_h2(cur.vl[u][0]), v23 = as_h2(cur.vl[u][1]), w01 = as_h2(cur.vh[u][0]), w23 = as_h2(cur.vh[u][1]);
                    st.o[0] += pr * (float)v01.x; st.o[2] += pr * (float)v01.y;
                    st.o[1] += pr * (float)v23.x; st.o[3] += pr * (float)v23.y;
                    st.o[4] += pr * (float)w01.x; st.o[6] += pr * (float)w01.y;
                    st.o[5] += pr * (float)w23.x; st.o[7] += pr * (float)w23.y;
                }
                cur = nxt;
                i0 = i1;
                i1 = i2;
            }
        } else if (WALK <= WALK_Q40 && q4_chunks > 0) {
            if (!FUSED) q4_prime();
            RowRegs qj[Q4_DW];                              // the query's dims this lane holds of a row: pieces Q4_DW e + j
#pragma unroll
            for (int j = 0; j < Q4_DW; ++j)
                qj[j] = FUSED ? row_from_fp16(&s_kv[wave][2][0], Q4_DW * e + j) : Q4_ONLY ? row_of_raw(q_raw[j < NQ ? j : 0]) : row_from_fp16(q_ptr, Q4_DW * e + j);
            float m = -INFINITY, l = 0.f;                   // m: common to the group; l, o: of this lane's row slot
            float o[Q4_DW][8];
#pragma unroll
            for (int j = 0; j < Q4_DW; ++j)
#pragma unroll
                for (int k = 0; k < 8; ++k) o[j][k] = 0.f;
            Q4Chunk cur = q4_first;
            const RowCodes codes;
            wait_loads();
            for (int n = 0; n < q4_chunks; ++n) {
                Q4Chunk nxt;
                if (n + 1 < q4_chunks) {
                    q4_rows(q4_next_id, nxt);
                    if (n + 2 < q4_chunks) q4_ids(n + 2, q4_next_id);
                }
                float sc[Q4_CH];
#pragma unroll
                for (int u = 0; u < Q4_CH; ++u) {
                    float d = 0.f;
#pragma unroll
                    for (int j = 0; j < Q4_DW; ++j) {
                        const RowRegs kr = row_from_q40(cur.k[u][j], cur.ks[u], codes);
                        d = __builtin_amdgcn_fdot2(kr.a02, qj[j].a02, d, false);
                        d = __builtin_amdgcn_fdot2(kr.a13, qj[j].a13, d, false);
                        d = __builtin_amdgcn_fdot2(kr.b02, qj[j].b02, d, false);
                        d = __builtin_amdgcn_fdot2(kr.b13, qj[j].b13, d, false);
                    }
                    d += dpp_move<DPP_QUAD_XOR1>(d);        // the lanes that share the row
                    d += dpp_move<DPP_QUAD_XOR2>(d);
                    if (Q4_LPR >= 8) d += dpp_move<DPP_ROW_HALF_MIRROR>(d);
                    if (Q4_LPR == 16) d += dpp_move<DPP_ROW_ROR8>(d);
                    sc[u] = q4_pos(n, u) < len ? d * p.scale_log2 : -INFINITY;
                }
                float mx = sc[0];
#pragma unroll
                for (int u = 1; u < Q4_CH; ++u) mx = fmaxf(mx, sc[u]);
                if (Q4_LPR <= 8) mx = fmaxf(mx, dpp_move<DPP_ROW_ROR8>(mx)); // the row slots of the group
                if (Q4_LPR == 4) mx = fmaxf(mx, dpp_move<DPP_ROW_ROR4>(mx));
                const float m_new = fmaxf(m, mx);
                const float m_ref = m_new == -INFINITY ? 0.f : m_new;    // a group without a row yet: every factor below is exp2(-inf) = 0
                const float corr = exp2f(m - m_ref);
                m = m_new;
                l *= corr;
#pragma unroll
                for (int j = 0; j < Q4_DW; ++j)
#pragma unroll
                    for (int k = 0; k < 8; ++k) o[j][k] *= corr;
#pragma unroll
                for (int u = 0; u < Q4_CH; ++u) {
                    const float pr = exp2f(sc[u] - m_ref);
                    l += pr;
#pragma unroll
                    for (int j = 0; j < Q4_DW; ++j) {
                        const RowRegs vr = row_from_q40(cur.v[u][j], cur.vs[u], codes);
                        o[j][0] += pr * (float)vr.a02.x; o[j][1] += pr * (float)vr.a02.y;
                        o[j][2] += pr * (float)vr.a13.x; o[j][3] += pr * (float)vr.a13.y;
                        o[j][4] += pr * (float)vr.b02.x; o[j][5] += pr * (float)vr.b02.y;
                        o[j][6] += pr * (float)vr.b13.x; o[j][7] += pr * (float)vr.b13.y;
                    }
                }
                cur = nxt;
            }
            // the group's row slots added up, then lane (rl, e) keeps piece Q4_DW e + rl = c
            if (Q4_LPR <= 8) l += dpp_move<DPP_ROW_ROR8>(l);
            if (Q4_LPR == 4) l += dpp_move<DPP_ROW_ROR4>(l);
#pragma unroll
            for (int j = 0; j < Q4_DW; ++j)
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    if (Q4_LPR <= 8) o[j][k] += dpp_move<DPP_ROW_ROR8>(o[j][k]);
                    if (Q4_LPR == 4) o[j][k] += dpp_move<DPP_ROW_ROR4>(o[j][k]);
                }
            st.m = m;
            st.l = l;
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                float v = o[0][k];
#pragma unroll
                for (int j = 1; j < Q4_DW; ++j) v = rl == j ? o[j][k] : v;
                st.o[k] = v;
            }
        }
        // ---- the new token's exact K/V (group 0 only) ----
        if (has_cur) {
            RowRegs qr, kr, vr;
            if constexpr (FUSED) {
                qr = q_first;
                kr = row_from_fp16(&s_kv[wave][0][0], c);
                vr = row_from_fp16(&s_kv[wave][1][0], c);
            } else {
                RawRow q_c = q_raw[0];                      // piece c
#pragma unroll
                for (int j = 1; j < NQ; ++j)
#pragma unroll
                    for (int i = 0; i < 2; ++i) {
                        q_c.lo[i] = rl == j ? q_raw[j].lo[i] : q_c.lo[i];
                        q_c.hi[i] = rl == j ? q_raw[j].hi[i] : q_c.hi[i];
                    }
                qr = row_of_raw(q_c);
                if constexpr (WALK >= WALK_F16) {
                    const long off = ((long)b * p.Hkv + hk) * ATT_D;
                    kr = row_from_fp16(p.cur_k + off, c);
                    vr = row_from_fp16(p.cur_v + off, c);
                } else {
                    kr = row_of_raw(cur_raw[0]);
                    vr = row_of_raw(cur_raw[1]);
                }
            }
            soft_add_row(st, row_dot(kr, qr) * p.scale_log2, vr);
        }
        // ---- prefix partials: the group folds in splits gg, gg + gstride, ... ----
#pragma unroll
        for (int i = 0; i < PRE; ++i) {
            if (!PARTIAL && gg + gstride * i < p.splits) {
                const float o2[8] = {pre_lo[i][0], pre_lo[i][2], pre_lo[i][1], pre_lo[i][3], pre_hi[i][0], pre_hi[i][2], pre_hi[i][1], pre_hi[i][3]};
                soft_merge(st, pre_m[i], pre_l[i], o2);
            }
        }
        for (int sp = gg + gstride * (PRE + TILE_PARTS); !PARTIAL && sp < p.splits; sp += gstride) {
            if (TILES && ((tiles >> sp) & 1) == 0) continue;
            const long base = ((long)sp * p.Hkv + hk) * p.Bq + qrow;
            const f4 lo = *reinterpret_cast<const f4 *>(p.part_o + base * ATT_D + 4 * c);
            const f4 hi = *reinterpret_cast<const f4 *>(p.part_o + base * ATT_D + 64 + 4 * c);
            const float o2[8] = {lo[0], lo[2], lo[1], lo[3], hi[0], hi[2], hi[1], hi[3]};
            soft_merge(st, p.part_ml[base * 2], p.part_ml[base * 2 + 1], o2);
        }
        // ---- merge the four groups (xor 16, xor 32) ----
#pragma unroll
        for (int sh = 16; sh <= 32; sh <<= 1) {
            const float m2 = __shfl_xor(st.m, sh, 64);
            const float l2 = __shfl_xor(st.l, sh, 64);
            float o2[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) o2[j] = __shfl_xor(st.o[j], sh, 64);
            soft_merge(st, m2, l2, o2);
        }
        if (nsub > 1) {                                // (uniform over the workgroup)
            if (g == 0) {
                float *mine = s_fold[wave][c];
                mine[0] = st.m; mine[1] = st.l;
#pragma unroll
                for (int j = 0; j < 8; ++j) mine[2 + j] = st.o[j];
            }
            __syncthreads();
            if (g == 0 && sub == 0)
                for (int k = 1; k < nsub; ++k) soft_merge(st, s_fold[wave + k][c][0], s_fold[wave + k][c][1], &s_fold[wave + k][c][2]);
        }
        if (g == 0 && PARTIAL) {
            if (sub != 0 || !live) return;
            const long base = ((long)p.splits * p.Hkv + hk) * p.Bq + qrow;
            st_f4(p.part_o + base * ATT_D + 4 * c, f4{st.o[0], st.o[2], st.o[1], st.o[3]});
            st_f4(p.part_o + base * ATT_D + 64 + 4 * c, f4{st.o[4], st.o[6], st.o[5], st.o[7]});
            if (c == 0) { st_f32(p.part_ml + base * 2, partial_max(st.m, st.l)); st_f32(p.part_ml + base * 2 + 1, st.l); }
        } else if (g == 0 && sub == 0 && live) {
            const float inv = st.l > 0.f ? 1.0f / st.l : 0.f;
            half_t *op = p.out + ((long)b * p.H + h) * ATT_D;
            h4 lo = {(half_t)(st.o[0] * inv), (half_t)(st.o[2] * inv), (half_t)(st.o[1] * inv), (half_t)(st.o[3] * inv)};
            h4 hi = {(half_t)(st.o[4] * inv), (half_t)(st.o[6] * inv), (half_t)(st.o[5] * inv), (half_t)(st.o[7] * inv)};
            *reinterpret_cast<h4 *>(op + 4 * c) = lo;
            *reinterpret_cast<h4 *>(op + 64 + 4 * c) = hi;
        }
    }
}

// (four waves a SIMD: with three, the 3168 waves of 99 branches x 32 heads left a second round of a few; 99 branches x 32 heads over 768
// positions of a page table 171 -> 150 us)
template <bool FUSED, int WALK, int PB>
__global__ __launch_bounds__(256, FUSED ? 1 : 4) void attn_suffix_kernel(AttnParams p) {
    args_ahead<sizeof(AttnParams)>();
    // suffix_waves (1, 2 or 4) waves per (branch, query head): more than one while branches x heads leave CUs idle.
    // Workgroups are dealt round-robin to the 8 XCDs (8 L2s); the heads of one branch share the 128-byte lines of that
    // branch's scales (2 fp16 per head and position), so ALL workgroups of a branch go to one XCD: workgroup L of the 1-D
    // grid sits on XCD L % 8 and takes branch 8 (L / 8 / per_branch) + L % 8, head group (L / 8) % per_branch.
    // (Branches share pages: the queries of a kv head on one XCD instead measured 104 us against 100 at 99 branches x 512 positions.)
    const int wave = threadIdx.x >> 6, nsub = p.suffix_waves;
    const int per_branch = (p.H * nsub + 3) >> 2;              // workgroups (four waves) per branch
    const int L = blockIdx.x, j = L >> 3;
    const int grp = uniform_divmod(j, per_branch).q;
    const int b = 8 * grp + (L & 7);
    if (b >= p.B) return;
    const int hq = (j - grp * per_branch) * 4 + wave;
    const int h = nsub == 4 ? hq >> 2 : (nsub == 2 ? hq >> 1 : hq);
    if (nsub == 1 && h >= p.H) return;
    // with shared queries every wave reaches the fold's barrier: one past the last head repeats it and writes nothing
    attn_suffix_body<FUSED, false, WALK, PB>(p, b, min(h, p.H - 1), hq & (nsub - 1), nsub, h < p.H);
}

// ---- prefix slices and suffix walks side by side, then a merge ------------------------------------------------------
// The walk waits for memory, the prefix slices for their own chain of staging and products: in one launch they overlap, and
// what is left for the second is to add the partials up.  Workgroups 0 .. prefix_wgs - 1 take (slice, 64 queries, kv head), the
// others walk.  Both kinds share a compute unit, so a prefix workgroup may hold no more LDS than a quarter of it: K and then
// V^T in the same 34 KB (V waits in registers), one tile of 16 queries a wave.
// fp16 suffixes only.  Against the prefix launch and then the walk: 100 branches x 32 heads after 512 shared rows, suffixes of up
// to 256 rows, 65.6 -> 59.0 us a call, 64 after 1024 45.5 -> 43.6, 16 after 512 15.6 -> 14.4, one branch 12.3 either way.  A walk over
// Q4_0 rows is a quarter of the bytes and hides less than the merge costs: decode steps of the 7B architecture at 17, 64 and 100 branches 2.59,
// 3.30 and 4.01 ms as two launches in turn, 2.64, 3.35 and 3.96 like this.
constexpr int AP_PITCH = ATT_TW_MAX + 8;
__device__ __forceinline__ void attn_prefix_round(const AttnParams &p, int split, int hk, int round) {
    static_assert(ATT_KPITCH == AP_PITCH && ATT_D == ATT_TW_MAX, "K and V^T have one shape");
    __shared__ __attribute__((aligned(16))) half_t kv_lds[ATT_D][AP_PITCH];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, c = lane & 15, g = lane >> 4;
    const int t0 = split * p.tw, cnt = min(p.tw, p.P - t0), tw32 = (cnt + 31) & ~31, t_tiles = tw32 / 16;
    const int qt = 4 * round + wave;
    const bool live = qt * 16 < p.Bq;                        // (uniform over the wave)
    h8 qb[4];
    {
        const int qr = min(qt * 16 + c, p.Bq - 1);
        const half_t *qp = p.q + ((long)div_rep(p, qr) * p.H + hk * p.n_rep + mod_rep(p, qr)) * ATT_D + 8 * g;
#pragma unroll
        for (int k4 = 0; k4 < 4; ++k4) qb[k4] = *reinterpret_cast<const h8 *>(qp + 32 * k4);
    }
    const int ch = tid & 15;
    u32x4 kr[2][4], vr[2][4];                                // this thread's 8 dims of rows 4 kg .. 4 kg + 3, kg = tid / 16 and 16 more
    auto fetch = [&](const half_t *base, u32x4 (&r)[2][4]) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int t = 4 * ((tid >> 4) + 16 * i) + e;
                r[i][e] = u32x4{0, 0, 0, 0};
                if (t < cnt) r[i][e] = *reinterpret_cast<const u32x4 *>(base + (long)(t0 + t) * p.pfx_row_stride + (long)hk * p.pfx_head_stride + ch * 8);
            }
    };
    fetch(p.prefix_k, kr);
    fetch(p.prefix_v, vr);
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int t = 4 * ((tid >> 4) + 16 * i) + e;
            if (t < tw32) *reinterpret_cast<u32x4 *>(&kv_lds[t][ch * 8]) = kr[i][e];
        }
    __syncthreads();
    f4 st[ATT_TW_MAX / 16];                                  // S^T: element r of st[j] is row 16 j + 4 g + r, column (query) c
    float mx = -INFINITY, sum = 0.f;
    if (live) {
#pragma unroll
        for (int j = 0; j < ATT_TW_MAX / 16; ++j) {
            st[j] = f4{0.f, 0.f, 0.f, 0.f};
            if (j < t_tiles) {
#pragma unroll
                for (int k4 = 0; k4 < 4; ++k4)
                    st[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(*reinterpret_cast<const h8 *>(&kv_lds[16 * j + c][32 * k4 + 8 * g]), qb[k4], st[j], 0, 0, 0);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    st[j][r] = 16 * j + 4 * g + r < cnt ? st[j][r] * p.scale_log2 : -INFINITY;
                    mx = fmaxf(mx, st[j][r]);
                }
            }
        }
        mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
#pragma unroll
        for (int j = 0; j < ATT_TW_MAX / 16; ++j)
            if (j < t_tiles) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    st[j][r] = exp2f(st[j][r] - mx);         // masked rows: exp2(-inf) = 0
                    sum += st[j][r];
                }
            }
        sum += __shfl_xor(sum, 16, 64);
        sum += __shfl_xor(sum, 32, 64);
    }
    __syncthreads();                                         // every wave has read K
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int kg = (tid >> 4) + 16 * i;
        if (4 * kg < tw32) {
            const int pos = vt_pos(4 * kg);
            const h8 v0 = __builtin_bit_cast(h8, vr[i][0]), v1 = __builtin_bit_cast(h8, vr[i][1]);
            const h8 v2 = __builtin_bit_cast(h8, vr[i][2]), v3 = __builtin_bit_cast(h8, vr[i][3]);
#pragma unroll
            for (int j = 0; j < 8; ++j) *reinterpret_cast<h4 *>(&kv_lds[ch * 8 + j][pos]) = h4{v0[j], v1[j], v2[j], v3[j]};
        }
    }
    __syncthreads();
    if (!live) return;
    f4 ot[8];                                                // O^T: element r of ot[dt] is dim 16 dt + 4 g + r, column (query) c
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) ot[dt] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int jj = 0; jj < ATT_TW_MAX / 32; ++jj)
        if (2 * jj < t_tiles) {
            h8 pb;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                pb[r] = (half_t)st[2 * jj][r];
                pb[4 + r] = (half_t)st[2 * jj + 1][r];
            }
#pragma unroll
            for (int dt = 0; dt < 8; ++dt)
                ot[dt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(*reinterpret_cast<const h8 *>(&kv_lds[16 * dt + c][32 * jj + 8 * g]), pb, ot[dt], 0, 0, 0);
        }
    const int qrow = qt * 16 + c;
    if (qrow >= p.Bq) return;
    const long base = ((long)split * p.Hkv + hk) * p.Bq + qrow;
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) *reinterpret_cast<f4 *>(p.part_o + base * ATT_D + 16 * dt + 4 * g) = ot[dt];
    if (g == 0) { p.part_ml[base * 2] = partial_max(mx, sum); p.part_ml[base * 2 + 1] = sum; }
}

// prefix_wgs: a multiple of 8, so that the others sit on the XCDs that attn_suffix_kernel's would
template <int PB>
__global__ __launch_bounds__(256, 4) void attn_parts_kernel(AttnParams p, int prefix_wgs, int rounds) {
    // (No args_ahead: a walk's first request needs two of the arguments' six lines, and waiting for all of them costs more than the later trips.  us a call with
    // the merge behind it, without and with: 64 heads over 8, 13 branches after 108 rows 12.1 and 12.6, 81 after 30 24.8 and 25.8; 32 heads, 40 after
    // 500 25.8 and 26.8.  The merge has it.)
    int L = blockIdx.x;
    if (L < prefix_wgs) {
        const DivMod head = uniform_divmod(L, p.Hkv), slice = uniform_divmod(head.q, rounds);
        if (slice.q < p.splits) attn_prefix_round(p, slice.q, head.r, slice.r);
        return;
    }
    L -= prefix_wgs;
    const int wave = threadIdx.x >> 6, nsub = p.suffix_waves, per_branch = (p.H * nsub + 3) >> 2, j = L >> 3, grp = uniform_divmod(j, per_branch).q, b = 8 * grp + (L & 7);
    if (b >= p.B) return;
    const int hq = (j - grp * per_branch) * 4 + wave, h = nsub == 4 ? hq >> 2 : (nsub == 2 ? hq >> 1 : hq);
    if (nsub == 1 && h >= p.H) return;
    attn_suffix_body<false, true, WALK_F16, PB>(p, b, min(h, p.H - 1), hq & (nsub - 1), nsub, h < p.H);
}

// One wave per query adds its splits + 1 partials up, in split order: lane d holds dims 2 d, 2 d + 1.  N partials are on their way at a time: what another XCD
// has just written takes ~2 us to come, so all of them are asked for at once where they are at most 17 (us a call, 64 branches after 1024 rows, nine partials,
// of which eight came in a first trip before, 44.3 and 43.0; 13 after 1740, 64 heads over 8, 23.4 and 21.2; one after 1011 14.4 and 11.5).
template <int N>
__global__ __launch_bounds__(256) void attn_merge_kernel(AttnParams p) {
    args_ahead<sizeof(AttnParams)>();
    const int qi = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;       // kv head * Bq + query of the kv head
    const int queries = p.Hkv * p.Bq;
    if (qi >= queries) return;
    float m = -INFINITY, l = 0.f;
    f2 o = {0.f, 0.f};
    for (int s0 = 0; s0 <= p.splits; s0 += N) {
        f2 v[N], ml[N];
#pragma unroll
        for (int i = 0; i < N; ++i) {                        // (past the last one: it again, which weighs nothing)
            const long base = (long)min(s0 + i, p.splits) * queries + qi;
            ml[i] = *reinterpret_cast<const f2 *>(p.part_ml + base * 2);
            v[i] = *reinterpret_cast<const f2 *>(p.part_o + base * ATT_D + 2 * lane);
        }
        float m_new = m;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            if (s0 + i > p.splits) {
                ml[i] = f2{-INFINITY, 0.f};
                v[i] = f2{0.f, 0.f};
            }
            m_new = fmaxf(m_new, ml[i][0]);
        }
        const float m_ref = m_new == -INFINITY ? 0.f : m_new, corr = exp2f(m - m_ref);       // (nothing yet: every factor is exp2(-inf) = 0)
        m = m_new;
        l *= corr;
        o[0] *= corr;
        o[1] *= corr;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const float c = exp2f(ml[i][0] - m_ref);
            l += ml[i][1] * c;
            o[0] += v[i][0] * c;
            o[1] += v[i][1] * c;
        }
    }
    const int hk = qi / p.Bq, qrow = qi - hk * p.Bq;
    const float inv = l > 0.f ? 1.0f / l : 0.f;
    half_t *op = p.out + ((long)div_rep(p, qrow) * p.H + hk * p.n_rep + mod_rep(p, qrow)) * ATT_D + 2 * lane;
    *reinterpret_cast<h2 *>(op) = h2{(half_t)(o[0] * inv), (half_t)(o[1] * inv)};
}

// ---- the whole decode attention in ONE launch -----------------------------------------------------------------
// grid (splits + ceil(Bq / per_wg), kv heads): workgroups x < splits take a slice of the prefix, the others the suffix
// + new token of per_wg = 1, 2 or 4 of the kv head's Bq = B x n_rep queries (4, 2 or 1 waves per query: with few
// queries a query's rows are spread over the waves, which shortens the longest chain of loads in the launch).  Every workgroup leaves partials with device-scope
// stores and counts itself in on the counters of the query tiles (16 queries of a kv head) it contributed to;
// the workgroup that completes a tile's count merges that tile's partials in split order (so the result does
// not depend on which workgroup that is), normalises and writes the output.  Nobody waits for anybody.
// FUSED: q and the new token's k, v come from the wq|wk|wv slabs (up to 16 branches); otherwise from p.q, p.cur_k/v.
constexpr int ATT_ONE_MAX_TILES = ATT_FUSED_MAX_Q / 16;

template <bool FUSED, int PB, int QKS = 16>
__global__ __launch_bounds__(256, 2) void attn_one_kernel(AttnParams p) {
    args_ahead<sizeof(AttnParams)>();
    __shared__ uint32_t s_last[ATT_ONE_MAX_TILES];
    const int hk = blockIdx.y;
    const int tid = threadIdx.x;
    const int q_tiles = (p.Bq + 15) / 16;
    const int sw_shift = p.suffix_waves == 4 ? 2 : (p.suffix_waves == 2 ? 1 : 0);
    const int per_wg = 4 >> sw_shift;          // queries of one suffix workgroup (suffix_waves = 1, 2 or 4 waves each)
    int tile_lo = 0, tile_hi = q_tiles - 1;    // query tiles this workgroup contributed to
    if ((int)blockIdx.x < p.splits) {
        attn_prefix_body<FUSED, true, ATT_ONE_TW, QKS>(p, blockIdx.x, hk);
    } else {
        const int j = (int)blockIdx.x - p.splits, wave_ = __builtin_amdgcn_readfirstlane(tid >> 6);
        const int qrow = per_wg * j + (wave_ >> sw_shift);        // query of this kv head: branch qrow / n_rep, its query head qrow % n_rep
        const int qc = min(qrow, p.Bq - 1);
        attn_suffix_body<FUSED, true, FUSED ? WALK_Q40 : WALK_ANY, PB, QKS>(p, div_rep(p, qc), hk * p.n_rep + mod_rep(p, qc), wave_ & (p.suffix_waves - 1), p.suffix_waves, qrow < p.Bq);
        tile_lo = tile_hi = (per_wg * j) / 16;  // a workgroup's 1, 2 or 4 consecutive queries never straddle a tile of 16
    }
    wait_vmem();                               // this wave's partials have reached memory ...
    __syncthreads();                           // ... and those of the whole workgroup
    if (tid < q_tiles) {
        uint32_t last = 0u;
        if (tid >= tile_lo && tid <= tile_hi) {
            // arrivals a tile waits for: every prefix slice + the suffix workgroups whose queries fall into it
            const int pw_shift = 2 - sw_shift;       // per_wg = 1 << pw_shift
            const int j_lo = (16 * tid) >> pw_shift, j_hi = (min(p.Bq, 16 * tid + 16) - 1) >> pw_shift;
            const uint32_t expected = (uint32_t)(p.splits + j_hi - j_lo + 1);
            uint32_t *cnt = p.counters + hk * q_tiles + tid;
            const uint32_t prev = __hip_atomic_fetch_add(cnt, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (prev == expected - 1u) {
                st_u32(cnt, 0u);               // ready for the next launch
                last = 1u;
            }
        }
        s_last[tid] = last;
    }
    __syncthreads();

    // ---- merge the completed tiles: 16 lanes per query (dims 4cc.. and 64+4cc..), 16 groups of 16 lanes ----
    // A tile of nq queries (npow = nq rounded up to a power of two) gives each query sub = 16 / npow consecutive
    // groups; group `si` of a query folds partials si, si + sub, ... (its loads go out together, four partials at
    // a time).  The groups of a query are then folded within their wave by lane exchange and across waves through
    // LDS.  The order depends only on the shape, not on which workgroup merges.
    __shared__ float s_merge[4][16][10];
    const int cc = tid & 15, gi = tid >> 4, wave = tid >> 6;
    const int n_part = p.splits + 1;
    for (int qt = tile_lo; qt <= tile_hi; ++qt) {
        if (s_last[qt] == 0u) continue;                       // (uniform over the workgroup)
        const int nq = min(16, p.Bq - 16 * qt);
        int npow = 1;
        while (npow < nq) npow <<= 1;
        const int sub = 16 / npow;
        const int qi = gi / sub, si = gi & (sub - 1);
        const int qrow = 16 * qt + qi;
        const bool live = qi < nq;
        float m = -INFINITY, l = 0.f;
        float o[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) o[j] = 0.f;
        auto fold = [&](float pm, float pl, const float (&po)[8]) {
            const float m_new = fmaxf(m, pm);
            if (m_new != -INFINITY) {
                const float c1 = exp2f(m - m_new), c2 = exp2f(pm - m_new);
                m = m_new;
                l = l * c1 + pl * c2;
#pragma unroll
                for (int j = 0; j < 8; ++j) o[j] = o[j] * c1 + po[j] * c2;
            }
        };
        for (int s0 = si; live && s0 < n_part; s0 += 4 * sub) {
            f4 lo[4], hi[4];
            float pm[4], pl[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                if (s0 + u * sub < n_part) {
                    const long base = ((long)(s0 + u * sub) * p.Hkv + hk) * p.Bq + qrow;
                    lo[u] = ld_f4(p.part_o + base * ATT_D + 4 * cc);
                    hi[u] = ld_f4(p.part_o + base * ATT_D + 64 + 4 * cc);
                    pm[u] = ld_f32(p.part_ml + base * 2);
                    pl[u] = ld_f32(p.part_ml + base * 2 + 1);
                }
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                if (s0 + u * sub < n_part) {
                    const float po[8] = {lo[u][0], lo[u][1], lo[u][2], lo[u][3], hi[u][0], hi[u][1], hi[u][2], hi[u][3]};
                    fold(pm[u], pl[u], po);
                }
            }
        }
        // groups of one wave (sub >= 2: neighbours, sub >= 4: all four); every lane of the wave takes part
        for (int sh = 16; sh <= 32 && sh < 16 * sub; sh <<= 1) {
            const float m2 = __shfl_xor(m, sh, 64), l2 = __shfl_xor(l, sh, 64);
            float o2[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) o2[j] = __shfl_xor(o[j], sh, 64);
            fold(m2, l2, o2);
        }
        if (sub > 4) {                                        // a query spans sub / 4 waves (uniform over the workgroup)
            if ((gi & 3) == 0) {
                float *mine = s_merge[wave][cc];
                mine[0] = m; mine[1] = l;
#pragma unroll
                for (int j = 0; j < 8; ++j) mine[2 + j] = o[j];
            }
            __syncthreads();
            if (si == 0 && live) {
                for (int k = 1; k < sub / 4; ++k) {
                    const float *other = s_merge[wave + k][cc];
                    const float po[8] = {other[2], other[3], other[4], other[5], other[6], other[7], other[8], other[9]};
                    fold(other[0], other[1], po);
                }
            }
            __syncthreads();                                  // s_merge is free for the next tile
        }
        if (si != 0 || !live) continue;
        const float inv = l > 0.f ? 1.0f / l : 0.f;
        const int b = div_rep(p, qrow), h = hk * p.n_rep + mod_rep(p, qrow);
        half_t *op = p.out + ((long)b * p.H + h) * ATT_D;
        *reinterpret_cast<h4 *>(op + 4 * cc) = h4{(half_t)(o[0] * inv), (half_t)(o[1] * inv), (half_t)(o[2] * inv), (half_t)(o[3] * inv)};
        *reinterpret_cast<h4 *>(op + 64 + 4 * cc) = h4{(half_t)(o[4] * inv), (half_t)(o[5] * inv), (half_t)(o[6] * inv), (half_t)(o[7] * inv)};
    }
}

// ---- a step's attention in one launch, 16 or 8 queries of a kv head a workgroup -------------------------------------
// (Of 16; of 8, a wave has one.)  Wave w of eight has queries 2 w and 2 w + 1 of the tile, one in either half of its lanes: it adds up their q, k and v
// from the slabs of wq|wk|wv, rotates, appends k and v, and walks the two branches' own rows.  In between all waves multiply the prefix for all 16 queries,
// 32 rows at a time (a wave takes every eighth such chunk), with K and V in registers as they come from memory; the waves' partials meet in LDS, so nothing
// but the output leaves the workgroup, and it waits for no other.
//   S^T = K . Q^T: element r of tile i is prefix row 16 i + 4 g + r of query c.  O^T = V^T . P^T in eight products: lane (c, g) holds dims
//   8 c .. + 7 of the eight rows whose probabilities it has, product e takes dims 8 c + e (a transpose of pairs of halves in registers), and
//   lane (c, g) ends with dims 32 g .. 32 g + 31 of query c.
// Workgroups of a kv head sit on one XCD (blockIdx.x), which then reads its prefix once, and neighbouring heads on the same one, which share
// the lines of the scales (heads dealt to two or four XCDs: 1 and 6 % slower).
// In place of the RoPE launch, the prefix slices and the walks (7B, 100 branches after 512 rows, 5 / 60 / 120 rows of their own: 26.0 / 34.1 /
// 42.8 us -> 13.7 / 24.2 / 35; 37 branches, 221 and 40 rows, 20.5 -> 14.0; 64 heads over 8, 50 branches after 2047 rows 40 -> 25; a step of 100
// branches 3.90 -> 3.58 ms, of 37 2.92 -> 2.77).  Which of them a layer takes: attn_way in model_layer.hip.
// Bound by the vector ALU: ~2000 instructions a wave and 110 a pass of four rows for two queries, at 4.4 cycles, two waves a SIMD; and, before
// that, by the compute unit's address unit and the latency of HBM (256 KB of K and V a workgroup: 5.5 us alone).
// (16 waves of one query each spill their registers: 20 us, where eight took 17.  Eight waves of two queries with a page table keep three in 16 bytes of
// scratch a lane.)
constexpr int AT_WAVES = 8, AT_CHUNK = 32;
constexpr int AT_PITCH = ATT_D + 4;                        // floats of a partial: o[128], maximum, sum
constexpr int AT_MINE = 16 * AT_PITCH;                     // floats of LDS of a wave: its partials, before that a chunk of K
constexpr int AT_QPITCH = ATT_D + 8;
constexpr int AT_LDS = AT_WAVES * AT_MINE * 4 + 3 * 16 * AT_QPITCH * 2;
static_assert(AT_MINE * 4 >= AT_CHUNK * 256 && AT_LDS <= 160 * 1024, "K fits");
typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t row16_max_bits(uint32_t v) {
    auto step = [&](auto ctrl) { v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, decltype(ctrl)::value, 0xf, 0xf, false)); };
    step(std::integral_constant<int, DPP_QUAD_XOR1>());
    step(std::integral_constant<int, DPP_QUAD_XOR2>());
    step(std::integral_constant<int, DPP_ROW_HALF_MIRROR>());
    step(std::integral_constant<int, DPP_ROW_ROR8>());
    return v;
}
// Half a row of 32 lanes: lane hl holds dims 4 hl .. + 3, its partner of the rotation is lane hl ^ 16 (roundings of rope_pair2)
__device__ __forceinline__ h4 rope_lanes(h4 x, h4 cs, h4 sn, bool lower) {
#pragma clang fp contract(off)
    const u32x2 mine = __builtin_bit_cast(u32x2, x);
    const h4 other = __builtin_bit_cast(h4, u32x2{(uint32_t)__shfl_xor((int)mine[0], 16, 64), (uint32_t)__shfl_xor((int)mine[1], 16, 64)});
    const h4 a = x * cs, b = (lower ? -other : other) * sn;
    return a + b;
}
// kv_store_row2 in that layout; `store`: the half's row is one to be written.  Both quotients are those of its divisions (corrected_quotient).  Scales
// that are zero, subnormal or not finite are left to the divisions.
__device__ __forceinline__ void kv_store_lanes(h4 x, uint8_t *row, half_t *scales, int hl, bool store) {
    const u32x2 bits = __builtin_bit_cast(u32x2, x) & 0x7fff7fffu;
    uint32_t big = max(max(bits[0] & 0xffffu, bits[0] >> 16), max(bits[1] & 0xffffu, bits[1] >> 16));
    big = row16_max_bits(big);
    const float top = (float)__builtin_bit_cast(half_t, (uint16_t)big);
    half_t s = (half_t)corrected_quotient(top, 7.0f, 1.0f / 7.0f);
    uint32_t codes = 0;
    const uint32_t exponent = __builtin_bit_cast(uint16_t, s) & 0x7c00u;
    if (__any(exponent == 0 || exponent == 0x7c00u)) {
        s = (half_t)(top / 7.0f);
#pragma unroll
        for (int j = 0; j < 4; ++j) codes |= (uint32_t)(kv_code2(x[j], (float)s) & 15) << (8 * j);
    } else {
        const float rcp = __builtin_amdgcn_rcpf((float)s);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const half_t q = __builtin_rintf16((half_t)corrected_quotient((float)x[j], (float)s, rcp));
            codes |= ((uint32_t)(int)(short)q & 15u) << (8 * j);
        }
    }
    const uint32_t upper = (uint32_t)__shfl_xor((int)codes, 16, 64);
    if (store && hl < 16) reinterpret_cast<uint32_t *>(row)[hl] = codes << 4 | upper;
    if (store && (hl & 15) == 0) scales[hl >> 4] = s;
}

// QKS: most slabs of the q|k|v product, LEAST: the fewest.  QT: queries of a workgroup, 16 or 8 (then a wave's halves share one query and take
// its rows 16 at a time in turn).  Grid: (XCD, kv head of it, tile); Ask = TileAsk: workgroups past the tiles ask for the next launch's weights (q40_warm.hpp).
// (A kernel of its own: with the arguments and the branch in every launch calls that ask for nothing took 0.2 to 0.4 us longer, 32 heads, 17 branches behind 256 rows
// without rows of their own 8.04 us and 7.65 so; 64 over 8 7.63 and 7.36.)
struct TileAsk {
    int tiles;
    WarmWeights next;
};
template <bool PAGES, int LEAST, int QKS, int QT, class... Ask>
__global__ __launch_bounds__(64 * AT_WAVES) void attn_tile_kernel(AttnParams p, int chunks, Ask... ask) {
    args_ahead<sizeof(AttnParams) + (sizeof...(Ask) > 0 ? 16 : 4)>();
    if constexpr (sizeof...(Ask) > 0) {
        const TileAsk &a = (ask, ...);
        if (__builtin_expect((int)blockIdx.z >= a.tiles, 0)) return warm_weights(a.next, blockIdx.x, (blockIdx.z - a.tiles) * gridDim.y + blockIdx.y, threadIdx.x, 64 * AT_WAVES);
    }
    extern __shared__ __attribute__((aligned(16))) float at_lds[];
    half_t *const s_q = reinterpret_cast<half_t *>(at_lds + AT_WAVES * AT_MINE), *const s_k = s_q + 16 * AT_QPITCH, *const s_v = s_k + 16 * AT_QPITCH;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int hk = blockIdx.x * gridDim.y + blockIdx.y, tile = blockIdx.z;
    if (hk >= p.Hkv) return;
    const int c = lane & 15, g = lane >> 4;                  // of the matrix products
    const int hl = lane & 31, half = lane >> 5, qi = QT == 16 ? 2 * wave + half : wave;      // this half's lane and query
    const int e = lane & 7, rs = (lane >> 3) & 3;            // of the walk: eight lanes a row, dims 8 e .. and 64 + 8 e ..; four rows a half
    const int qrow = QT * tile + qi, qc = min(qrow, p.Bq - 1);
    const int b = div_rep(p, qc), rep = mod_rep(p, qc), h = hk * p.n_rep + rep;
    const bool live = qrow < p.Bq && (QT == 16 || half == 0);
    auto meet = [] { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };

    // ---- requests: slabs, rotation factors, page ids, prefix ----
    const int pos = *p.pos_dev, t = *p.app_t, len = min(max(t, 0), (int)p.suffix_batch_stride_rows);
    const int cols = (p.H + 2 * p.Hkv) * ATT_D;
    const long slab = (long)p.B * cols;
    const float *src = p.qkv + (long)b * cols + 4 * hl;
    // (QT == 8: k in the lower half of the lanes, v in the upper one)
    f4 qv[QKS], kv[QKS], vv[QT == 16 ? QKS : 1];
    auto slabs = [&](int col, f4 (&v)[QKS]) {
#pragma unroll
        for (int s = 0; s < QKS; ++s) v[s] = *reinterpret_cast<const f4 *>(src + (col + (s < LEAST ? s : min(s, p.qkv_ks - 1)) * slab));
    };
    slabs(h * ATT_D, qv);
    slabs((p.H + hk + (QT == 8 && half == 1 ? p.Hkv : 0)) * ATT_D, kv);
    if constexpr (QT == 16) slabs((p.H + p.Hkv + hk) * ATT_D, vv);
    const h4 cs = *reinterpret_cast<const h4 *>(p.cos_tab + (long)pos * 64 + 4 * (hl & 15));
    const h4 sn = *reinterpret_cast<const h4 *>(p.sin_tab + (long)pos * 64 + 4 * (hl & 15));
    // a wave's turns of its walk: QT == 16: 16 rows of either half's query, 8: 32 of the one, 16 a half.  Four passes of four rows a half.
    constexpr int TURN = QT == 16 ? 16 : 32;
    const int turns = (len + TURN - 1) / TURN;
    auto row_at = [&](int s, int u) { return QT == 16 ? 16 * s + 4 * u + rs : 32 * s + 16 * half + 4 * u + rs; };
    const int32_t *ids = reinterpret_cast<const int32_t *>(p.pages) + (long)b * p.pages_stride;
    auto ids_of = [&](int blk) { return ids[min(32 * blk + hl, len - 1)]; };           // of 32 positions, one a lane
    int id_now = 0, id_next = 0;
    if (PAGES && len > 0) {
        id_now = ids_of(0);
        if (len > 32) id_next = ids_of(1);
    }

    // This wave's chunks are kind, kind + 8, ..: the waves of different tiles begin at different ones (where they begin at the same, all wait for the
    // same lines to come from HBM: 16.1 us instead of 14.3 at 100 branches after 512 rows), and every tile does the same sums in the same order.
    const int kind = (wave + (int)(__brev((uint32_t)tile) >> 29)) & (AT_WAVES - 1);
    char *const s_mine = reinterpret_cast<char *>(at_lds + kind * AT_MINE);
    const uint32_t pfx_row = (uint32_t)p.pfx_row_stride * 2;
    const char *kb = reinterpret_cast<const char *>(p.prefix_k + (long)hk * p.pfx_head_stride), *vb = reinterpret_cast<const char *>(p.prefix_v + (long)hk * p.pfx_head_stride);
    const uint32_t k_off = g * pfx_row + 16 * c, v_off = 4 * g * pfx_row + 16 * c;
    // whole rows a load (one whose neighbouring lanes are in different rows takes 64 cycles, not 16): K's row 4 i + g, V's 4 g + i, from 16 on for i >= 4
    struct Chunk { u32x4 k[8], v[8]; };
    auto fetch = [&](int j, Chunk &ck) {
        if (AT_CHUNK * (j + 1) <= p.P) {
            const long at = (long)(AT_CHUNK * j) * pfx_row;
#pragma unroll
            for (int i = 0; i < 8; ++i) ck.k[i] = *reinterpret_cast<const u32x4 *>(kb + at + (long)(4 * i) * pfx_row + k_off);
#pragma unroll
            for (int i = 0; i < 8; ++i) ck.v[i] = *reinterpret_cast<const u32x4 *>(vb + at + (long)(i < 4 ? i : 12 + i) * pfx_row + v_off);
        } else {                                             // past the end: the last row again, which weighs nothing
#pragma unroll
            for (int i = 0; i < 8; ++i) ck.k[i] = *reinterpret_cast<const u32x4 *>(kb + ((uint32_t)min(AT_CHUNK * j + 4 * i + g, p.P - 1) * pfx_row + 16 * c));
#pragma unroll
            for (int i = 0; i < 8; ++i)
                ck.v[i] = *reinterpret_cast<const u32x4 *>(vb + ((uint32_t)min(AT_CHUNK * j + (i < 4 ? i : 12 + i) + 4 * g, p.P - 1) * pfx_row + 16 * c));
        }
    };
    Chunk ck[2];
    __builtin_amdgcn_sched_barrier(0);                       // (loads are waited for in their order: what the query needs comes first)
    if (QKS <= 6 && kind < chunks) fetch(kind, ck[0]);

    // ---- this branch's rows: a turn's four a request.  Half the lanes of a row have its K scales, half its V scales ----
    struct Rows { u32x2 k[4], v[4]; uint32_t sc[4]; };
    const char *sc_base = reinterpret_cast<const char *>(e < 4 ? p.suffix_ks : p.suffix_vs);
    auto row_of = [&](int id) { return (uint32_t)min(max(id, 0), (int)p.pool_rows - 1) * (uint32_t)p.Hkv + hk; };
    uint32_t row_now = PAGES ? 0u : (uint32_t)(b * (int)p.suffix_batch_stride_rows) * (uint32_t)p.Hkv + hk;
    auto rows = [&](int s, Rows &r) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            // (past the end: the last row again)
            const uint32_t row = PAGES ? (uint32_t)__shfl((int)row_now, (lane & 32) | (row_at(s, u) & 31), 64)
                                       : row_now + (uint32_t)min(row_at(s, u), len - 1) * (uint32_t)p.Hkv;
            r.k[u] = *reinterpret_cast<const u32x2 *>((const char *)p.suffix_k + (row * 64 + 8 * e));
            r.v[u] = *reinterpret_cast<const u32x2 *>((const char *)p.suffix_v + (row * 64 + 8 * e));
            r.sc[u] = *reinterpret_cast<const uint32_t *>(sc_base + (unsigned long)row * 4);
        }
    };
    Rows cur;

    // ---- q, k, v ----
    {
        auto total = [&](const f4 (&v)[QKS]) {
            f4 tot = v[0];
#pragma unroll
            for (int s = 1; s < QKS; ++s) {
                const f4 next = tot + v[s];
                tot = s < LEAST || s < p.qkv_ks ? next : tot;
            }
            return h4{(half_t)tot[0], (half_t)tot[1], (half_t)tot[2], (half_t)tot[3]};
        };
        const bool lower = hl < 16;
        const h4 q = rope_lanes(total(qv), cs, sn, lower), raw = total(kv), k = rope_lanes(raw, cs, sn, lower);
        h4 v = raw;
        if constexpr (QT == 16) v = total(vv);
        *reinterpret_cast<h4 *>(s_q + qi * AT_QPITCH + 4 * hl) = q;
        if constexpr (QT == 16) {
            *reinterpret_cast<h4 *>(s_k + qi * AT_QPITCH + 4 * hl) = k;
            *reinterpret_cast<h4 *>(s_v + qi * AT_QPITCH + 4 * hl) = v;
        } else {
            *reinterpret_cast<h4 *>((half == 0 ? s_k : s_v) + qi * AT_QPITCH + 4 * hl) = half == 0 ? k : v;
        }
        if (len > 0) {
            if (PAGES) row_now = row_of(id_now);
            rows(0, cur);
        }
        if (QKS > 6 && kind < chunks) fetch(kind, ck[0]);
        meet();                                              // every query is in LDS
        if (kind + AT_WAVES < chunks) fetch(kind + AT_WAVES, ck[1]);
        if (t >= 0 && t < p.app_smax) {                      // (uniform) the first query head of a kv head appends the rows
            const long row = ((long)b * p.app_smax + t) * p.Hkv + hk;
            const bool store = qrow < p.Bq && rep == 0;
            if constexpr (QT == 16) {
                kv_store_lanes(k, p.app_k + row * 64, p.app_ks + row * 2, hl, store);
                kv_store_lanes(v, p.app_v + row * 64, p.app_vs + row * 2, hl, store);
            } else {
                kv_store_lanes(half == 0 ? k : v, (half == 0 ? p.app_k : p.app_v) + row * 64, (half == 0 ? p.app_ks : p.app_vs) + row * 2, hl, store);
            }
        }
    }

    // ---- the prefix, two chunks at a time ----
    if (kind < chunks) {
        f4 o[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) o[i] = f4{0.f, 0.f, 0.f, 0.f};
        float m = -INFINITY, l = 0.f;                        // m: of query c, in all its lanes; l: over this lane's rows
        auto scores = [&](int j, Chunk &ch, f4 *st) {
            // K to the operand's layout through this wave's part of LDS: piece k of row r lies at k ^ (r % 16)
#pragma unroll
            for (int i = 0; i < 8; ++i) *reinterpret_cast<u32x4 *>(s_mine + (4 * i + g) * 256 + 16 * (c ^ ((4 * i + g) & 15))) = ch.k[i];
#pragma unroll
            for (int k4 = 0; k4 < 4; ++k4) {
                const h8 qb = *reinterpret_cast<const h8 *>(s_q + (c & (QT - 1)) * AT_QPITCH + 32 * k4 + 8 * g);
#pragma unroll
                for (int i = 0; i < 2; ++i)
                    st[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(*reinterpret_cast<const h8 *>(s_mine + (16 * i + c) * 256 + 16 * ((4 * k4 + g) ^ c)), qb, st[i], 0, 0, 0);
            }
            if (AT_CHUNK * (j + 1) > p.P) {                  // (uniform) the last chunk
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    if (AT_CHUNK * j + (i < 4 ? i : 12 + i) + 4 * g >= p.P) {
                        st[i >> 2][i & 3] = -INFINITY;
                        ch.v[i] = u32x4{0, 0, 0, 0};
                    }
            }
        };
        // Probabilities are 2^15 times themselves (the partial's maximum says so) and enter the product as two fp16 terms, 22 bits of them.  The first is
        // cut, not rounded, and the second at least 2^-24 (2^-39 of the largest probability): both have a probability's sign, and where V is
        // infinite the sum is, not infinity less infinity or times zero.  A NaN stays in the first.  (Error against 64 bits as with a rounded first
        // term, to seven digits: 2.08e-4 at 100 branches after 512 rows, all of it the output's fp16.)
        struct Terms { h8 p, left; };
        auto products = [&](const Chunk &ch, const Terms &pb) {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                u32x4 va;
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    va[k] = (i & 1) == 0 ? pack_lo16(ch.v[2 * k][i >> 1], ch.v[2 * k + 1][i >> 1]) : pack_hi16(ch.v[2 * k][i >> 1], ch.v[2 * k + 1][i >> 1]);
                o[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, va), pb.p, o[i], 0, 0, 0);
                o[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, va), pb.left, o[i], 0, 0, 0);
            }
        };
        for (int j = kind; j < chunks; j += 2 * AT_WAVES) {
            const bool two = j + AT_WAVES < chunks;          // (uniform)
            f4 st[4] = {f4{0.f, 0.f, 0.f, 0.f}, f4{0.f, 0.f, 0.f, 0.f}, f4{0.f, 0.f, 0.f, 0.f}, f4{0.f, 0.f, 0.f, 0.f}};
            scores(j, ck[0], st);
            if (two) scores(j + AT_WAVES, ck[1], st + 2);
            float mx = fmaxf(fmaxf(fmaxf(st[0][0], st[0][1]), fmaxf(st[0][2], st[0][3])), fmaxf(fmaxf(st[1][0], st[1][1]), fmaxf(st[1][2], st[1][3])));
            if (two) mx = fmaxf(mx, fmaxf(fmaxf(fmaxf(st[2][0], st[2][1]), fmaxf(st[2][2], st[2][3])), fmaxf(fmaxf(st[3][0], st[3][1]), fmaxf(st[3][2], st[3][3]))));
            mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
            mx = fmaxf(mx, __shfl_xor(mx, 32, 64)) * p.scale_log2;
            if (j != kind) {                                 // (uniform)
                const float m_new = fmaxf(m, mx), corr = __builtin_amdgcn_exp2f(m - (m_new == -INFINITY ? 0.f : m_new));
                l *= corr;
#pragma unroll
                for (int i = 0; i < 8; ++i)
#pragma unroll
                    for (int r = 0; r < 4; ++r) o[i][r] *= corr;
                mx = m_new;
            }
            m = mx;
            const float m_ref = (m == -INFINITY ? 0.f : m) - 15.f;
            auto probabilities = [&](const f4 *s4) {
                u32x4 cut, left;
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    float pr[2];
#pragma unroll
                    for (int i = 0; i < 2; ++i) {
                        pr[i] = __builtin_amdgcn_exp2f(__builtin_fmaf(s4[k >> 1][2 * (k & 1) + i], p.scale_log2, -m_ref));
                        l += pr[i];
                    }
                    const h2 first = __builtin_bit_cast(h2, __builtin_amdgcn_cvt_pkrtz(pr[0], pr[1]));
                    const h2 second = {(half_t)(pr[0] - (float)first.x), (half_t)(pr[1] - (float)first.y)};
                    cut[k] = as_u32(first);
                    left[k] = __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(u16x2, second), u16x2{1, 1}));
                }
                return Terms{__builtin_bit_cast(h8, cut), __builtin_bit_cast(h8, left)};
            };
            products(ck[0], probabilities(st));
            if (two) products(ck[1], probabilities(st + 2));
            if (j + 2 * AT_WAVES < chunks) fetch(j + 2 * AT_WAVES, ck[0]);
            if (j + 3 * AT_WAVES < chunks) fetch(j + 3 * AT_WAVES, ck[1]);
        }
        l += __shfl_xor(l, 16, 64);
        l += __shfl_xor(l, 32, 64);
        float *po = reinterpret_cast<float *>(s_mine) + c * AT_PITCH;
        if (c < QT) {
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int i = 0; i < 2; ++i) *reinterpret_cast<f4 *>(po + 32 * g + 8 * r + 4 * i) = f4{o[4 * i][r], o[4 * i + 1][r], o[4 * i + 2][r], o[4 * i + 3][r]};
            if (g == 0) *reinterpret_cast<f2 *>(po + ATT_D) = f2{m - 15.f, l};
        }
    }

    // ---- the branch's own rows: m, l of this lane's row slot, o of its dims: as RowRegs orders them, first 8 e .., 64 + 8 e .., then 8 e + 4 .., 68 + 8 e .. ----
    RowRegs q[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) q[j] = row_from_fp16(s_q + qi * AT_QPITCH, 2 * e + j);
    float m, l, o[2][8];
    auto score = [&](const RowRegs &k0, const RowRegs &k1) {
        float d = 0.f;
        const RowRegs *kr[2] = {&k0, &k1};
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            d = __builtin_amdgcn_fdot2(kr[j]->a02, q[j].a02, d, false);
            d = __builtin_amdgcn_fdot2(kr[j]->a13, q[j].a13, d, false);
            d = __builtin_amdgcn_fdot2(kr[j]->b02, q[j].b02, d, false);
            d = __builtin_amdgcn_fdot2(kr[j]->b13, q[j].b13, d, false);
        }
        d += dpp_move<DPP_QUAD_XOR1>(d);
        d += dpp_move<DPP_QUAD_XOR2>(d);
        d += dpp_move<DPP_ROW_HALF_MIRROR>(d);
        return d * p.scale_log2;
    };
    auto add = [&](float pr, int j, const RowRegs &v) {
        o[j][0] += pr * (float)v.a02.x; o[j][1] += pr * (float)v.a02.y;
        o[j][2] += pr * (float)v.a13.x; o[j][3] += pr * (float)v.a13.y;
        o[j][4] += pr * (float)v.b02.x; o[j][5] += pr * (float)v.b02.y;
        o[j][6] += pr * (float)v.b13.x; o[j][7] += pr * (float)v.b13.y;
    };
    // the state relative to another maximum; returned: what to subtract from scores
    auto raise = [&](float m_new) {
        const float m_ref = m_new == -INFINITY ? 0.f : m_new, corr = __builtin_amdgcn_exp2f(m - m_ref);
        m = m_new;
        l *= corr;
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int k = 0; k < 8; ++k) o[j][k] *= corr;
        return m_ref;
    };
    {
        // the new token's exact row begins slot 0 (in the others an infinite value would weigh 0, and 0 times it is NaN)
        const bool mine = rs == 0 && (QT == 16 || half == 0);
        const float sc = score(row_from_fp16(s_k + qi * AT_QPITCH, 2 * e), row_from_fp16(s_k + qi * AT_QPITCH, 2 * e + 1));
        m = mine ? fmaxf(sc, -INFINITY) : -INFINITY;
        const float pr = __builtin_amdgcn_exp2f(sc - (m == -INFINITY ? 0.f : m));
        l = 0.f;
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int k = 0; k < 8; ++k) o[j][k] = 0.f;
        if (mine) {
            l = pr;
#pragma unroll
            for (int j = 0; j < 2; ++j) add(pr, j, row_from_fp16(s_v + qi * AT_QPITCH, 2 * e + j));
        }
    }
    const RowCodes codes;
    // N passes from u0 on: one maximum, one rescale.  ends: some may lie past the last row
    auto passes = [&](int s, auto N, int u0, bool ends) {
        float sc[N];
        uint32_t vs[N];
        float mx = m;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const uint32_t mine = cur.sc[u0 + i], other = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)mine, DPP_ROW_HALF_MIRROR, 0xf, 0xf, false);
            const uint32_t ks = e < 4 ? mine : other;
            vs[i] = e < 4 ? other : mine;
            sc[i] = score(row_from_q40(cur.k[u0 + i][0], ks, codes), row_from_q40(cur.k[u0 + i][1], ks, codes));
            if (ends && row_at(s, u0 + i) >= len) sc[i] = -INFINITY;
            mx = fmaxf(mx, sc[i]);
        }
        const float m_ref = raise(mx);
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const float pr = __builtin_amdgcn_exp2f(sc[i] - m_ref);
            l += pr;
#pragma unroll
            for (int j = 0; j < 2; ++j) add(pr, j, row_from_q40(cur.v[u0 + i][j], vs[i], codes));
        }
    };
    for (int s = 0; s < turns; ++s) {
        Rows nxt;
        if (s + 1 < turns) {
            const int blk = TURN * (s + 1) / 32;
            if (PAGES && TURN * (s + 1) % 32 == 0) {
                row_now = row_of(id_next);
                if (32 * (blk + 1) < len) id_next = ids_of(blk + 1);
            }
            rows(s + 1, nxt);
        }
        if (TURN * (s + 1) <= len) {                         // (uniform)
            passes(s, std::integral_constant<int, 4>(), 0, false);
        } else {
            passes(s, std::integral_constant<int, 2>(), 0, true);
            if (QT == 8 || TURN * s + 8 < len) passes(s, std::integral_constant<int, 2>(), 2, true);
        }
        cur = nxt;
    }
    meet();                                                  // the prefix's partials are in LDS
    {
        constexpr int N = AT_WAVES / 4 * QT / 16;            // of this slot
        f4 part[N][2][2];
        f2 ml[N];
        float mx = m;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const int sp = QT == 16 ? rs + 4 * i : 4 * half + rs;
            ml[i] = f2{-INFINITY, 0.f};
#pragma unroll
            for (int j = 0; j < 2; ++j) part[i][j][0] = part[i][j][1] = f4{0.f, 0.f, 0.f, 0.f};
            if (sp < chunks) {
                const float *po = at_lds + sp * AT_MINE + qi * AT_PITCH;
                ml[i] = *reinterpret_cast<const f2 *>(po + ATT_D);
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    part[i][j][0] = *reinterpret_cast<const f4 *>(po + 8 * e + 4 * j);
                    part[i][j][1] = *reinterpret_cast<const f4 *>(po + 64 + 8 * e + 4 * j);
                }
            }
            mx = fmaxf(mx, ml[i][0]);
        }
        // ... and the maximum of the slots of the query
        mx = fmaxf(mx, dpp_move<DPP_ROW_ROR8>(mx));
        mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
        if (QT == 8) mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        const float m_ref = raise(mx);
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const float f = __builtin_amdgcn_exp2f(ml[i][0] - m_ref);
            l += f * ml[i][1];
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int k = 0; k < 4; ++k) {                // (RowRegs order: dims 0, 2, 1, 3)
                    o[j][k] += f * part[i][j][0][(k & 1) * 2 + (k >> 1)];
                    o[j][4 + k] += f * part[i][j][1][(k & 1) * 2 + (k >> 1)];
                }
        }
    }
    // ---- the slots added up: slot (second, first bit) ends with dims 64 second + 8 e + 4 first .. + 3 ----
    l += dpp_move<DPP_ROW_ROR8>(l);
    l += __shfl_xor(l, 16, 64);
    if (QT == 8) l += __shfl_xor(l, 32, 64);
    const int first = rs & 1, second = rs >> 1;
    float w[8], y[4];
#pragma unroll
    for (int k = 0; k < 8; ++k) w[k] = (first ? o[1][k] : o[0][k]) + dpp_move<DPP_ROW_ROR8>(first ? o[0][k] : o[1][k]);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        y[k] = (second ? w[4 + k] : w[k]) + __shfl_xor(second ? w[k] : w[4 + k], 16, 64);
        if (QT == 8) y[k] += __shfl_xor(y[k], 32, 64);
    }
    if (!live) return;
    const float inv = l > 0.f ? 1.0f / l : 0.f;
    *reinterpret_cast<h4 *>(p.out + ((long)b * p.H + h) * ATT_D + 64 * second + 8 * e + 4 * first) =
        h4{(half_t)(y[0] * inv), (half_t)(y[2] * inv), (half_t)(y[1] * inv), (half_t)(y[3] * inv)};
}

static int attn_plan_tw(int P, int Hkv) {
    // rows of the prefix per workgroup: as large as fits while still giving the 256 CUs work
    int tw = ATT_TW_MAX;
    while (tw > 32 && (long)((P + tw - 1) / tw) * Hkv < 256) tw >>= 1;
    return tw;
}

// The one-launch kernel fed by the q|k|v product.  From 32 kv heads on slices of ATT_ONE_TW rows, also where narrower ones would give each compute unit one: what
// they leave to the merge, and the second wave of a query's own rows that they take the place of, cost more (us a step of the 7B architecture, slices of 32 rows and of
// 64, 10 / 60 / 120 rows of their own: 5 branches behind 100 rows 1905 / 1913 / 1938 and 1892 / 1896 / 1916; 16 behind 256 2072 / 2116 / 2168 and 2010 / 2026 / 2088; 10
// behind 400 2085 / 2188 / 2347 and 1986 / 1999 / 2066; us a call of 32 / 40 / 64 heads, slices as narrow and of 64 rows, 10 rows of their own: one branch behind 128 rows 10.1
// / 10.1 / 10.6 and 9.9 / 9.8 / 10.2, four behind 256 11.1 / 11.1 / 12.0 and 10.1 / 10.5 / 12.0, 16 behind 128 12.7 / 12.7 / 13.6 and 11.9 / 11.8 / 12.4; 384 sizes of 4 to 16 branches, 10 to 120 own
// rows, with the waves below: 1.08 times as fast at the mean, slowest 0.97, 64 heads of 12 branches behind 96 rows, 11.3 and 11.7 at 10 own rows, 19.9 and 14.2 at 120;
// 64 and 80 heads over 32 and 40, 1 to 8 branches: 0.97 .. 1.7.)  One query keeps three slices of 32 rows
// behind 96: 9.2 and 9.7 us with two.  Below 96 rows results stay what they were (ATTN_TILES_MIN_PROMPT).
// (smh_shared_prefix_attn_one, whose queries are ready and whose slices end sooner, keeps the narrow ones: with wide ones 0.91 .. 0.97 times as fast
// at 1 to 5 branches behind 96 and 128 rows, 32 and 40 heads, 1.0 .. 1.9 behind 256 and more.)
static bool attn_wide_slices(int P, int Hkv, int queries) { return Hkv >= 32 && P >= (queries > 1 ? 96 : 97) && attn_plan_tw(P, Hkv) < ATT_ONE_TW; }
static int attn_plan_one_tw(int P, int Hkv, int queries) { return attn_wide_slices(P, Hkv, queries) ? ATT_ONE_TW : min(attn_plan_tw(P, Hkv), ATT_ONE_TW); }

// Two launches: rows of the prefix per workgroup and the number of workgroups that share one slice's query tiles.
// Every slice leaves a partial per query, so wide slices mean less partial traffic; the CUs are filled first by
// dealing the rounds of query tiles (four tiles, one per wave) of a slice to several workgroups, which re-read the
// slice from the cache but write nothing extra, and only then by narrower slices.
static void attn_plan(int P, int Hkv, int Bq, int *tw_out, int *qgroups_out) {
    const int rounds = ((Bq + 15) / 16 + 3) / 4;
    constexpr int wgs_least = 256;
    int tw = ATT_TW_MAX, qg = 1;
    while ((long)((P + tw - 1) / tw) * Hkv * qg < wgs_least) {
        if (qg < rounds) qg = min(rounds, 2 * qg);
        else if (tw > 32) tw >>= 1;
        else break;
    }
    *tw_out = tw;
    *qgroups_out = qg;
}

// Suffix launch of the two-launch form: waves per (branch, query head) - more than one while the launch still fits
// the GPU in one round (4 waves of this kernel per SIMD, 1024 SIMDs).
static int attn_plan_suffix_waves_two(long queries) {
    int nsub = 4;
    constexpr int cap = 4096;                  // measured again with the 8-lanes-a-row walk: 2048 and 8192 are both slower
    while (nsub > 1 && queries * nsub > cap) nsub >>= 1;
    return nsub;
}

// One-launch kernel: waves that share a query's suffix rows - as many as keep the launch within one round of
// workgroups (two fit a compute unit).  wide (attn_wide_slices): four only where they leave a sixteenth of the round free.  A launch that four waves fill costs
// more than two waves' longer walks (us a call, 10 / 30 / 60 / 120 own rows, two waves and four: 32 heads, 12 branches behind 200 rows 12.1 / 12.3 / 12.9 / 14.0 and
// 13.5 / 13.7 / 13.8 / 14.5, 14 behind 128 11.7 / 11.8 / 12.4 / 13.4 and 12.9 / 13.1 / 13.3 / 14.3; 64 heads, 6 behind 96 10.3 / 10.4 / 11.0 / 12.7 and 11.3 /
// 11.5 / 11.6 / 12.0); two waves where one would do may fill it (64 heads, 12 behind 96, one and two: 11.1 / 11.9 / 14.0 / 18.3 and 11.7 / 11.8 / 12.4 / 14.2).
static int attn_plan_suffix_waves(int splits, int Bq, int Hkv, bool wide) {
    int nsub = 4;
    while (nsub > 1 && (long)(splits + (Bq + 4 / nsub - 1) / (4 / nsub)) * Hkv > (wide && nsub == 4 ? 479 : 512)) nsub >>= 1;
    return nsub;
}

}  // namespace smh

// Partials and marks of attn_page_tile_kernel for pages_cols positions, 0 where the pass does not pay or apply.
static size_t attn_tiles_bytes(int B, int H, int Hkv, int cols) {
    const size_t slices = (size_t)(cols + smh::PT_TW - 1) / smh::PT_TW, tiles = ((size_t)B * (H / Hkv) + 15) / 16;
    if (B < 2 || slices > smh::PT_MAX_SLICES || tiles > 65535) return 0;
    return slices * B * H * (smh::ATT_D + 2) * sizeof(float) + slices * tiles * Hkv;
}

extern "C" size_t smh_attn_workspace_bytes(int B, int H, int P) {
    if (P <= 0 || B <= 0 || H <= 0) return 256;
    size_t splits = (size_t)(P + 31) / 32 + 1;      // worst case: 32 rows per workgroup; the suffix's partial
    return splits * (size_t)B * (size_t)H * (smh::ATT_D + 2) * sizeof(float) + 256;
}

extern "C" size_t smh_paged_attn_workspace_bytes(int B, int H, int Hkv, int P, int pages_cols) {
    const size_t least = smh_attn_workspace_bytes(B, H, P);
    if (P > 0 || B <= 0 || H <= 0 || Hkv <= 0 || H % Hkv != 0 || pages_cols <= 0) return least;
    const size_t tiles = attn_tiles_bytes(B, H, Hkv, pages_cols);
    return tiles > least ? tiles : least;
}

constexpr size_t ATT_COUNTER_BYTES = 4096;     // one-launch variants: arrival counters at the start of the workspace

// what the paged entry point adds to the arguments of smh_shared_prefix_attn (zero strides: token-major tensors)
struct AttnExtras {
    const void *pages = nullptr;
    long pages_stride = 0;
    int page_bytes = 4;
    long pool_rows = 0;
    long pfx_row = 0, pfx_head = 0, sfx_row = 0, sfx_head = 0;
};

static int shared_prefix_attn(const char *who, bool one, const void *q, void *out, int B, int H, int Hkv, int D,
                              const void *prefix_k, const void *prefix_v, int P,
                              int suffix_format, const void *suffix_k, const void *suffix_v,
                              const void *suffix_ks, const void *suffix_vs, int Smax,
                              const int32_t *lens, int lens_stride, const void *cur_k, const void *cur_v,
                              void *workspace, size_t workspace_bytes, smh_stream_t stream, const AttnExtras &ex = AttnExtras()) {
    using namespace smh;
    SMH_REQUIRE(D == ATT_D, "%s: head dim %d (only 128)", who, D);
    SMH_REQUIRE(B >= 0 && B <= 65535 && H > 0 && Hkv > 0 && H % Hkv == 0 && P >= 0, "%s: B=%d (at most 65535) H=%d Hkv=%d P=%d", who, B, H, Hkv, P);
    SMH_REQUIRE(suffix_format == SMH_KV_NONE || suffix_format == SMH_KV_FP16 || suffix_format == SMH_KV_Q40,
                "%s: suffix_format=%d", who, suffix_format);
    if (B == 0) return 0;
    SMH_REQUIRE(q && out, "%s: null q/out", who);
    SMH_REQUIRE(P == 0 || (prefix_k && prefix_v), "%s: null prefix", who);
    if (suffix_format != SMH_KV_NONE) {
        SMH_REQUIRE(suffix_k && suffix_v && (lens || ex.pages) && Smax > 0 && (lens_stride == 0 || lens_stride == 1),
                    "%s: suffix arguments incomplete", who);
        SMH_REQUIRE(suffix_format != SMH_KV_Q40 || (suffix_ks && suffix_vs), "%s: null suffix scales", who);
    }
    SMH_REQUIRE((cur_k == nullptr) == (cur_v == nullptr), "%s: cur_k/cur_v must both be given or both be null", who);
    AttnParams p{};
    p.q = (const half_t *)q; p.out = (half_t *)out;
    p.prefix_k = (const half_t *)prefix_k; p.prefix_v = (const half_t *)prefix_v;
    p.suffix_k = suffix_k; p.suffix_v = suffix_v;
    p.suffix_ks = (const half_t *)suffix_ks; p.suffix_vs = (const half_t *)suffix_vs;
    p.lens = lens; p.lens_stride = lens_stride;
    p.cur_k = (const half_t *)cur_k; p.cur_v = (const half_t *)cur_v;
    p.suffix_batch_stride_rows = Smax;
    p.pages = ex.pages; p.pages_stride = ex.pages_stride; p.page_bytes = ex.page_bytes; p.pool_rows = ex.pool_rows;
    p.pfx_row_stride = ex.pfx_row ? ex.pfx_row : (long)Hkv * ATT_D; p.pfx_head_stride = ex.pfx_head ? ex.pfx_head : ATT_D;
    p.sfx_row_stride = ex.sfx_row ? ex.sfx_row : (long)Hkv * ATT_D; p.sfx_head_stride = ex.sfx_head ? ex.sfx_head : ATT_D;
    p.B = B; p.H = H; p.Hkv = Hkv; p.n_rep = H / Hkv; p.Bq = B * p.n_rep;
    p.P = P; p.suffix_format = suffix_format;
    p.scale_log2 = LOG2E / sqrtf((float)D);
    int qgroups = 1;
    if (one) p.tw = min(attn_plan_tw(P, Hkv), ATT_ONE_TW);
    else attn_plan(P, Hkv, p.Bq, &p.tw, &qgroups);
    p.splits = P > 0 ? (P + p.tw - 1) / p.tw : 0;
    if (one) {
        p.suffix_waves = attn_plan_suffix_waves(p.splits, p.Bq, Hkv, false);
        const int q_tiles = (p.Bq + 15) / 16;
        SMH_REQUIRE(q_tiles <= ATT_ONE_MAX_TILES && (size_t)Hkv * q_tiles * sizeof(uint32_t) <= ATT_COUNTER_BYTES,
                    "%s: %d queries per kv head (at most %d), %d kv heads", who, p.Bq, ATT_FUSED_MAX_Q, Hkv);
        size_t n_part = (size_t)(p.splits + 1) * Hkv * p.Bq;
        size_t need = ATT_COUNTER_BYTES + n_part * (ATT_D + 2) * sizeof(float);
        SMH_REQUIRE(workspace && workspace_bytes >= need, "%s: workspace %zu < %zu bytes", who, workspace_bytes, need);
        p.counters = (uint32_t *)workspace;
        p.part_o = (float *)((char *)workspace + ATT_COUNTER_BYTES);
        p.part_ml = p.part_o + n_part * ATT_D;
        hipLaunchKernelGGL((attn_one_kernel<false, PB_ANY>), dim3(p.splits + (p.Bq + 4 / p.suffix_waves - 1) / (4 / p.suffix_waves), Hkv), dim3(256), 0, (hipStream_t)stream, p);
        return launch_status();
    }
    size_t n_part = (size_t)p.splits * Hkv * p.Bq;
    SMH_REQUIRE(p.splits == 0 || (workspace && workspace_bytes >= n_part * (ATT_D + 2) * sizeof(float)),
                "%s: workspace %zu < %zu bytes", who, workspace_bytes, n_part * (ATT_D + 2) * sizeof(float));
    p.part_o = (float *)workspace;
    p.part_ml = p.part_o + n_part * ATT_D;
    p.suffix_waves = attn_plan_suffix_waves_two((long)B * H);
    const unsigned wgs = (unsigned)(((H * p.suffix_waves + 3) / 4) * ((B + 7) / 8 * 8));
    const int pb = p.pages == nullptr ? 0 : p.page_bytes;
    const size_t n_parts = (size_t)(p.splits + 1) * Hkv * p.Bq;
    const int rounds = ((p.Bq + 15) / 16 + 3) / 4;
    const long prefix_wgs = ((long)p.splits * Hkv * rounds + 7) / 8 * 8;
    if (p.splits > 0 && suffix_format == SMH_KV_FP16 && workspace_bytes >= n_parts * (ATT_D + 2) * sizeof(float) && prefix_wgs + wgs < (1L << 31)) {
        p.part_ml = p.part_o + n_parts * ATT_D;
        const dim3 grid((unsigned)(prefix_wgs + wgs));
        const auto parts = pb == 0 ? attn_parts_kernel<0> : pb == 2 ? attn_parts_kernel<2> : pb == 4 ? attn_parts_kernel<4> : attn_parts_kernel<8>;
        hipLaunchKernelGGL(parts, grid, dim3(256), 0, (hipStream_t)stream, p, (int)prefix_wgs, rounds);
        const auto merge = p.splits < 5 ? attn_merge_kernel<5> : p.splits < 9 ? attn_merge_kernel<9> : attn_merge_kernel<17>;
        hipLaunchKernelGGL(merge, dim3((unsigned)(((long)Hkv * p.Bq + 3) / 4)), dim3(256), 0, (hipStream_t)stream, p);
        return launch_status();
    }
    if (p.splits > 0)
        hipLaunchKernelGGL(attn_prefix_kernel<false>, dim3(p.splits, Hkv, qgroups), dim3(256), 0, (hipStream_t)stream, p);
    const bool fp16_pages = p.pages != nullptr && suffix_format == SMH_KV_FP16;
    const size_t tile_bytes = fp16_pages && P == 0 && lens == nullptr ? attn_tiles_bytes(B, H, Hkv, Smax) : 0;
    if (tile_bytes > 0 && workspace && workspace_bytes >= tile_bytes) {
        const int tiles = (p.Bq + 15) / 16;
        p.splits = (Smax + PT_TW - 1) / PT_TW;
        n_part = (size_t)p.splits * Hkv * p.Bq;
        p.part_ml = p.part_o + n_part * ATT_D;
        p.tile_done = (uint8_t *)(p.part_ml + n_part * 2);
        const int each = (long)Hkv * p.splits * tiles > PT_ROUND ? 2 : 1;
        const auto one = pb == 2 ? attn_page_tile_kernel<2, 1> : pb == 4 ? attn_page_tile_kernel<4, 1> : attn_page_tile_kernel<8, 1>;
        const auto two = pb == 2 ? attn_page_tile_kernel<2, 2> : pb == 4 ? attn_page_tile_kernel<4, 2> : attn_page_tile_kernel<8, 2>;
        const auto walk = pb == 2 ? attn_suffix_kernel<false, WALK_TILES, 2> : pb == 4 ? attn_suffix_kernel<false, WALK_TILES, 4> : attn_suffix_kernel<false, WALK_TILES, 8>;
        hipLaunchKernelGGL(each == 2 ? two : one, dim3(Hkv, (tiles + each - 1) / each, p.splits), dim3(256), 0, (hipStream_t)stream, p);
        hipLaunchKernelGGL(walk, dim3(wgs), dim3(256), 0, (hipStream_t)stream, p);
        return launch_status();
    }
    const auto f16 = pb == 0 ? attn_suffix_kernel<false, WALK_F16, 0> : pb == 2 ? attn_suffix_kernel<false, WALK_F16, 2>
                     : pb == 4 ? attn_suffix_kernel<false, WALK_F16, 4> : attn_suffix_kernel<false, WALK_F16, 8>;
    const auto q40 = pb == 0 ? attn_suffix_kernel<false, WALK_Q40, 0> : pb == 2 ? attn_suffix_kernel<false, WALK_Q40, 2>
                     : pb == 4 ? attn_suffix_kernel<false, WALK_Q40, 4> : attn_suffix_kernel<false, WALK_Q40, 8>;
    hipLaunchKernelGGL(suffix_format == SMH_KV_FP16 ? f16 : q40, dim3(wgs), dim3(256), 0, (hipStream_t)stream, p);
    return launch_status();
}

extern "C" int smh_shared_prefix_attn(const void *q, void *out, int B, int H, int Hkv, int D,
                                      const void *prefix_k, const void *prefix_v, int P,
                                      int suffix_format, const void *suffix_k, const void *suffix_v,
                                      const void *suffix_ks, const void *suffix_vs, int Smax,
                                      const int32_t *lens, int lens_stride, const void *cur_k, const void *cur_v,
                                      void *workspace, size_t workspace_bytes, smh_stream_t stream) {
    return shared_prefix_attn("smh_shared_prefix_attn", false, q, out, B, H, Hkv, D, prefix_k, prefix_v, P, suffix_format, suffix_k,
                              suffix_v, suffix_ks, suffix_vs, Smax, lens, lens_stride, cur_k, cur_v, workspace, workspace_bytes, stream);
}

extern "C" int smh_paged_prefix_attn(const void *q, void *out, int B, int H, int Hkv, int D,
                                     const void *prefix_k, const void *prefix_v, int P, long prefix_row_stride, long prefix_head_stride,
                                     int pool_format, const void *pool_k, const void *pool_v, const void *pool_ks, const void *pool_vs,
                                     long pool_row_stride, long pool_head_stride, long pool_rows,
                                     const void *pages, int page_bytes, long pages_stride, int pages_cols, const int32_t *lens, int lens_stride,
                                     const void *cur_k, const void *cur_v, int single_launch,
                                     void *workspace, size_t workspace_bytes, smh_stream_t stream) {
    using namespace smh;
    const char *who = "smh_paged_prefix_attn";
    SMH_REQUIRE(pages_cols >= 1 && pages_cols <= pages_stride, "%s: pages_cols=%d must lie in 1 .. pages_stride=%ld", who, pages_cols, pages_stride);
    SMH_REQUIRE(pool_format == SMH_KV_FP16 || pool_format == SMH_KV_Q40, "%s: pool_format=%d", who, pool_format);
    SMH_REQUIRE(pages != nullptr && (page_bytes == 2 || page_bytes == 4 || page_bytes == 8) && pages_stride >= 1,
                "%s: pages=%p page_bytes=%d (2, 4 or 8) pages_stride=%ld", who, pages, page_bytes, pages_stride);
    SMH_REQUIRE(pages_stride <= 0x7fffffffL, "%s: pages_stride=%ld", who, pages_stride);
    SMH_REQUIRE(pool_rows >= 1, "%s: pool_rows=%ld", who, pool_rows);
    SMH_REQUIRE(prefix_row_stride >= 0 && prefix_head_stride >= 0 && pool_row_stride >= 0 && pool_head_stride >= 0 &&
                prefix_row_stride % 8 == 0 && prefix_head_stride % 8 == 0 && pool_row_stride % 4 == 0 && pool_head_stride % 4 == 0,
                "%s: strides must be non-negative (0 = token-major), prefix strides multiples of 8 and pool strides multiples of 4 elements", who);
    SMH_REQUIRE(pool_format != SMH_KV_Q40 || (pool_row_stride == 0 && pool_head_stride == 0), "%s: Q4_0 pools are token-major (strides 0)", who);
    AttnExtras ex;
    ex.pages = pages; ex.page_bytes = page_bytes; ex.pages_stride = pages_stride; ex.pool_rows = pool_rows;
    ex.pfx_row = prefix_row_stride; ex.pfx_head = prefix_head_stride; ex.sfx_row = pool_row_stride; ex.sfx_head = pool_head_stride;
    // (the kernels cut lens[b] to the row count they are given: the ids a table row holds, not the distance between rows)
    return shared_prefix_attn(who, single_launch != 0, q, out, B, H, Hkv, D, prefix_k, prefix_v, P, pool_format, pool_k, pool_v, pool_ks, pool_vs,
                              pages_cols, lens, lens_stride, cur_k, cur_v, workspace, workspace_bytes, stream, ex);
}

// copies entries 0 .. n - 1 of row `origin` of a page table [rows, stride] to rows curr .. curr + forks - 1
__global__ __launch_bounds__(256) void page_fork_kernel(int32_t *table, long stride, int origin, int curr, int n) {
    const int32_t *src = table + (long)origin * stride;
    int32_t *dst = table + (long)(curr + blockIdx.y) * stride;
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) dst[i] = src[i];
}

extern "C" int smh_page_fork(int32_t *table, int rows, long stride, int origin, int curr, int forks, int n, smh_stream_t stream) {
    SMH_REQUIRE(table && rows > 0 && stride > 0 && n >= 0 && n <= stride, "smh_page_fork: table=%p rows=%d stride=%ld n=%d", (void *)table, rows, stride, n);
    SMH_REQUIRE(origin >= 0 && origin < rows && forks >= 0 && curr >= 0 && curr + forks <= rows && forks <= 65535,
                "smh_page_fork: origin=%d curr=%d forks=%d outside the table's %d rows", origin, curr, forks, rows);
    SMH_REQUIRE(origin < curr || origin >= curr + forks, "smh_page_fork: the origin row lies inside the rows it is copied to");
    if (forks == 0 || n == 0) return 0;
    hipLaunchKernelGGL(page_fork_kernel, dim3((unsigned)((n + 255) / 256), (unsigned)forks), dim3(256), 0, (hipStream_t)stream, table, stride, origin, curr, n);
    return smh::launch_status();
}

// ---- the same attention for callers that cannot allocate ---------------------------------------------------------
// The prefix partials of smh_shared_prefix_attn_static live in this array instead of a caller's workspace.  Every GPU
// the library runs on holds its own copy at its own address for the life of the process; host code never uses the
// array's name as an address, only what hipGetSymbolAddress returned for the current device.
// ATT_STATIC_SCRATCH_BYTES limits the partials of the prefix slices; behind them the array has room for the suffixes' partials (as many
// bytes as one slice's, so never more than the slices' together), so that a call takes the same launches as with a workspace of
// smh_attn_workspace_bytes and returns the same bits.
constexpr size_t ATT_STATIC_SCRATCH_BYTES = (size_t)16 << 20;
static __device__ __align__(256) unsigned char scratch[2 * ATT_STATIC_SCRATCH_BYTES];
constexpr int ATT_STATIC_MAX_DEVICES = 64;
static std::mutex g_scratch_mutex;
static void *g_scratch_ptr[ATT_STATIC_MAX_DEVICES] = {};

// Device address of `scratch` on the current device, looked up once per device.
static int static_scratch(void **ptr_out) {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) { smh::set_error("smh_shared_prefix_attn_static: hipGetDevice: %s", hipGetErrorString(e)); return (int)e; }
    if (dev < 0 || dev >= ATT_STATIC_MAX_DEVICES) { smh::set_error("smh_shared_prefix_attn_static: device %d outside [0,%d)", dev, ATT_STATIC_MAX_DEVICES); return -1; }
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (g_scratch_ptr[dev] == nullptr) {
        void *ptr = nullptr;
        e = hipGetSymbolAddress((void **)&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || ptr == nullptr) {
            smh::set_error("smh_shared_prefix_attn_static: hipGetSymbolAddress: %s", hipGetErrorString(e));
            return e != hipSuccess ? (int)e : -1;
        }
        g_scratch_ptr[dev] = ptr;
    }
    *ptr_out = g_scratch_ptr[dev];
    return 0;
}

extern "C" size_t smh_attn_static_scratch_bytes(void) { return ATT_STATIC_SCRATCH_BYTES; }

extern "C" int smh_shared_prefix_attn_static(const void *q, void *out, int B, int H, int Hkv, int D,
                                             const void *prefix_k, const void *prefix_v, int P,
                                             int suffix_format, const void *suffix_k, const void *suffix_v,
                                             const void *suffix_ks, const void *suffix_vs, int Smax,
                                             const int32_t *lens, int lens_stride, const void *cur_k, const void *cur_v,
                                             smh_stream_t stream) {
    using namespace smh;
    const char *who = "smh_shared_prefix_attn_static";
    // (every argument check comes before the scratch array's address is asked for: a refused call does not touch the device)
    SMH_REQUIRE(D == ATT_D, "%s: head dim %d (only 128)", who, D);
    SMH_REQUIRE(B >= 0 && B <= 65535 && H > 0 && Hkv > 0 && H % Hkv == 0 && P >= 0, "%s: B=%d (at most 65535) H=%d Hkv=%d P=%d", who, B, H, Hkv, P);
    // the partials the two launches exchange: one (max, sum, o[128]) per prefix slice and query, as smh_shared_prefix_attn plans them
    int tw = ATT_TW_MAX, qgroups = 1;
    attn_plan(P, Hkv, B * (H / Hkv), &tw, &qgroups);
    const size_t splits = P > 0 ? (size_t)(P + tw - 1) / tw : 0;
    const size_t need = splits * (size_t)B * H * (ATT_D + 2) * sizeof(float);
    SMH_REQUIRE(need <= ATT_STATIC_SCRATCH_BYTES, "%s: B=%d H=%d P=%d needs %zu bytes of scratch, the static array holds %zu (use smh_shared_prefix_attn with a workspace)",
                who, B, H, P, need, ATT_STATIC_SCRATCH_BYTES);
    SMH_REQUIRE(B == 0 || (q && out), "%s: null q/out", who);
    SMH_REQUIRE(P == 0 || (prefix_k && prefix_v), "%s: null prefix", who);
    SMH_REQUIRE(suffix_format == SMH_KV_NONE || (suffix_k && suffix_v && lens && Smax > 0), "%s: suffix arguments incomplete", who);
    if (B == 0) return 0;
    void *ws = nullptr;
    const int st = static_scratch(&ws);
    if (st) return st;
    return shared_prefix_attn(who, false, q, out, B, H, Hkv, D, prefix_k, prefix_v, P, suffix_format, suffix_k, suffix_v, suffix_ks, suffix_vs,
                              Smax, lens, lens_stride, cur_k, cur_v, ws, sizeof(scratch), stream);
}

extern "C" int smh_shared_prefix_attn_one(const void *q, void *out, int B, int H, int Hkv, int D,
                                          const void *prefix_k, const void *prefix_v, int P,
                                          int suffix_format, const void *suffix_k, const void *suffix_v,
                                          const void *suffix_ks, const void *suffix_vs, int Smax,
                                          const int32_t *lens, int lens_stride, const void *cur_k, const void *cur_v,
                                          void *workspace, size_t workspace_bytes, smh_stream_t stream) {
    return shared_prefix_attn("smh_shared_prefix_attn_one", true, q, out, B, H, Hkv, D, prefix_k, prefix_v, P, suffix_format, suffix_k,
                              suffix_v, suffix_ks, suffix_vs, Smax, lens, lens_stride, cur_k, cur_v, workspace, workspace_bytes, stream);
}


extern "C" size_t smh_attn_qkv_workspace_bytes(int B, int H, int P) {
    if (B <= 0 || H <= 0) return ATT_COUNTER_BYTES + 256;
    size_t splits = (size_t)(P > 0 ? (P + 31) / 32 : 0) + 1;      // worst case: 32 rows per workgroup; + the suffix partial
    return ATT_COUNTER_BYTES + splits * (size_t)B * (size_t)H * (smh::ATT_D + 2) * sizeof(float) + 256;
}

extern "C" int smh_shared_prefix_attn_qkv(const void *qkv_partial, int ksplit, void *out, int B, int H, int Hkv, int D,
                                          const void *cos_tab, const void *sin_tab, const int32_t *pos_dev,
                                          const void *prefix_k, const void *prefix_v, int P,
                                          void *cache_k, void *cache_ks, void *cache_v, void *cache_vs, int Smax,
                                          const int32_t *t_dev, const int32_t *pages, int pages_stride, int single_launch,
                                          void *workspace, size_t workspace_bytes, smh_stream_t stream) {
    using namespace smh;
    const char *who = "smh_shared_prefix_attn_qkv";
    SMH_REQUIRE(pages == nullptr || pages_stride >= Smax, "%s: pages_stride=%d must cover the %d rows of a branch", who, pages_stride, Smax);
    SMH_REQUIRE(D == ATT_D, "%s: head dim %d (only 128)", who, D);
    SMH_REQUIRE(B >= 0 && B <= 16 && H > 0 && Hkv > 0 && H % Hkv == 0 && P >= 0, "%s: B=%d (at most 16) H=%d Hkv=%d P=%d", who, B, H, Hkv, P);
    SMH_REQUIRE(ksplit >= 1 && ksplit <= 16, "%s: ksplit=%d", who, ksplit);
    SMH_REQUIRE(B * (H / Hkv) <= ATT_FUSED_MAX_Q, "%s: %d queries per kv head (at most %d)", who, B * (H / Hkv), ATT_FUSED_MAX_Q);
    if (B == 0) return 0;
    SMH_REQUIRE(qkv_partial && out && cos_tab && sin_tab && pos_dev, "%s: null pointer", who);
    SMH_REQUIRE(P == 0 || (prefix_k && prefix_v), "%s: null prefix", who);
    SMH_REQUIRE(cache_k && cache_ks && cache_v && cache_vs && t_dev && Smax > 0, "%s: the suffix cache and its row counter are required", who);
    AttnParams p{};
    p.out = (half_t *)out;
    p.prefix_k = (const half_t *)prefix_k; p.prefix_v = (const half_t *)prefix_v;
    p.suffix_k = cache_k; p.suffix_v = cache_v;
    p.suffix_ks = (const half_t *)cache_ks; p.suffix_vs = (const half_t *)cache_vs;
    p.lens = t_dev; p.lens_stride = 0;
    p.suffix_batch_stride_rows = Smax;
    p.pages = pages; p.pages_stride = pages_stride; p.page_bytes = 4; p.pool_rows = (long)B * Smax;   // a branch reads its own rows and its ancestors', all below B
    p.pfx_row_stride = (long)Hkv * ATT_D; p.pfx_head_stride = ATT_D;
    p.sfx_row_stride = (long)Hkv * ATT_D; p.sfx_head_stride = ATT_D;
    p.B = B; p.H = H; p.Hkv = Hkv; p.n_rep = H / Hkv; p.Bq = B * p.n_rep;
    p.P = P; p.suffix_format = SMH_KV_Q40;
    p.scale_log2 = LOG2E / sqrtf((float)D);
    int qgroups = 1;
    if (single_launch) p.tw = attn_plan_one_tw(P, Hkv, p.Bq);
    else attn_plan(P, Hkv, p.Bq, &p.tw, &qgroups);
    p.splits = P > 0 ? (P + p.tw - 1) / p.tw : 0;
    p.qkv = (const float *)qkv_partial; p.qkv_ks = ksplit;
    p.cos_tab = (const half_t *)cos_tab; p.sin_tab = (const half_t *)sin_tab; p.pos_dev = pos_dev;
    p.app_k = (uint8_t *)cache_k; p.app_v = (uint8_t *)cache_v;
    p.app_ks = (half_t *)cache_ks; p.app_vs = (half_t *)cache_vs;
    p.app_t = t_dev; p.app_smax = Smax;
    if (single_launch) {
        p.suffix_waves = attn_plan_suffix_waves(p.splits, p.Bq, Hkv, attn_wide_slices(P, Hkv, p.Bq));
        // workspace = [arrival counters | partials of splits + 1 passes]
        SMH_REQUIRE((size_t)Hkv * ((p.Bq + 15) / 16) * sizeof(uint32_t) <= ATT_COUNTER_BYTES, "%s: %d kv heads x %d query tiles", who, Hkv, (p.Bq + 15) / 16);
        size_t n_part = (size_t)(p.splits + 1) * Hkv * p.Bq;
        size_t need = ATT_COUNTER_BYTES + n_part * (ATT_D + 2) * sizeof(float);
        SMH_REQUIRE(workspace && workspace_bytes >= need, "%s: workspace %zu < %zu bytes", who, workspace_bytes, need);
        p.counters = (uint32_t *)workspace;
        p.part_o = (float *)((char *)workspace + ATT_COUNTER_BYTES);
        p.part_ml = p.part_o + n_part * ATT_D;
        const auto kern = ksplit <= 2    ? (pages != nullptr ? attn_one_kernel<true, 4, 2> : attn_one_kernel<true, 0, 2>)
                          : ksplit <= 8  ? (pages != nullptr ? attn_one_kernel<true, 4, 8> : attn_one_kernel<true, 0, 8>)
                          : ksplit <= 12 ? (pages != nullptr ? attn_one_kernel<true, 4, 12> : attn_one_kernel<true, 0, 12>)
                                         : (pages != nullptr ? attn_one_kernel<true, 4, 16> : attn_one_kernel<true, 0, 16>);
        hipLaunchKernelGGL(kern, dim3(p.splits + (p.Bq + 4 / p.suffix_waves - 1) / (4 / p.suffix_waves), Hkv), dim3(256), 0, (hipStream_t)stream, p);
        return launch_status();
    }
    size_t n_part = (size_t)p.splits * Hkv * p.Bq;
    SMH_REQUIRE(p.splits == 0 || (workspace && workspace_bytes >= n_part * (ATT_D + 2) * sizeof(float)),
                "%s: workspace %zu < %zu bytes", who, workspace_bytes, n_part * (ATT_D + 2) * sizeof(float));
    p.part_o = (float *)workspace;
    p.part_ml = p.part_o + n_part * ATT_D;
    if (p.splits > 0)
        hipLaunchKernelGGL(attn_prefix_kernel<true>, dim3(p.splits, Hkv, qgroups), dim3(256), 0, (hipStream_t)stream, p);
    p.suffix_waves = attn_plan_suffix_waves_two((long)B * H);
    hipLaunchKernelGGL((pages != nullptr ? attn_suffix_kernel<true, WALK_Q40, 4> : attn_suffix_kernel<true, WALK_Q40, 0>), dim3((unsigned)(((H * p.suffix_waves + 3) / 4) * ((B + 7) / 8 * 8))), dim3(256), 0, (hipStream_t)stream, p);
    return launch_status();
}

int smh::shared_prefix_attn_qkv_tiles(const void *qkv_partial, int ksplit, void *out, int B, int H, int Hkv, int D, const void *cos_tab, const void *sin_tab,
                                      const int32_t *pos_dev, const void *prefix_k, const void *prefix_v, int P, void *cache_k, void *cache_ks, void *cache_v,
                                      void *cache_vs, int Smax, const int32_t *t_dev, const int32_t *pages, int pages_stride, long cache_rows,
                                      const smh::WarmWeights &next, smh_stream_t stream) {
    using namespace smh;
    const char *who = "smh_shared_prefix_attn_qkv_tiles";
    SMH_REQUIRE(D == ATT_D, "%s: head dim %d (only 128)", who, D);
    SMH_REQUIRE(B >= 0 && B <= 65535 && H > 0 && Hkv > 0 && H % Hkv == 0 && P >= 0, "%s: B=%d (at most 65535) H=%d Hkv=%d P=%d", who, B, H, Hkv, P);
    SMH_REQUIRE(ksplit >= 1 && ksplit <= 16, "%s: ksplit=%d", who, ksplit);
    if (B == 0) return 0;
    SMH_REQUIRE(qkv_partial && out && cos_tab && sin_tab && pos_dev, "%s: null pointer", who);
    SMH_REQUIRE(P == 0 || (prefix_k && prefix_v), "%s: null prefix", who);
    SMH_REQUIRE(cache_k && cache_ks && cache_v && cache_vs && t_dev && Smax > 0, "%s: the suffix cache and its row counter are required", who);
    SMH_REQUIRE(pages == nullptr || (pages_stride >= Smax && cache_rows >= 1), "%s: pages_stride=%d must cover the %d rows of a branch, cache_rows=%ld", who,
                pages_stride, Smax, cache_rows);
    const char *const why = attn_tiles_refuse({qkv_partial, out, cos_tab, sin_tab, prefix_k, prefix_v, cache_k, cache_ks, cache_v, cache_vs, B, H, Hkv, P,
                                               pages != nullptr ? cache_rows : (long)B * Smax});
    SMH_REQUIRE(why == nullptr, "%s: %s", who, why);
    AttnParams p{};
    p.out = (half_t *)out;
    p.prefix_k = (const half_t *)prefix_k; p.prefix_v = (const half_t *)prefix_v;
    p.suffix_k = cache_k; p.suffix_v = cache_v;
    p.suffix_ks = (const half_t *)cache_ks; p.suffix_vs = (const half_t *)cache_vs;
    p.lens = t_dev; p.lens_stride = 0;
    p.suffix_batch_stride_rows = Smax;
    p.pages = pages; p.pages_stride = pages_stride; p.page_bytes = 4; p.pool_rows = cache_rows;
    p.pfx_row_stride = (long)Hkv * ATT_D; p.pfx_head_stride = ATT_D;
    p.sfx_row_stride = (long)Hkv * ATT_D; p.sfx_head_stride = ATT_D;
    p.B = B; p.H = H; p.Hkv = Hkv; p.n_rep = H / Hkv; p.Bq = B * p.n_rep;
    p.P = P; p.suffix_format = SMH_KV_Q40;
    p.scale_log2 = LOG2E / sqrtf((float)D);
    p.qkv = (const float *)qkv_partial; p.qkv_ks = ksplit;
    p.cos_tab = (const half_t *)cos_tab; p.sin_tab = (const half_t *)sin_tab; p.pos_dev = pos_dev;
    p.app_k = (uint8_t *)cache_k; p.app_v = (uint8_t *)cache_v;
    p.app_ks = (half_t *)cache_ks; p.app_vs = (half_t *)cache_vs;
    p.app_t = t_dev; p.app_smax = Smax;
#define TILE_KERNELS(...) {{{attn_tile_kernel<false, 1, 2, 8 __VA_ARGS__>, attn_tile_kernel<false, 3, 6, 8 __VA_ARGS__>, attn_tile_kernel<false, 7, 16, 8 __VA_ARGS__>}, \
                            {attn_tile_kernel<true, 1, 2, 8 __VA_ARGS__>, attn_tile_kernel<true, 3, 6, 8 __VA_ARGS__>, attn_tile_kernel<true, 7, 16, 8 __VA_ARGS__>}}, \
                           {{attn_tile_kernel<false, 1, 2, 16 __VA_ARGS__>, attn_tile_kernel<false, 3, 6, 16 __VA_ARGS__>, attn_tile_kernel<false, 7, 16, 16 __VA_ARGS__>}, \
                            {attn_tile_kernel<true, 1, 2, 16 __VA_ARGS__>, attn_tile_kernel<true, 3, 6, 16 __VA_ARGS__>, attn_tile_kernel<true, 7, 16, 16 __VA_ARGS__>}}}
    typedef void (*plain_t)(AttnParams, int);
    typedef void (*ask_t)(AttnParams, int, TileAsk);
    static const plain_t plain[2][2][3] = TILE_KERNELS();
    static const ask_t asking[2][2][3] = TILE_KERNELS(, TileAsk);
#undef TILE_KERNELS
    static const hipError_t lds_ok = [] {
        hipError_t e = hipSuccess;
        for (int i = 0; i < 12 && e == hipSuccess; ++i) {
            e = hipFuncSetAttribute((const void *)plain[i / 6][i / 3 % 2][i % 3], hipFuncAttributeMaxDynamicSharedMemorySize, AT_LDS);
            if (e == hipSuccess) e = hipFuncSetAttribute((const void *)asking[i / 6][i / 3 % 2][i % 3], hipFuncAttributeMaxDynamicSharedMemorySize, AT_LDS);
        }
        return e;
    }();
    if (lds_ok != hipSuccess) { set_error("%s: the kernel's LDS could not be reserved: %s", who, hipGetErrorString(lds_ok)); return (int)lds_ok; }
    const int qt = attn_tile_queries(p.Bq, Hkv), tiles = (p.Bq + qt - 1) / qt, rows = (Hkv + 7) / 8, slabs = ksplit <= 2 ? 0 : ksplit <= 6 ? 1 : 2;
    const int chunks = (P + AT_CHUNK - 1) / AT_CHUNK;
    const dim3 grid(8, rows, tiles + next.workgroups / (8 * rows)), threads(64 * AT_WAVES);
    if (next.workgroups >= 8 * rows) hipLaunchKernelGGL(asking[qt == 16][pages != nullptr][slabs], grid, threads, AT_LDS, (hipStream_t)stream, p, chunks, TileAsk{tiles, next});
    else hipLaunchKernelGGL(plain[qt == 16][pages != nullptr][slabs], grid, threads, AT_LDS, (hipStream_t)stream, p, chunks);
    return launch_status();
}
int smh::attn_tiles_idle(int B, int H, int Hkv) {
    const long queries = (long)B * (H / Hkv), qt = attn_tile_queries(queries, Hkv), row = (Hkv + 7) / 8 * 8, tiles = (queries + qt - 1) / qt;
    return row * tiles < 256 ? (int)((256 - row * tiles) / row * row) : 0;
}
extern "C" int smh_shared_prefix_attn_qkv_tiles(const void *qkv_partial, int ksplit, void *out, int B, int H, int Hkv, int D,
                                                const void *cos_tab, const void *sin_tab, const int32_t *pos_dev,
                                                const void *prefix_k, const void *prefix_v, int P,
                                                void *cache_k, void *cache_ks, void *cache_v, void *cache_vs, int Smax,
                                                const int32_t *t_dev, const int32_t *pages, int pages_stride, long cache_rows, smh_stream_t stream) {
    return smh::shared_prefix_attn_qkv_tiles(qkv_partial, ksplit, out, B, H, Hkv, D, cos_tab, sin_tab, pos_dev, prefix_k, prefix_v, P, cache_k, cache_ks, cache_v,
                                             cache_vs, Smax, t_dev, pages, pages_stride, cache_rows, smh::WarmWeights{}, stream);
}

// Causal prefill attention: query s attends to rows 0..s of the same K/V tensors.
extern "C" int smh_prefill_attn(const void *q, const void *k, const void *v, void *out, int S, int H, int Hkv,
                                int D, smh_stream_t stream) {
    using namespace smh;
    SMH_REQUIRE(D == ATT_D, "smh_prefill_attn: head dim %d (only 128)", D);
    SMH_REQUIRE(S >= 0 && H > 0 && Hkv > 0 && H % Hkv == 0, "smh_prefill_attn: S=%d H=%d Hkv=%d", S, H, Hkv);
    if (S == 0) return 0;
    SMH_REQUIRE(q && k && v && out, "smh_prefill_attn: null pointer");
    PrefillParams p;
    p.q = (const half_t *)q; p.k = (const half_t *)k; p.v = (const half_t *)v; p.out = (half_t *)out;
    p.S = S; p.H = H; p.Hkv = Hkv; p.n_rep = H / Hkv;
    p.scale_log2 = LOG2E / sqrtf((float)D);
    // four query groups (128 queries) a workgroup share a staged tile; two where that would leave compute units without a workgroup
    const long blocks4 = (long)((S + 127) / 128) * H, blocks2 = (long)((S + 63) / 64) * H;
    SMH_REQUIRE(blocks2 < (1L << 31) && Hkv <= 65536, "smh_prefill_attn: S=%d H=%d Hkv=%d (at most 65536: a pair of tiles spans 31 bits)", S, H, Hkv);
    static const hipError_t lds_ok = [] {
        const hipError_t e = hipFuncSetAttribute((const void *)attn_prefill_kernel<4>, hipFuncAttributeMaxDynamicSharedMemorySize, PF_LDS);
        return e != hipSuccess ? e : hipFuncSetAttribute((const void *)attn_prefill_kernel<2>, hipFuncAttributeMaxDynamicSharedMemorySize, PF_LDS);
    }();
    if (lds_ok != hipSuccess) { set_error("smh_prefill_attn: the kernel's LDS could not be reserved: %s", hipGetErrorString(lds_ok)); return (int)lds_ok; }
    if (blocks4 >= 256) hipLaunchKernelGGL(attn_prefill_kernel<4>, dim3((unsigned)blocks4), dim3(512), PF_LDS, (hipStream_t)stream, p);
    else hipLaunchKernelGGL(attn_prefill_kernel<2>, dim3((unsigned)blocks2), dim3(256), PF_LDS, (hipStream_t)stream, p);
    return launch_status();
}
