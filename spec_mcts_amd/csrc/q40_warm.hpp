// The weights that a launch of q40_gemm_kg_kernel or q40_gemm_swiglu_kernel (17 .. 128 rows, in layer calls 5 .. 128) will read first, asked for by workgroups of the
// launch in front of it.
//
// A workgroup of q40_gemm_kg_kernel or q40_gemm_swiglu_kernel waits ~2.5 us for its first stage (cold translations and HBM), a quarter of a launch at 37
// rows, and HBM idles meanwhile, as it does under the RMSNorm (a workgroup a row) and the attention.  Those launches, and SwiGLU's on 172 compute units, get
// `workgroups` more workgroups, which load one dword of every 128-byte line of the first stages of the workgroups to come - on the XCD whose L2 will be asked
// (from another one, through the Infinity Cache, half of the gain of w2's stages is left) - and drop it.  Nothing waits for them but the end of the launch.
// A step of the 7B architecture behind 512 rows, in turn with the launches without, two cards: 17 .. 32 branches 1.003 .. 1.009 times as fast, 33 .. 64 (us, 48:
// 2720 and 2616) 1.028 .. 1.043, 65 .. 100 (3494 and 3434, 3676 and 3665) 1.002 .. 1.018.
// (Dims of 3585 .. 4096; of others in model_layer.hip.)
// How many stages (us a step of the 7B architecture, 37 forked and 100 branches, 2418 and 3440 without): wq|wk|wv and w1|w3 from the norms 2: 2408 and 3427,
// 3: 2404 and 3425, 8: 2416 and 3446 (the norms end later), wo from the attention 4 more: 2395 and 3422, w2 from SwiGLU, too, all of its 22 stages: 2332 and
// 3387, 16: 2335 and 3367, 8: 2369 and 3384.  The prompt's rows for the attention, from wq|wk|wv's idle compute units: no gain.  GEMVs, which
// stream from their first microsecond on: no gain (7B and 70B, 10 branches).
#pragma once

#include "q40_matmul.hpp"

namespace smh {

struct WarmWeights {
    const uint8_t *w[SMH_MAX_SEGMENTS];        // tiled
    int unit0[SMH_MAX_SEGMENTS];               // first column unit of each
    int units, units_pad;                      // column units (swiglu: 128-column blocks of either weight)
    int slices, steps, steps_per_slice;        // of K
    int stages;                                // to ask for, of each workgroup to come
    int swiglu;                                // w: gate, up (q40_gemm_swiglu_kernel), else q40_gemm_kg_kernel
    int workgroups;                            // that ask, a multiple of 8 (0: none)
};

// What workgroup `at` of the launch to come reads: stages (two steps) start, start + 1, .. of `stages`, `piece` and, without swiglu, the piece behind it of
// the tiles from `tile0` on.  False: it has no work.  (The launches' own order: the kernels' blockIdx.)
struct WarmBlock {
    int sg, stages, start, piece;
    long tile0;
};
__host__ __device__ inline int warm_blocks(const WarmWeights &p) { return p.swiglu ? 2 * p.units : 2 * p.units_pad * p.slices; }
__host__ __device__ inline bool warm_block(const WarmWeights &p, int at, WarmBlock &b) {
    int hb = at;
    if (p.swiglu) {
        b.sg = 0;
        b.stages = p.steps / 2;
        b.piece = hb & 3;
        b.tile0 = (long)(hb >> 2) * p.steps;
    } else {
        const int slice = at / (2 * p.units_pad), step0 = slice * p.steps_per_slice;
        hb -= slice * 2 * p.units_pad;
        const int slot = hb >> 1, unit = (slot & 7) * (p.units_pad >> 3) + (slot >> 3);
        if (unit >= p.units) return false;
        b.sg = unit >= p.unit0[2] ? 2 : unit >= p.unit0[1] ? 1 : 0;
        b.stages = (p.steps - step0 < p.steps_per_slice ? p.steps - step0 : p.steps_per_slice) / 2;
        b.piece = 2 * (hb & 1);
        b.tile0 = (long)(unit - (b.sg == 2 ? p.unit0[2] : b.sg == 1 ? p.unit0[1] : 0)) * p.steps + step0;
    }
    if (b.stages < 1) return false;
    b.start = hb * 5 % b.stages;
    return true;
}
// Lines of a stage: two steps of two pieces, with the scales of a tile (swiglu: of either tile).  Line i: its weight and its byte there.
__host__ __device__ inline int warm_lines(const WarmWeights &p) { return p.swiglu ? 40 : 36; }
__host__ __device__ inline long warm_line(const WarmWeights &p, const WarmBlock &b, int i, int &sg) {
    const int per = warm_lines(p), st = i / per, r = i - st * per, kk = r >= per / 2 ? 1 : 0, r2 = r - kk * (per / 2);
    const int up = p.swiglu && r2 >= 10 ? 1 : 0, l = r2 - 10 * up, pieces = p.swiglu ? 8 : 16;
    int stage = b.start + st;
    stage -= stage >= b.stages ? b.stages : 0;
    sg = b.sg + up;
    return (b.tile0 + 2 * stage + kk) * TILE_BYTES + (l < pieces ? b.piece * 1024 + l * 128 : TILE_W_BYTES + (l - pieces) * 128);
}

// Workgroup `group` of `workgroups` / 8 on XCD `xcd`, all of its threads (a group past those: nothing)
__device__ __forceinline__ void warm_weights(const WarmWeights &p, int xcd, int group, int tid, int threads) {
    uint32_t seen = 0;
    if (8 * group >= p.workgroups) return;
    for (int at = 8 * group + xcd; at < warm_blocks(p); at += p.workgroups) {
        WarmBlock b;
        if (!warm_block(p, at, b)) continue;
        const int lines = (p.stages < b.stages ? p.stages : b.stages) * warm_lines(p);
        for (int i = tid; i < lines; i += threads) {
            int sg;
            const long off = warm_line(p, b, i, sg);
            const uint8_t *w = sg == 2 ? p.w[2] : sg == 1 ? p.w[1] : p.w[0];
            seen ^= *reinterpret_cast<const uint32_t *>(w + off);
        }
    }
    asm volatile("" ::"v"(seen));              // (a load that nothing uses would not be made)
}

// ... of the launch that smh_q40_matmul_partial_tiled (smh_q40_matmul_tiled_swiglu) makes for these arguments: no workgroups where it takes another kernel
// or would refuse the weights.
WarmWeights q40_warm(int M, int K, int nseg, const void *const *tiled, const int *n, bool swiglu, int stages, int workgroups);

// The entry points of these names, with workgroups for the launch behind them
int partial_rmsnorm(const void *partial, int ksplit, int M, int N, const void *h_in, const void *weight, float eps, void *h_out, void *xn_out,
                    const WarmWeights &next, smh_stream_t stream);
int matmul_tiled_swiglu(const void *a, int M, int K, long lda, const void *tiled_gate, const void *tiled_up, int n_half, void *out, long ldo,
                        const WarmWeights &next, smh_stream_t stream);
int shared_prefix_attn_qkv_tiles(const void *qkv_partial, int ksplit, void *out, int B, int H, int Hkv, int D, const void *cos_tab, const void *sin_tab,
                                 const int32_t *pos_dev, const void *prefix_k, const void *prefix_v, int P, void *cache_k, void *cache_ks, void *cache_v,
                                 void *cache_vs, int Smax, const int32_t *t_dev, const int32_t *pages, int pages_stride, long cache_rows,
                                 const WarmWeights &next, smh_stream_t stream);
// smh_q40_matmul_partial_tiled; blocks: up to 16 rows, too, on q40_gemm_kg_kernel, for which blocks_plan is not 0 (the slabs it leaves)
int matmul_partial_tiled(const void *a, int M, int K, long lda, int nseg, const void *const *tiled, const int *n, void *partial, size_t partial_bytes,
                         bool blocks, smh_stream_t stream);
int blocks_plan(int M, int K, int nseg, const int *n);
// smh_q40_matmul_partial_tiled_norm; steps: whatever smh_decode_norm_in_fits takes.
int matmul_partial_tiled_norm(const void *h, long ldh, const void *sums, const void *norm_weight, float eps, int M, int K, int nseg, const void *const *tiled,
                              const int *n, void *partial, size_t partial_bytes, bool steps, smh_stream_t stream);
// compute units that a launch of these leaves without a workgroup, in eights
int swiglu_idle(int n_half);
int attn_tiles_idle(int B, int H, int Hkv);

}  // namespace smh
