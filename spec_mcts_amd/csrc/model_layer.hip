// One transformer layer of a decode step or of a prefill as ONE host call.
//
// Issued operator by operator from Python a decode layer costs ~90 us of host time (eight or nine operators, each with its
// checks, its output tensors and a foreign call), which at one branch is more than the GPU needs for it: a step of the
// 32-layer model took 3.0 ms where a captured graph of the same launches takes 2.0.  Here the layer's launches are issued one
// behind the other (2-3 us each), out of buffers the caller allocated once for the whole pass.  The operators and their roundings are those of
// Transformer._forward_fused in hf_model_q40_kv_shared.py; which launches they share is decided here (as_blocks, attn_way, norm_linears, LayerRun::swiglu).
#include "attn_tiles.hpp"
#include "q40_warm.hpp"

namespace smh {

constexpr size_t align_up(size_t n) { return (n + 255) & ~(size_t)255; }

// Buffers of a pass over `rows` rows, carved out of one allocation.
struct LayerBuffers {
    char *h[2], *xn, *q, *k, *v, *att, *act;   // fp16; the residual stream moves from one h to the other at every norm
    float *sums, *slab_a, *slab_b;             // slabs of wq|wk|wv and w1|w3 (a), of wo and w2 (b)
    size_t slab_a_bytes, slab_b_bytes, total;
};

// Stages of the next launch's weights that a launch asks for (q40_warm.hpp).  The norms of layers whose w1|w3 leaves slabs do not ask (17 .. 28 branches of the 7B
// shape behind 64 prompt rows: 0.992 .. 0.997 times as fast); their attention does (17 .. 48 branches behind 256 and 512 rows, SwiGLU switched off: 1.001 .. 1.009).
// Up to three row tiles, that is: above, the attention's workgroups are many and long themselves (dim 4096, times as long with its asking as without, 17 / 32 / 48 / 64 / 65 / 80 / 100
// branches: FFN 11008 0.995 / 0.99 / level / level / 1.005 / 1.002 / 1.003, 8192 1.001 / 1.004 / 0.999 / - / 1.005 / 1.002 / 1.006, 12288 0.996 / 0.999 / 0.997 / - / 1.004 / 1.003 / 1.002, 16384
// 1.003 / 1.002 / 1.003 / - / 1.004 / 1.005 / 1.027).
// Nothing is asked for outside of dims 3585 .. 4096.  A wider RMSNorm takes two passes, and one of its workgroups a compute unit's registers, so that the asking ones wait
// for the rows or the rows for them; narrower layers' launches are shorter than the asking.  Times as long with the asking as without it, decode behind 96 to 1024
// rows at 33 / 48 / 65 / 100 branches: dim 4096, FFN 11008 0.97 / 0.96 / 0.985 / 0.995, dim 3840, FFN 10240 (32 branches) 0.98 / 0.97 / 0.995 / 0.98; dim 3584, FFN 9728
// 1.01 / 1.00 / 0.99 / 0.985, 3072, 8192 1.015 / 1.015 / 1.02 / 1.015, 2048, 8192 1.01 / 1.01 / 1.015 / 1.015, 2048, 5632 level / level / 1.01 / 1.01; 4608, 12288 1.03 / 1.02 / 1.02 / 1.01, 5120, 13824
// 1.025 / 1.015 / 1.015 / 1.005, 5120, 10240 1.01 / 1.07 / 0.985 / 0.985, 6144, 16384 1.01 / 1.01 / level / level; three layers of 64 heads over 8, dim 8192, 17 .. 100 branches behind
// 1024 rows 0.999 .. 1.002 from the norms, 1.000 .. 1.004 from the attention.
// SwiGLU's launch asks for w2 where 40 compute units and more are left to do it (dim 4096, times as long with its asking as without at 17 / 24 / 32 / 48 branches: FFN 13312, 48 units
// 1.00 / 0.99 / 0.995 / 0.98, 13824, 40 units 0.995 / - / 0.99 / 0.985; 14336, 32 units 1.00 / 1.02 / 1.03 / 1.015), and the norms do where it leaves 32 (14336, without w2's,
// 0.995 / 0.985 / 0.985 / 0.985; 16384, where it fills the chip, 1.01 / 1.01 / 1.02 / 1.00, at 5 and 16 branches 1.01 and 1.005).
constexpr int WARM_MIN_DIM = 3585, WARM_MAX_DIM = 4096, WARM_FROM_NORM = 3, WARM_FROM_ATTENTION = 4, WARM_FROM_ATTENTION_ROWS = 48, WARM_FROM_SWIGLU = 16, WARM_NORM_MIN_IDLE = 32, WARM_SWIGLU_MIN_IDLE = 40;

static int slices(int M, int K, int nseg, const int *n) { return smh_q40_matmul_plan_tiled(M, K, nseg, n); }
// Launches of 17 rows and more (128-column blocks, SwiGLU inside w1|w3, the norms and the attention asking for the next weights) for a layer of fewer, too,
// where all four linears have them: bound by latency both ways, they are fewer (no SiLU launch), leave 2 to 8 slabs instead of 5 to 16, and their weights are
// on their way earlier.  7B architecture, 512 + 50 rows, us a step with the GEMVs and so: 5 branches 1976 and 1946, 6 2009 and 1949, 8 2022 and 2007, 10 2119
// and 2018, 12 2149 and 2040, 16 2275 and 2126; 32 heads over 8 with FFN 14336 (five slabs of wq|wk|wv) the step is 1.07 .. 1.15 times as fast, eight layers, 5 to
// 16 branches behind 100 to 1024 rows, 20 and 110 of their own (5 branches behind 256 560 and 513, 16 596 and 522).  (4, which the launch of all layers takes with probabilities
// of 32 bits, not 16: 2150 there and 1950 so.)  SwiGLU inside at 17 / 24 / 32 branches: 2360 / 2432 / 2495 -> 2250 /
// 2318 / 2361, with FFN 14336 and 8 kv heads 1.03 .. 1.07 times as fast, with dim 5120 and FFN 13824 1.02 .. 1.03.  Behind short prompts a decode step stays what it was (ATTN_TILES_MIN_PROMPT: two evaluations that differ in one rounding drift apart there).
constexpr int BLOCKS_MIN_ROWS = 5, BLOCKS_MIN_PROMPT = 96;
static bool as_blocks(const smh_layer &L, int M, bool swiglu_in) {
    const int n_qkv[3] = {L.heads * 128, L.kv_heads * 128, L.kv_heads * 128}, n_dim[1] = {L.dim};
    return M >= BLOCKS_MIN_ROWS && M <= SMH_GEMV_MAX_M && swiglu_in && gemm_swiglu_fits(M, L.dim, L.ffn, true) && blocks_plan(M, L.dim, 3, n_qkv) > 0 &&
           blocks_plan(M, L.heads * 128, 1, n_dim) > 0 && blocks_plan(M, L.ffn, 1, n_dim) > 0;
}
// SwiGLU inside w1|w3 of a layer (far: a prefill, or a decode step behind a longer prompt).  17 .. 32 rows want more workgroups than more rows do, as the slabs
// they save are smaller: two thirds of the compute units up to 24 rows, the half and a sixteenth from there on.  Times as long as with slabs, decode behind 96 to 1024 rows at 17 / 24 /
// 32 branches and prefills of 17 / 24 / 32: 4096 -> 8192 (128 workgroups) 1.04 / 1.02 / 1.02 and 1.05 / 1.05 / 1.05, 3072 -> 8192 1.04 / 1.03 / 1.03 and 1.02 / 1.04 / 1.01,
// 4096 -> 9216 (144) 1.00 / 0.98 / 0.97 and level / 1.01 / level, 3584 -> 9728 (152) 1.01 / 1.01 / 1.00 and 1.03 / level / level, 4096 -> 10240 (160, 8 kv heads) 1.01 / 1.00 / 0.99 and
// 1.015 / 1.01 / level, 5120 -> 10240 1.01 / 1.00 / 0.99; 4096 -> 11008 (172) 0.94 / 0.93 / 0.93, 3072 -> 12288 0.93 / 0.92 / 0.90.
static bool swiglu_inside(const smh_layer &L, int M, bool blocks, bool far) {
    if (!gemm_swiglu_fits(M, L.dim, L.ffn, true)) return false;
    if (M <= SMH_GEMV_MAX_M) return blocks;
    return M > 32 || (far && 2 * (L.ffn / 128) >= (M <= 24 ? 171 : 144));
}
// A launch that stores its fp16 results itself (more than 128 rows, no K-split) leaves no slabs.  layer_buffers reserves none for it,
// so every linear below asks here before it takes the slab form.
static bool direct(int M, int K, int nseg, const int *n) { return smh_q40_matmul_tiled_direct_fits(M, K, nseg, n) == 1; }

// The attention of a decode layer: in one launch whose last workgroups merge (ONE, up to 16 queries a kv head), in one launch of 8 or 16
// queries a workgroup (TILES), or RoPE, prefix slices and walks (LAUNCHES).  us a call with RoPE and append, caches in HBM (32 heads, up to 16 branches: two slabs, 10 own rows):
//   32 heads, branches after prompt rows   ONE   TILES LAUNCHES  |  64 heads over 8                ONE   TILES LAUNCHES
//     5 /  512                             11.7   13.4   14.2    |     1 /  512 (8 queries)        12.2   13.7   13.6
//    16 /  256                             12.1    9.8   14.4    |     1 / 2047                    17.0   22.6   16.6
//    10 /  768                             15.7   14.1   16.9    |     2 /  128 (16 queries)       10.7   11.2   12.7
//    10 / 1024                             21.8   17.3   17.9    |     2 /  512                    15.6   13.7   14.1
//    10 / 2047                             36.2   25.8   20.8    |     2 / 2047                    24.2   22.4   17.9
//    17 /  512                               -    16.9   18.9    |     3 /  512                      -    11.8   14.9
//    17 / 1024                               -    21.5   21.8    |     3 / 1024                      -    18.6   17.5
//    17 / 2047                               -    29.3   26.0    |    10 / 1024                      -    18.0   21.4
//    32 / 2047                               -    29.3   28.5    |    10 / 2047                      -    25.2   23.4
//    48 / 2047                               -    31.5   32.0    |    16 / 2047                      -    24.4   26.3
//   100 / 2047                               -    34.7   47.7    |   100 / 2047                      -    48.8   65.6
//                                                                |  40 heads, 100 / 512 (two rounds) -   39.5   39.0
// (Multi-head attention, with ONE's slices of 64 rows and two slabs, us a step of the 7B architecture with ONE and LAUNCHES, 10 / 60 / 120 rows of their own: 700 prompt
// rows, 10 branches 2097 / 2112 / 2164 and 2142 / 2154 / 2206, 16 2158 / 2225 / 2382 and 2183 / 2196 / 2251; 768 rows, 8 branches 2046 / 2060 / 2124 and 2104 / 2113 /
// 2138, 9 2093 / 2185 / 2343 and 2138 / 2150 / 2200, where its waves no longer fit one round in pairs.  With more heads they stop fitting earlier, but LAUNCHES is the
// faster way behind 705 .. 768 rows there too: eight layers of 40 heads behind 730, 9 / 16 branches, 110 own rows 801 / 903 and 732 / 778, four of 64 heads behind 720 696 / 774
// and 676 / 701, quotients above those of the same trees behind 704.)
// A long prompt wants more workgroups than few tiles are, and ONE's merge grows with the slices.  Where the table has a faster form than the rule takes,
// the line is not drawn yet: multi-head attention of 6 to 16 branches (with TILES the step is faster at 10 own rows and slower at 120) and one grouped branch
// behind a long prompt stay with ONE up to the lines of the rule.  Behind fewer than 96 prompt rows results stay
// where they are: there two evaluations that differ in one rounding drift 3e-2 (40 rows) to 6e-2 (16 rows) apart within eight steps of the 7B
// architecture, 1.5e-2 behind 96.
enum AttnWay { ATTN_ONE, ATTN_TILES, ATTN_LAUNCHES };
constexpr int ATTN_TILES_MIN_PROMPT = 96;
static AttnWay attn_way(int M, int heads, int kv_heads, int P, bool one, bool tiles, bool launches) {
    const int rep = heads / kv_heads;
    const long queries = (long)M * rep;                      // of a kv head
    if (one && (rep == 1 ? P <= (M > 8 ? 704 : 768) : queries <= 8 || P <= 256)) return ATTN_ONE;
    const bool round = (kv_heads + 7) / 8 * 8 * ((queries + 15) / 16) <= 256;
    if (tiles && P >= ATTN_TILES_MIN_PROMPT && (rep > 1 || (M > SMH_GEMV_MAX_M && round)) &&
        (P <= 512 || P <= kv_heads * ((queries + 7) / 8) * (rep == 1 ? 12 : 24)))
        return ATTN_TILES;
    return one && !launches ? ATTN_ONE : ATTN_LAUNCHES;
}

static int layer_buffers(const smh_layer &L, int M, bool swiglu_in, char *base, LayerBuffers &b) {
    const int nq = L.heads * 128, nkv = L.kv_heads * 128;
    const int n_qkv[3] = {nq, nkv, nkv}, n_gu[2] = {L.ffn, L.ffn}, n_dim[1] = {L.dim};
    const int ks_qkv = slices(M, L.dim, 3, n_qkv), ks_gu = slices(M, L.dim, 2, n_gu), ks_o = slices(M, nq, 1, n_dim), ks_d = slices(M, L.ffn, 1, n_dim);
    if (ks_qkv < 1 || ks_gu < 1 || ks_o < 1 || ks_d < 1) return -1;
    const bool blocks = as_blocks(L, M, swiglu_in);
    const size_t m = (size_t)M;
    auto most = [](size_t x, size_t y) { return x > y ? x : y; };
    const bool gu_slabs = !(M > 128 && swiglu_in && smh_q40_swiglu_fits(M, L.dim, L.ffn));
    const bool qkv_slabs = !direct(M, L.dim, 3, n_qkv), o_slabs = !direct(M, nq, 1, n_dim), d_slabs = !direct(M, L.ffn, 1, n_dim);
    auto slabs = [&](int ks, int K, int nseg, const int *n) { return most((size_t)ks, blocks ? (size_t)blocks_plan(M, K, nseg, n) : 0); };
    b.slab_a_bytes = align_up(most(qkv_slabs ? slabs(ks_qkv, L.dim, 3, n_qkv) * m * (nq + 2 * (size_t)nkv) : 1, gu_slabs ? ks_gu * m * 2 * (size_t)L.ffn : 1) * sizeof(float));
    b.slab_b_bytes = align_up((size_t)most(o_slabs ? slabs(ks_o, nq, 1, n_dim) : 0, d_slabs ? slabs(ks_d, L.ffn, 1, n_dim) : 0) * m * L.dim * sizeof(float));
    size_t at = 0;
    auto take = [&](size_t bytes) { char *p = base ? base + at : nullptr; at += align_up(bytes); return p; };
    b.h[0] = take(m * L.dim * 2);
    b.h[1] = take(m * L.dim * 2);
    b.xn = take(m * L.dim * 2);
    b.q = take(m * nq * 2);
    b.k = take(m * nkv * 2);
    b.v = take(m * nkv * 2);
    b.att = take(m * nq * 2);
    b.act = take(m * L.ffn * 2);
    b.sums = (float *)take(m * 16 * sizeof(float));
    b.slab_a = (float *)take(b.slab_a_bytes);
    b.slab_b = (float *)take(b.slab_b_bytes);
    b.total = at;
    return 0;
}

// What a decode layer and a prefill layer share: the arguments checked, the buffers, and the residual stream on its way through them.
struct LayerRun {
    const smh_layer &L;
    smh_pass &S;
    smh_stream_t stream;
    const int M, nq, nkv;
    const bool blocks, swiglu;                 // far: not a decode step behind a short prompt
    const int n_qkv[3], n_gu[2], n_dim[1];
    const void *w_qkv[3], *w_o[1], *w_gu[2], *w_d[1];
    LayerBuffers b;

    LayerRun(const smh_layer &l, smh_pass &s, smh_stream_t st, bool far)
        : L(l), S(s), stream(st), M(s.rows), nq(l.heads * 128), nkv(l.kv_heads * 128), blocks(far && as_blocks(l, s.rows, s.swiglu_in != 0)),
          swiglu(s.swiglu_in != 0 && swiglu_inside(l, s.rows, blocks, far)), n_qkv{nq, nkv, nkv}, n_gu{l.ffn, l.ffn}, n_dim{l.dim},
          w_qkv{l.wq, l.wk, l.wv}, w_o{l.wo}, w_gu{l.w1, l.w3}, w_d{l.w2} {}
    // What the launches of a decode layer ask for ahead: the norms, where SwiGLU is inside, for the product behind them, the attention of tiles for wo, SwiGLU for w2
    bool asks() const { return L.dim >= WARM_MIN_DIM && L.dim <= WARM_MAX_DIM && (M > SMH_GEMV_MAX_M || blocks); }
    WarmWeights ask_qkv() const { return asks() && swiglu && swiglu_idle(L.ffn) >= WARM_NORM_MIN_IDLE ? q40_warm(M, L.dim, 3, w_qkv, n_qkv, false, WARM_FROM_NORM, 256) : WarmWeights{}; }
    WarmWeights ask_gu() const { return asks() && swiglu && swiglu_idle(L.ffn) >= WARM_NORM_MIN_IDLE ? q40_warm(M, L.dim, 2, w_gu, n_gu, true, WARM_FROM_NORM, 256) : WarmWeights{}; }
    WarmWeights ask_o() const {
        const int row = (L.kv_heads + 7) / 8 * 8;
        WarmWeights wo = asks() && M <= WARM_FROM_ATTENTION_ROWS ? q40_warm(M, nq, 1, w_o, n_dim, false, WARM_FROM_ATTENTION, attn_tiles_idle(M, L.heads, L.kv_heads)) : WarmWeights{};
        wo.workgroups = wo.workgroups / row * row;
        return wo;
    }
    WarmWeights ask_d() const { return asks() && swiglu && swiglu_idle(L.ffn) >= WARM_SWIGLU_MIN_IDLE ? q40_warm(M, L.ffn, 1, w_d, n_dim, false, WARM_FROM_SWIGLU, swiglu_idle(L.ffn)) : WarmWeights{}; }
    int slabs(int K, int nseg, const int *n) const { return blocks ? blocks_plan(M, K, nseg, n) : slices(M, K, nseg, n); }
    int begin(const char *who) {
        SMH_REQUIRE(M >= 1 && L.heads > 0 && L.kv_heads > 0 && L.heads % L.kv_heads == 0, "%s: rows=%d heads=%d kv_heads=%d", who, M, L.heads, L.kv_heads);
        if (layer_buffers(L, M, S.swiglu_in != 0, (char *)S.scratch, b) != 0) return -1;
        SMH_REQUIRE(S.scratch && S.scratch_bytes >= b.total, "%s: scratch %zu < %zu bytes", who, S.scratch_bytes, b.total);
        return 0;
    }
    // S.h += the product of the linear before (S.pending slabs in slab_b), then its RMSNorm: to b.xn
    int norm(const void *weight, float eps, const WarmWeights &next = WarmWeights{}) {
        void *h_out = S.pending > 0 ? b.h[S.h == b.h[0]] : nullptr;
        const int r = partial_rmsnorm(S.pending > 0 ? b.slab_b : nullptr, S.pending > 0 ? S.pending : 1, M, L.dim, S.h, weight, eps, h_out, b.xn, next, stream);
        if (h_out != nullptr) S.h = h_out;
        S.pending = 0;
        return r;
    }
    // S.h += x . w, at once or as slabs that the next norm adds
    int residual_linear(const void *x, int K, const void *const *w) {
        if (direct(M, K, 1, n_dim)) {
            void *out[1] = {b.h[S.h == b.h[0]]};
            const int r = smh_q40_matmul_tiled_direct(x, M, K, K, 1, w, n_dim, out, S.h, L.dim, stream);
            S.h = out[0];
            return r;
        }
        S.pending = slabs(K, 1, n_dim);
        return matmul_partial_tiled(x, M, K, K, 1, w, n_dim, b.slab_b, b.slab_b_bytes, blocks, stream);
    }
};

}  // namespace smh

using namespace smh;

extern "C" size_t smh_decode_scratch_bytes(const smh_layer *layer, int rows, int swiglu_in) {
    LayerBuffers b;
    if (layer == nullptr || rows < 1 || layer_buffers(*layer, rows, swiglu_in != 0, nullptr, b) != 0) return 0;
    return b.total;
}

extern "C" int smh_decode_layer_form(const smh_layer *layer, int rows, int swiglu_in, int *slabs) {
    const char *who = "smh_decode_layer_form";
    SMH_REQUIRE(layer && slabs, "%s: null pointer", who);
    smh_pass pass{};
    pass.rows = rows;
    pass.swiglu_in = swiglu_in != 0;
    LayerBuffers b;
    SMH_REQUIRE(rows >= 1 && layer->heads > 0 && layer->kv_heads > 0 && layer->heads % layer->kv_heads == 0, "%s: rows=%d heads=%d kv_heads=%d", who, rows, layer->heads, layer->kv_heads);
    if (layer_buffers(*layer, rows, pass.swiglu_in, nullptr, b) != 0) return -1;
    const LayerRun run(*layer, pass, nullptr, layer->prompt_len >= BLOCKS_MIN_PROMPT);
    auto left = [&](int K, int nseg, const int *n) { return direct(rows, K, nseg, n) ? 0 : run.slabs(K, nseg, n); };
    slabs[0] = left(layer->dim, 3, run.n_qkv);
    slabs[1] = left(run.nq, 1, run.n_dim);
    slabs[2] = run.swiglu ? 0 : slices(rows, layer->dim, 2, run.n_gu);
    slabs[3] = left(layer->ffn, 1, run.n_dim);
    return (run.blocks ? 1 : 0) | (run.swiglu ? 2 : 0);
}

extern "C" int smh_decode_layer_asks(const smh_layer *layer, int rows, int swiglu_in) {
    const char *who = "smh_decode_layer_asks";
    SMH_REQUIRE(layer, "%s: null pointer", who);
    int slabs[4];
    const int form = smh_decode_layer_form(layer, rows, swiglu_in, slabs);
    if (form < 0) return form;
    smh_layer L = *layer;
    const void *const some = (const void *)128;             // (weights that a product would take)
    L.wq = L.wk = L.wv = L.wo = L.w1 = L.w2 = L.w3 = some;
    smh_pass pass{};
    pass.rows = rows;
    pass.swiglu_in = swiglu_in != 0;
    const LayerRun run(L, pass, nullptr, L.prompt_len >= BLOCKS_MIN_PROMPT);
    return (run.ask_qkv().workgroups > 0 ? 1 : 0) | (run.ask_gu().workgroups > 0 ? 2 : 0) | (run.ask_o().workgroups > 0 ? 4 : 0) | (run.ask_d().workgroups > 0 ? 8 : 0);
}

extern "C" int smh_decode_layer(const smh_layer *layer, smh_pass *pass, smh_stream_t stream) {
    const char *who = "smh_decode_layer";
    SMH_REQUIRE(layer && pass && pass->h, "%s: null pointer", who);
    LayerRun run(*layer, *pass, stream, layer->prompt_len >= BLOCKS_MIN_PROMPT);
    int st = run.begin(who);
    if (st) return st;
    const smh_layer &L = *layer;
    smh_pass &S = *pass;
    const LayerBuffers &b = run.b;
    const int M = run.M, nq = run.nq;
    // the RMSNorm of the residual stream and the linears behind it: to slab_a.  With few rows the RMSNorm is made inside the linears' launch.
    auto norm_linears = [&](const void *weight, float eps, int nseg, const void *const *w, const int *n) -> int {
        if (S.pending == 0 || M > S.norm_in_rows || run.blocks || ((uintptr_t)weight & 15) != 0 || smh_decode_norm_in_fits(M, L.dim, nseg, n) != 1) {
            if (int r = run.norm(weight, eps, nseg == 3 ? run.ask_qkv() : WarmWeights{})) return r;
            return matmul_partial_tiled(b.xn, M, L.dim, L.dim, nseg, w, n, b.slab_a, b.slab_a_bytes, run.blocks, stream);
        }
        void *h_out = b.h[S.h == b.h[0]];
        if (int r = smh_partial_residual_sumsq(b.slab_b, S.pending, M, L.dim, S.h, h_out, b.sums, stream)) return r;
        S.h = h_out;
        S.pending = 0;
        return matmul_partial_tiled_norm(h_out, L.dim, b.sums, weight, eps, M, L.dim, nseg, w, n, b.slab_a, b.slab_a_bytes, true, stream);
    };
    // ---- attention ----
    const int rep = L.heads / L.kv_heads;
    const bool qkv_direct = direct(M, L.dim, 3, run.n_qkv);
    const long rows = S.pages != nullptr ? S.cache_rows : (long)M * S.smax;
    // What only some of the three ask for never decides whether a pass is taken.  A table of another width than a branch has rows: TILES and ONE cut the
    // walks at the rows, LAUNCHES at the table.  TILES and LAUNCHES check page ids against cache_rows, LAUNCHES writes partials to attn_ws.
    const bool may_one = S.attn_one != 0 && M * rep <= 16, table = S.pages == nullptr || (S.pages_stride == S.smax && S.cache_rows >= 1);
    const bool can_launch = table && S.attn_ws != nullptr && S.attn_ws_bytes >= smh_attn_workspace_bytes(M, L.heads, L.prompt_len);
    const bool can_tile = S.attn_from_qkv != 0 && !qkv_direct && table &&
                          attn_tiles_refuse({b.slab_a, b.att, S.cos_tab, S.sin_tab, L.prompt_k, L.prompt_v, L.cache_k, L.cache_ks, L.cache_v, L.cache_vs, M,
                                             L.heads, L.kv_heads, L.prompt_len, rows}) == nullptr;
    const AttnWay way = attn_way(M, L.heads, L.kv_heads, L.prompt_len, may_one, can_tile, can_launch);
    const int one = way == ATTN_ONE;
    void *ws = one ? S.attn_one_ws : S.attn_ws;
    const size_t ws_bytes = one ? S.attn_one_ws_bytes : S.attn_ws_bytes;
    if (qkv_direct) {
        if ((st = run.norm(L.att_norm, L.att_eps))) return st;
        void *out[3] = {b.q, b.k, b.v};
        st = smh_q40_matmul_tiled_direct(b.xn, M, L.dim, L.dim, 3, run.w_qkv, run.n_qkv, out, nullptr, 0, stream);
    } else {
        st = norm_linears(L.att_norm, L.att_eps, 3, run.w_qkv, run.n_qkv);
    }
    if (st) return st;
    const int ks_qkv = run.slabs(L.dim, 3, run.n_qkv);
    // (Only in one launch: in two, each of the 256 prefix workgroups adds up and rotates all queries of its kv head.  Grouped queries,
    // three layers of 64 heads over 8 kv heads: 10 branches after 2047 rows 594 us a step so, 552 with the RoPE launch in front; 3
    // branches 523 against 511, 16 branches 629 against 571.)
    if (S.attn_from_qkv != 0 && one && M <= SMH_GEMV_MAX_M) {
        st = smh_shared_prefix_attn_qkv(b.slab_a, ks_qkv, b.att, M, L.heads, L.kv_heads, 128, S.cos_tab, S.sin_tab, S.pos_dev, L.prompt_k, L.prompt_v,
                                        L.prompt_len, L.cache_k, L.cache_ks, L.cache_v, L.cache_vs, S.smax, S.t_dev, S.pages, S.pages_stride, one, ws,
                                        ws_bytes, stream);
    } else if (way == ATTN_TILES) {
        st = shared_prefix_attn_qkv_tiles(b.slab_a, ks_qkv, b.att, M, L.heads, L.kv_heads, 128, S.cos_tab, S.sin_tab, S.pos_dev, L.prompt_k, L.prompt_v,
                                          L.prompt_len, L.cache_k, L.cache_ks, L.cache_v, L.cache_vs, S.smax, S.t_dev, S.pages, S.pages_stride,
                                          S.cache_rows, run.ask_o(), stream);
    } else {
        st = qkv_direct ? smh_rope_append_kv(b.q, b.k, b.v, M, L.heads, L.kv_heads, 128, S.cos_tab, S.sin_tab, S.pos_dev, L.cache_k, L.cache_ks, L.cache_v,
                                             L.cache_vs, S.smax, S.t_dev, stream)
                        : smh_partial_rope_append_kv(b.slab_a, ks_qkv, M, L.heads, L.kv_heads, 128, b.q, b.k, b.v, S.cos_tab, S.sin_tab, S.pos_dev, L.cache_k,
                                                     L.cache_ks, L.cache_v, L.cache_vs, S.smax, S.t_dev, stream);
        if (st == 0 && S.pages != nullptr)
            st = smh_paged_prefix_attn(b.q, b.att, M, L.heads, L.kv_heads, 128, L.prompt_k, L.prompt_v, L.prompt_len, 0, 0, SMH_KV_Q40, L.cache_k,
                                       L.cache_v, L.cache_ks, L.cache_vs, 0, 0, S.cache_rows, S.pages, 4, S.pages_stride, S.pages_stride, S.t_dev, 0,
                                       b.k, b.v, one, ws, ws_bytes, stream);
        else if (st == 0)
            st = (one ? smh_shared_prefix_attn_one : smh_shared_prefix_attn)(b.q, b.att, M, L.heads, L.kv_heads, 128, L.prompt_k, L.prompt_v, L.prompt_len,
                                                                             SMH_KV_Q40, L.cache_k, L.cache_v, L.cache_ks, L.cache_vs, S.smax, S.t_dev, 0,
                                                                             b.k, b.v, ws, ws_bytes, stream);
    }
    if (st) return st;
    if ((st = run.residual_linear(b.att, nq, run.w_o))) return st;
    // ---- feed forward ----
    if (run.swiglu) {
        if ((st = run.norm(L.ffn_norm, L.ffn_eps, run.ask_gu()))) return st;
        if ((st = matmul_tiled_swiglu(b.xn, M, L.dim, L.dim, L.w1, L.w3, L.ffn, b.act, L.ffn, run.ask_d(), stream))) return st;
        return run.residual_linear(b.act, L.ffn, run.w_d);
    }
    if ((st = norm_linears(L.ffn_norm, L.ffn_eps, 2, run.w_gu, run.n_gu))) return st;
    const int ks_gu = slices(M, L.dim, 2, run.n_gu);
    if (M <= S.silu_in_rows && L.ffn % 32 == 0) {
        S.pending = slices(M, L.ffn, 1, run.n_dim);
        return smh_q40_matmul_partial_tiled_silu(b.slab_a, ks_gu, M, L.ffn, 1, run.w_d, run.n_dim, b.slab_b, b.slab_b_bytes, stream);
    }
    if ((st = smh_partial_silu_mul(b.slab_a, ks_gu, M, L.ffn, b.act, stream))) return st;
    return run.residual_linear(b.act, L.ffn, run.w_d);
}

// One layer of a prefill of `rows` tokens (TransformerBlock.forward with start_pos == 0): k and v go straight to the prompt cache.
// Above 128 rows the linears store their fp16 results themselves wherever their launch needs no K-split (the residual adds of
// wo and w2 inside, and RoPE), and SiLU(gate) * up is made inside w1|w3's launch.
extern "C" int smh_prefill_layer(const smh_layer *layer, smh_pass *pass, smh_stream_t stream) {
    const char *who = "smh_prefill_layer";
    SMH_REQUIRE(layer && pass && pass->h, "%s: null pointer", who);
    LayerRun run(*layer, *pass, stream, true);
    int st = run.begin(who);
    if (st) return st;
    const smh_layer &L = *layer;
    smh_pass &S = *pass;
    const LayerBuffers &b = run.b;
    const int M = run.M, nq = run.nq;
    if ((st = run.norm(L.att_norm, L.att_eps))) return st;
    if (direct(M, L.dim, 3, run.n_qkv)) {
        void *out[3] = {b.q, L.prompt_k, L.prompt_v};
        if ((((uintptr_t)S.cos_tab | (uintptr_t)S.sin_tab) & 15) == 0 && M < 1 << 24) {
            st = smh_q40_matmul_tiled_direct_rope(b.xn, M, L.dim, L.dim, 3, run.w_qkv, run.n_qkv, out, L.heads + L.kv_heads, S.cos_tab, S.sin_tab, stream);
        } else {
            if ((st = smh_q40_matmul_tiled_direct(b.xn, M, L.dim, L.dim, 3, run.w_qkv, run.n_qkv, out, nullptr, 0, stream))) return st;
            st = smh_rope(b.q, L.prompt_k, M, L.heads, L.kv_heads, 128, S.cos_tab, S.sin_tab, 0, stream);
        }
    } else {
        if ((st = matmul_partial_tiled(b.xn, M, L.dim, L.dim, 3, run.w_qkv, run.n_qkv, b.slab_a, b.slab_a_bytes, run.blocks, stream))) return st;
        st = smh_partial_rope_rows(b.slab_a, run.slabs(L.dim, 3, run.n_qkv), M, L.heads, L.kv_heads, 128, b.q, L.prompt_k, L.prompt_v, S.cos_tab, S.sin_tab, 0,
                                   stream);
    }
    if (st) return st;
    if ((st = smh_prefill_attn(b.q, L.prompt_k, L.prompt_v, b.att, M, L.heads, L.kv_heads, 128, stream))) return st;
    if ((st = run.residual_linear(b.att, nq, run.w_o))) return st;
    if ((st = run.norm(L.ffn_norm, L.ffn_eps))) return st;
    if (run.swiglu) {
        st = matmul_tiled_swiglu(b.xn, M, L.dim, L.dim, L.w1, L.w3, L.ffn, b.act, L.ffn, WarmWeights{}, stream);
    } else if ((st = smh_q40_matmul_partial_tiled(b.xn, M, L.dim, L.dim, 2, run.w_gu, run.n_gu, b.slab_a, b.slab_a_bytes, stream)) == 0) {
        st = smh_partial_silu_mul(b.slab_a, slices(M, L.dim, 2, run.n_gu), M, L.ffn, b.act, stream);
    }
    return st ? st : run.residual_linear(b.act, L.ffn, run.w_d);
}

// The last layer's product added to the residual stream, and the final RMSNorm -> out [rows, dim].
extern "C" int smh_decode_finish(const smh_layer *last, smh_pass *pass, const void *norm_weight, float eps, void *out, smh_stream_t stream) {
    SMH_REQUIRE(last && pass && pass->h && out, "smh_decode_finish: null pointer");
    LayerBuffers b;
    if (layer_buffers(*last, pass->rows, pass->swiglu_in != 0, (char *)pass->scratch, b) != 0) return -1;
    return smh_partial_rmsnorm(pass->pending > 0 ? b.slab_b : nullptr, pass->pending > 0 ? pass->pending : 1, pass->rows, last->dim, pass->h, norm_weight,
                               eps, nullptr, out, stream);
}
