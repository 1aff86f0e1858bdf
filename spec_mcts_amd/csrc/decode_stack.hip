// The transformer layers of a decode step of a few branches as ONE launch.
//
// Layer by layer such a step is seven dependent launches of ~27 MB a layer, and each of them pays ~3.6 us before its bytes stream
// (launch floor, start of the workgroups, first request to first data) and ~1 us behind them.  Here 256 workgroups stay for all
// layers.  What a linear reads of its weights depends on no other workgroup, so the weights of the linears to come are already on
// their way into LDS while a workgroup waits for its activations.
//
// A workgroup (one a compute unit) has 16 waves:
//   * two LOADING waves bring its tiles into a ring of 26 in LDS by DMA, linear after linear, layer after layer, as far ahead as
//     the ring has room.  (In the multiplying waves, a ring each, the loads stopped with the multiplying: 57 us a layer against 46.)
//   * eight MULTIPLYING waves: wave (piece q, class e) multiplies piece q (64 of the 256 columns, 1 KB of nibbles) of every third tile
//     with the activations in LDS (16 x 16 x 32 products, decoded as in q40_gemv.hip).  Its first five or six tiles are in registers
//     before the activations come, which makes the ring 15 to 18 tiles longer, and two of them decoded with one or two branches.
//   * six COMMUNICATING waves: they wait for a linear's activations, leave them in LDS, add up and publish the products, and do
//     what lies between the linears (RMSNorm, attention, SiLU, residual adds).  Four of them multiply the third class of tiles.
// They meet at counters in LDS: a barrier would stop the loads, too.
// Tasks of a linear are equal runs of tiles in the order (column unit, step), one per workgroup; a run touches two units at most, and
// a unit's products are added, in task order, by whoever reads them: results do not depend on scheduling.
//
// Hand-off.  Every value that crosses workgroups travels as an 8-byte word (32 bits of data, 32 bits of tag) in one device-scope
// store, and the reader polls the word itself: 1.6 - 2.0 us from store to use, where stores, a counter and loads behind it
// take 5.1 us (three dependent trips; both measured with 256 workgroups).  The tag counts layers over all launches on a workspace,
// so nothing is cleared.  Words are reused from layer to layer: whoever writes one has waited, through the sums of squares of a
// whole row, for every workgroup's work of the layer before.
//
// Who takes part.  Waiting needs partners that run.  Workgroups sign in when they start; when all have (or 50 us after, if
// others hold compute units) the list is closed, tasks are dealt to those on it, and a workgroup that starts later leaves at
// once.  So any number of running workgroups finishes the work, whatever else the GPU does.  Every wait is bounded all the same:
// a workgroup that has waited too long publishes nothing more and leaves NaN in its part of the result.
//
// A step of the 7B architecture (512 prompt rows and 63 of their own), layer by layer and in one launch, in us: 1 branch 1981 and
// 1451, 2 branches 2100 and 1590, 3 branches 2134 and 1872, 4 branches 2161 and 2094 (after 2047 and 127 rows 3057 and 2585), all of it before
// pieces were decoded ahead (Multiplier).  What a branch adds is the communication:
// its activations go through every workgroup.  So four is where the rule of the sizes (stack_plan) ends.
#include "attn_rows.hpp"
#include "q40_matmul.hpp"
#include "rope_kv.hpp"

namespace smh {

constexpr int DS_WGS = 256;                    // workgroups of a launch = most tasks of a linear
constexpr int DS_LAYERS = 32;                  // layers of a launch (their pointers are kernel arguments)
constexpr int DS_MAX_M = 4;
constexpr int DS_MUL = 8, DS_DMA = 2, DS_COM = 6;      // waves that multiply, load and communicate
constexpr int DS_CLASSES = 3;                  // every third tile of a run: two for the multiplying waves, one for four of the communicating ones
constexpr int DS_THREADS = (DS_MUL + DS_DMA + DS_COM) * 64;
constexpr int DS_COM_THREADS = DS_COM * 64;
constexpr int DS_RING = 26;                    // tiles of the ring
constexpr int DS_BATCH = 4, DS_FLIGHT = 8;     // tiles that a loading wave issues at once; has on their way before it waits for some
constexpr int DS_TILE_LOADS = 5;               // vector-memory instructions of a tile
static_assert(DS_TILE_LOADS * (DS_FLIGHT + DS_BATCH - 1) < 64, "the counter of a wave's loads");
constexpr int DS_MAX_SLOTS = 17;               // tasks that contribute to one column unit, at most
constexpr int DS_MAX_SPLITS = 8;               // partials of one query, at most
constexpr int DS_SUMS = 256;                   // room for a row's sums of squares, one a task (at least DS_WGS)
constexpr int DS_PART = 132;                   // words of a partial: o[128], max, sum
constexpr int DS_LDS = 160 * 1024;
constexpr uint64_t DS_WAIT_LIMIT = 500000000; // 100 MHz: 5 s
constexpr int DS_JOIN_US = 50;                 // the first to sign in wait so long for the others

struct StackLayer {
    const uint8_t *w[7];                       // wq, wk, wv, wo, w1, w3, w2
    const half_t *att_norm, *ffn_norm, *prompt_k, *prompt_v;
    uint8_t *cache_k, *cache_v;
    half_t *cache_ks, *cache_vs;
};
// A linear's tiles, (unit, step) by (unit, step), in runs of `run`; each of its weights is `part` of them.
// (by_run, by_step: multiplied by them, the upper word of the product is the quotient by run and steps.)
struct StackLinear { int steps, run, tiles, part; uint32_t by_run, by_step; };
struct StackParams {
    StackLayer layer[DS_LAYERS];
    StackLinear lin[4];                        // wq|wk|wv, wo, w1|w3, w2
    const half_t *h_in;
    half_t *h_out;
    const half_t *cos_tab, *sin_tab;
    const int32_t *pos_dev, *t_dev, *pages;
    uint8_t *ws;
    long cache_rows;
    int workgroups, join_ticks;                // of the launch; DS_JOIN_US in ticks of 10 ns
    int layers, dim, ffn, heads, P, smax, pages_stride;
    int slices, slice_rows;                    // attention: the prompt's rows in `slices` tasks a head
    uint32_t by_att, by_red, by_act;           // quotients by the tasks of a head, by red_cols and by act_cols
    int red_cols, act_cols;                    // columns of a task that adds up wo / w2, and that makes SiLU(gate) * up
    int x_pitch;                               // halves of a row of activations in LDS
    float att_eps, ffn_eps;
};

// workspace: control words, then tagged words
struct StackSpace {
    uint32_t slab[4], h[2], ss[2], part, act, bytes;
};
__host__ __device__ inline StackSpace stack_space(int M, int dim, int ffn, int heads) {
    StackSpace s;
    uint32_t at = 1024;
    for (int i = 0; i < 4; ++i) { s.slab[i] = at; at += (uint32_t)DS_WGS * 2 * M * 256 * 8; }
    for (int i = 0; i < 2; ++i) { s.h[i] = at; at += (uint32_t)M * dim / 2 * 8; }
    for (int i = 0; i < 2; ++i) { s.ss[i] = at; at += (uint32_t)M * DS_SUMS * 8; }
    s.part = at;
    at += (uint32_t)M * heads * DS_MAX_SPLITS * DS_PART * 8;
    s.act = at;
    at += (uint32_t)M * ffn / 2 * 8;
    s.bytes = at;
    return s;
}

// LDS behind the rings: sums of the multiplying waves (also the attention's states), the attention's rows, activations, gates
struct StackLds { int red, q, x, misc, bytes; };
__host__ __device__ inline StackLds stack_lds(int M, int x_pitch) {
    StackLds s;
    s.red = DS_RING * TILE_BYTES;
    const int sums = 2 * DS_CLASSES * M * 256 * 4, states = M * DS_COM * 16 * 10 * 4;
    s.q = s.red + (sums > states ? sums : states);      // (written while slower waves still read the sums)
    s.x = s.q + (DS_MAX_M + 2) * 128 * 2;
    s.misc = s.x + (M * x_pitch * 2 + 15) / 16 * 16;
    s.bytes = s.misc + 256;
    return s;
}

typedef const __attribute__((address_space(1))) void *gptr_t;
typedef __attribute__((address_space(3))) void *lptr_t;

// The waves of a workgroup meet at counters in LDS (s_barrier would hold up the waves that load): whoever is due adds one, whoever
// needs it waits for the count.  A wave's own LDS operations are done when it adds.
struct Gates {
    uint32_t gave_up, x, sums, com;            // a wait was too long; arrivals: activations, sums of the multiplying waves, communicating waves
    float row_sums[DS_MAX_M][4];               // of squares: a row's in four parts
    uint32_t used[4 * DS_CLASSES];             // a wave's tiles below this one have been read; tiles are counted over the launch
    uint32_t landed[DS_DMA];                   // tiles that a loading wave has seen arrive
    int32_t n, id;
    uint32_t epoch;
};
__device__ __forceinline__ uint32_t lds_load(const uint32_t *p) {
    return (uint32_t)__builtin_amdgcn_readfirstlane((int)__hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
}
__device__ __forceinline__ void lds_store(uint32_t *p, uint32_t v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP); }
__device__ __forceinline__ void arrive(uint32_t *gate, int lane) {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (lane == 0) __hip_atomic_fetch_add(gate, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void wait_for(const uint32_t *gate, uint32_t count) {
    while ((int32_t)(lds_load(gate) - count) < 0) __builtin_amdgcn_s_sleep(1);
    asm volatile("" ::: "memory");
}
__device__ __forceinline__ uint64_t ticks() { return __builtin_amdgcn_s_memrealtime(); }
__device__ __forceinline__ float as_f(uint32_t v) { return __builtin_bit_cast(float, v); }
__device__ __forceinline__ int quotient(int x, uint32_t by) { return (int)__umulhi((uint32_t)x, by); }
// N words of every lane of the wave, at byte offsets of the workspace, once all of them carry the tag
template <int N>
__device__ __forceinline__ void get(const uint8_t *ws, const uint32_t (&off)[N], uint32_t tag, uint32_t (&out)[N], bool &late) {
    uint64_t since = 0;
    for (int tries = 0;; ++tries) {
        u32x2 v[N];
#pragma unroll
        for (int i = 0; i < N; ++i) {
            uint32_t o = off[i];
            asm volatile("" : "+v"(o));            // (made in front of the loop, the addresses would take twice the registers)
            v[i] = ld_u64(ws + o);
        }
        uint32_t differ = 0;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            out[i] = v[i][0];
            differ |= v[i][1] ^ tag;
        }
        if (late || __all(differ == 0u)) return;
        if ((tries & 63) == 63) {              // (reading the clock takes longer than a try)
            const uint64_t now = ticks();
            if (since == 0) since = now;
            else if (now - since > DS_WAIT_LIMIT) late = true;
        }
    }
}
// Sum over the 16 lanes of a group, over the wave, without the LDS where lanes allow it.
__device__ __forceinline__ float sum16(float v) {
    v += dpp_move<DPP_QUAD_XOR1>(v);
    v += dpp_move<DPP_QUAD_XOR2>(v);
    v += dpp_move<DPP_ROW_HALF_MIRROR>(v);
    return v + dpp_move<DPP_ROW_ROR8>(v);
}
__device__ __forceinline__ float sum64(float v) {
    v = sum16(v);
    v += __shfl_xor(v, 16, 64);
    return v + __shfl_xor(v, 32, 64);
}

// ---- the tasks that hold a column unit's products -----------------------------------------------------------------------
struct Slots { int first, count, piece; };     // the first task's piece that belongs to the unit; the others' is 0
__device__ __forceinline__ Slots slots_of(const StackLinear &L, int unit) {
    const int lo = unit * L.steps;
    Slots s;
    s.first = quotient(lo, L.by_run);
    s.count = quotient(lo + L.steps - 1, L.by_run) - s.first + 1;
    s.piece = s.first * L.run < lo ? 1 : 0;
    return s;
}
// byte offset of part i (past the end: the last one) of column `col`, row m of M, of a product
__device__ __forceinline__ uint32_t slab_word(uint32_t slab, const Slots &s, int i, int M, int m, int col) {
    const int k = min(i, s.count - 1), piece = k == 0 ? s.piece : 0;
    return slab + (uint32_t)((((s.first + k) * 2 + piece) * M + m) * 256 + (col & 255)) * 8u;
}
// Columns `col` of two products' rows m, added in task order; C words of each are in flight at a time.
template <int M, int C>
__device__ __forceinline__ void slab_columns(const uint8_t *ws, uint32_t slab, const StackLinear &L, int m, const int (&col)[2], uint32_t tag, float (&sum)[2],
                                             bool &late) {
    Slots s[2];
#pragma unroll
    for (int w = 0; w < 2; ++w) { s[w] = slots_of(L, col[w] >> 8); sum[w] = 0.f; }
    const int most = quotient(L.steps - 1, L.by_run) + 2;      // (enough for any unit)
    for (int c0 = 0; c0 < most; c0 += C) {
        uint32_t off[2 * C], v[2 * C];
#pragma unroll
        for (int w = 0; w < 2; ++w)
#pragma unroll
            for (int i = 0; i < C; ++i) off[w * C + i] = slab_word(slab, s[w], c0 + i, M, m, col[w]);
        get(ws, off, tag, v, late);
#pragma unroll
        for (int w = 0; w < 2; ++w)
#pragma unroll
            for (int i = 0; i < C; ++i) sum[w] += c0 + i < s[w].count ? as_f(v[w * C + i]) : 0.f;
    }
}

// ---- loading waves -----------------------------------------------------------------------------------------------------
struct StackWave {
    const StackParams &p;
    int id, n;                                 // this workgroup among those that take part
    int wave, lane;
};
__device__ __forceinline__ int run_len(const StackLinear &L, int task) { return min(L.run, L.tiles - task * L.run); }
template <int CTRL>
__device__ __forceinline__ uint32_t lane_move(uint32_t v) { return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, false); }
// LDS by hand: the compiler lets an access of its own wait for all loads to LDS that the wave has on their way.
__device__ __forceinline__ uint32_t lds_offset(const uint32_t *p) { return (uint32_t)(uintptr_t)p; }
__device__ __forceinline__ uint32_t lds_load_unordered(const uint32_t *p) {
    uint32_t v;
    asm volatile("ds_read_b32 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=v"(v) : "v"(lds_offset(p)) : "memory");
    return v;
}
__device__ __forceinline__ void lds_store_unordered(uint32_t *p, uint32_t v) {
    asm volatile("ds_write_b32 %0, %1" ::"v"(lds_offset(p)), "v"(v) : "memory");
}
// Two waves load the workgroup's tiles into the ring in turn - layer by layer, linear by linear, task by task - whenever all waves
// that read them have left room.  What bounds them is their own instructions (a scalar one takes a lone wave ~8 cycles: with a
// walk, a check and a wait a tile they took 0.9 us a tile and the layer 46 us), so they go by stretches of tiles that lie one
// behind the other and by up to DS_BATCH tiles at a time.
__device__ __forceinline__ void load_wave(const StackWave &s, uint8_t *lds, Gates *gates) {
    const StackParams &p = s.p;
    const uint32_t w_off = (uint32_t)(16 * s.lane), s_off = (uint32_t)(TILE_W_BYTES + 4 * s.lane);
    static_assert(DS_RING % DS_DMA == 0, "a wave's tiles stay in its slots");
    __builtin_amdgcn_s_setprio(3);
    int layer = 0, lin = 0, task = s.id - s.n, len = 0, tile0 = 0, j = s.wave;     // j: this wave's next tile of the run
    int left = 0;                                                                  // its tiles in the stretch, from ptr on
    const uint8_t *ptr = nullptr;
    bool more = true;
    uint32_t issued = 0, landed = 0, used = 0, tile_no = (uint32_t)s.wave;
    int slot = s.wave;
    for (;;) {
        if (left == 0 && more) {
            while (more && j >= len) {                                             // the next run
                j -= len;
                len = 0;
                task += s.n;
                if (task * p.lin[lin].run >= p.lin[lin].tiles) {
                    task = s.id - s.n;
                    const int wrap = lin == 3 ? 1 : 0;
                    lin = wrap ? 0 : lin + 1;
                    layer += wrap;
                    more = layer < p.layers;
                } else {
                    len = run_len(p.lin[lin], task);
                    tile0 = task * p.lin[lin].run;
                }
            }
            if (more) {
                // (no branches over the linears: one of those in here came out of the compiler with wo's address for w2)
                const int part = p.lin[lin].part, r = tile0 + j, first = 0x6430 >> 4 * lin & 15;
                const int which = (r >= part ? 1 : 0) + (r >= 2 * part ? 1 : 0);
                ptr = p.layer[layer].w[min(first + which, 6)] + (size_t)(r - which * part) * TILE_BYTES;
                const int end = min(len, (which + 1) * part - tile0);
                left = (end - j + DS_DMA - 1) / DS_DMA;
                j += left * DS_DMA;
            }
        }
        const int room = ((int)(used + DS_RING - tile_no) + DS_DMA - 1) / DS_DMA, n = more ? min(min(left, room), DS_BATCH) : 0;
        if (n > 0) {
            for (int i = 0; i < n; ++i) {
                uint8_t *stage = lds + slot * TILE_BYTES;
#pragma unroll
                for (int q = 0; q < 4; ++q) __builtin_amdgcn_global_load_lds((gptr_t)(ptr + q * 1024 + w_off), (lptr_t)(stage + q * 1024), 16, 0, 0);
                __builtin_amdgcn_global_load_lds((gptr_t)(ptr + s_off), (lptr_t)(stage + TILE_W_BYTES), 4, 0, 0);
                slot = slot + DS_DMA >= DS_RING ? s.wave : slot + DS_DMA;
                ptr += DS_DMA * TILE_BYTES;
            }
            issued += (uint32_t)n;
            tile_no += (uint32_t)(n * DS_DMA);
            left -= n;
            if (issued - landed < DS_FLIGHT) continue;
        }
        // loads to LDS end in the order they were issued
        if (issued - landed > DS_BATCH) {
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(DS_TILE_LOADS * DS_BATCH) : "memory");
            landed = issued - DS_BATCH;
        } else if (issued != landed) {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            landed = issued;
        } else if (!more) {
            return;
        } else {
            __builtin_amdgcn_s_sleep(1);
        }
        if (s.lane == 0) lds_store_unordered(&gates->landed[s.wave], landed);
        uint32_t u = lds_load_unordered(&gates->used[min(s.lane, 4 * DS_CLASSES - 1)]);
        u = min(u, lane_move<DPP_QUAD_XOR1>(u));
        u = min(u, lane_move<DPP_QUAD_XOR2>(u));
        u = min(u, lane_move<DPP_ROW_HALF_MIRROR>(u));
        u = min(u, lane_move<DPP_ROW_ROR8>(u));
        used = (uint32_t)__builtin_amdgcn_readfirstlane((int)u);
    }
}

// ---- multiplying -------------------------------------------------------------------------------------------------------
// Wave (piece q, class e) multiplies piece q (64 of a tile's 256 columns) of the tiles e, e + DS_CLASSES, .. of a run.  While it waits
// for the activations it holds its first AHEAD pieces in registers: as much room more in the ring.  DECODED of them it decodes there already, which leaves
// their products alone between the activations and the sums (us a step of the 7B architecture, five pieces, none decoded, and now, in turn: 1 branch behind 512
// rows 1435 and 1398, behind 2047 1612 and 1582, 2 branches behind 512 1586 and 1548; three of five pieces decoded 1398, 1588, 1555, four 1436, three of six,
// which spills, 1509).  From three branches on it gained nothing (1822 and 1830; 4: 2115 and 2145): five pieces, as they come.
template <int M, int AHEAD, int DECODED>
struct Multiplier {
    const StackParams &p;
    uint8_t *lds;
    Gates *gates;
    int piece, cls, lane;
    uint32_t first, landed0, landed1, x_due;   // the run's first tile; tiles known to be in LDS; arrivals at the gate of the activations
    struct Piece { u32x4 w, sh, sl; };

    __device__ __forceinline__ void await(uint32_t tile) {
        static_assert(DS_DMA == 2, "two loading waves");
        const uint32_t want = tile >> 1;
        if ((tile & 1) == 0) {
            while (landed0 <= want) {
                landed0 = lds_load(&gates->landed[0]);
                if (landed0 <= want) __builtin_amdgcn_s_sleep(1);
            }
        } else {
            while (landed1 <= want) {
                landed1 = lds_load(&gates->landed[1]);
                if (landed1 <= want) __builtin_amdgcn_s_sleep(1);
            }
        }
        asm volatile("" ::: "memory");
    }
    __device__ __forceinline__ Piece fetch(uint32_t tile) const {
        constexpr uint32_t BY_RING = (uint32_t)(((1ull << 32) + DS_RING - 1) / DS_RING);
        const uint8_t *stage = lds + (tile - __umulhi(tile, BY_RING) * DS_RING) * TILE_BYTES;
        const int s_off = TILE_W_BYTES + (lane >> 4) * 64 + (piece >> 1) * 32;
        Piece t;
        t.w = *reinterpret_cast<const u32x4 *>(stage + piece * 1024 + lane * 16);
        t.sh = *reinterpret_cast<const u32x4 *>(stage + s_off);
        t.sl = *reinterpret_cast<const u32x4 *>(stage + s_off + 16);
        return t;
    }
    __device__ __forceinline__ void release(uint32_t next) const {             // what was fetched is in registers
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (lane == 0) lds_store(&gates->used[4 * cls + piece], next);
    }
    // rows 4 g + r of the accumulators (column 4 c + 2 (q & 1) + half, nibble h); columns 128 blk + 64 h + 4 c + b
    __device__ __forceinline__ void flush(const StackLds &at, int pc, f4 (&acc)[2][2]) const {
        const int c = lane & 15, g = lane >> 4;
        float *dst = reinterpret_cast<float *>(lds + at.red) + ((pc * DS_CLASSES + cls) * M) * 256 + 128 * (piece >> 1) + 4 * c + 2 * (piece & 1);
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (4 * g + r < M) {
#pragma unroll
                for (int h = 0; h < 2; ++h) *reinterpret_cast<f2 *>(dst + (4 * g + r) * 256 + 64 * h) = f2{acc[0][h][r], acc[1][h][r]};
            }
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int h = 0; h < 2; ++h) acc[i][h] = f4{0.f, 0.f, 0.f, 0.f};
    }
    __device__ __forceinline__ void run(const StackLinear &L, int task, const StackLds &at) {
        const int c = lane & 15, g = lane >> 4;
        const half_t *xrow = reinterpret_cast<const half_t *>(lds + at.x) + min(c, M - 1) * p.x_pitch + 8 * g;
        // constants of the decoder the compiler cannot see through (q40_gemv.hip)
        uint32_t mask_hi = 0x00F000F0u, mask_lo = 0x000F000Fu, magic_hi = 0x54005400u, magic_lo = 0x64006400u;
        const h2 off_hi = {(half_t)-72.f, (half_t)-72.f}, off_lo = {(half_t)-1032.f, (half_t)-1032.f};
        asm volatile("" : "+s"(mask_hi), "+s"(mask_lo));
        asm volatile("" : "+v"(magic_hi), "+v"(magic_lo));
        const int len = run_len(L, task), r0 = task * L.run;
        const int cut = L.steps - (r0 - quotient(r0, L.by_step) * L.steps);     // tiles of the run before the next unit
        f4 acc[2][2];
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int h = 0; h < 2; ++h) acc[i][h] = f4{0.f, 0.f, 0.f, 0.f};
        int pc = 0, j = cls;
        auto decode = [&](const Piece &t, int half, u32x4 &vh, u32x4 &vl) {
            const uint32_t pr[4] = {t.w[2 * half], t.w[2 * half + 1], t.w[2 * half] >> 8, t.w[2 * half + 1] >> 8};
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                vh[k] = as_u32((as_h2((pr[k] & mask_hi) | magic_hi) + off_hi) * as_h2(t.sh[k]));
                vl[k] = as_u32((as_h2((pr[k] & mask_lo) | magic_lo) + off_lo) * as_h2(t.sl[k]));
            }
        };
        auto product = [&](int half, const u32x4 &vh, const u32x4 &vl, const h8 &xv) {
            acc[half][0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xv, __builtin_bit_cast(h8, vh), acc[half][0], 0, 0, 0);
            acc[half][1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xv, __builtin_bit_cast(h8, vl), acc[half][1], 0, 0, 0);
        };
        auto multiply = [&](const Piece &t, const h8 &xv) {
#pragma unroll
            for (int half = 0; half < 2; ++half) {
                u32x4 vh, vl;
                decode(t, half, vh, vl);
                product(half, vh, vl, xv);
            }
        };
        auto next = [&](int i) { return first + (uint32_t)(i < len ? i : len + cls); };      // this wave's tile at or behind i of the run
        auto cross = [&]() {                                                   // into the next unit
            if (pc == 0 && j >= cut) {
                flush(at, 0, acc);
                pc = 1;
            }
        };
        Piece pre[AHEAD];
#pragma unroll
        for (int u = 0; u < AHEAD; ++u)
            if (j + u * DS_CLASSES < len) {
                await(first + j + u * DS_CLASSES);
                pre[u] = fetch(first + j + u * DS_CLASSES);
            }
        release(next(j + AHEAD * DS_CLASSES));
        u32x4 ready[DECODED + 1][2][2];
#pragma unroll
        for (int u = 0; u < DECODED; ++u)
            if (j + u * DS_CLASSES < len) {
#pragma unroll
                for (int half = 0; half < 2; ++half) {
                    decode(pre[u], half, ready[u][half][0], ready[u][half][1]);
                    asm volatile("" : "+v"(ready[u][half][0]), "+v"(ready[u][half][1]));       // (here, not where it is needed)
                }
            }
        x_due += DS_COM;
        wait_for(&gates->x, x_due);
        Piece cur = pre[0];
#pragma unroll
        for (int u = 0; u < AHEAD; ++u)
            if (j < len) {
                cross();
                const h8 xv = *reinterpret_cast<const h8 *>(xrow + j * 32);
                const bool another = u == AHEAD - 1 && j + DS_CLASSES < len;   // the loop's first tile
                if (another) {
                    await(first + j + DS_CLASSES);
                    cur = fetch(first + j + DS_CLASSES);
                }
                if (u < DECODED) {
#pragma unroll
                    for (int half = 0; half < 2; ++half) product(half, ready[u][half][0], ready[u][half][1], xv);
                } else {
                    multiply(pre[u], xv);
                }
                j += DS_CLASSES;
                if (another) release(next(j + DS_CLASSES));
            }
        while (j < len) {
            cross();
            const h8 xv = *reinterpret_cast<const h8 *>(xrow + j * 32);
            const bool another = j + DS_CLASSES < len;
            Piece nxt = cur;
            if (another) {                                                     // the next tile is read under this one's decoding
                await(first + j + DS_CLASSES);
                nxt = fetch(first + j + DS_CLASSES);
            }
            multiply(cur, xv);
            j += DS_CLASSES;
            if (another) release(next(j + DS_CLASSES));
            cur = nxt;
        }
        if (pc == 0 && cut < len) {                                            // (a wave may have no tile of the second unit)
            flush(at, 0, acc);
            pc = 1;
        }
        flush(at, pc, acc);
        release(next(len));                                                    // (a run may have no tile for it)
        first += (uint32_t)len;
        arrive(&gates->sums, lane);
    }
};

template <int M>
__device__ __forceinline__ void multiply_waves(const StackWave &s, uint8_t *lds, Gates *gates) {
    const StackParams &p = s.p;
    const StackLds at = stack_lds(M, p.x_pitch);
    Multiplier<M, M <= 2 ? 6 : 5, M <= 2 ? 2 : 0> mul{p, lds, gates, s.wave & 3, s.wave >> 2, s.lane, 0u, 0u, 0u, 0u};
    for (int layer = 0; layer < p.layers; ++layer)
        for (int lin = 0; lin < 4; ++lin) {
            const StackLinear L = p.lin[lin];
            for (int task = s.id; task * L.run < L.tiles; task += s.n) mul.run(L, task, at);
        }
}

// ---- communicating waves ---------------------------------------------------------------------------------------------------
// A softmax in parts, base 2.  A score of -infinity weighs nothing; a part without rows has the maximum -infinity.
// (Which products become fused is written out: the compiler chose otherwise for one branch than for the next.)
__device__ __forceinline__ void soft_fold(float &m, float &l, float (&o)[8], float m2, float l2, const float (&o2)[8]) {
#pragma clang fp contract(off)
    const float m_new = fmaxf(m, m2);
    if (m_new == -INFINITY) return;
    const float c1 = __builtin_amdgcn_exp2f(m - m_new), c2 = __builtin_amdgcn_exp2f(m2 - m_new);
    m = m_new;
    l = fmaf(l, c1, l2 * c2);
#pragma unroll
    for (int j = 0; j < 8; ++j) o[j] = fmaf(o[j], c1, o2[j] * c2);
}
__device__ __forceinline__ float dot_row(const RowRegs &k, const RowRegs &q) {
    float d = __builtin_amdgcn_fdot2(k.a02, q.a02, 0.f, false);
    d = __builtin_amdgcn_fdot2(k.a13, q.a13, d, false);
    d = __builtin_amdgcn_fdot2(k.b02, q.b02, d, false);
    d = __builtin_amdgcn_fdot2(k.b13, q.b13, d, false);
    return sum16(d);
}
__device__ __forceinline__ void soft_row(SoftState &st, float score, const RowRegs &v) {
#pragma clang fp contract(off)
    const float m_new = fmaxf(st.m, score), m_ref = m_new == -INFINITY ? 0.f : m_new;
    const float corr = __builtin_amdgcn_exp2f(st.m - m_ref), pr = __builtin_amdgcn_exp2f(score - m_ref);
    st.m = m_new;
    st.l = fmaf(st.l, corr, pr);
    st.o[0] = fmaf(pr, (float)v.a02.x, st.o[0] * corr);
    st.o[1] = fmaf(pr, (float)v.a02.y, st.o[1] * corr);
    st.o[2] = fmaf(pr, (float)v.a13.x, st.o[2] * corr);
    st.o[3] = fmaf(pr, (float)v.a13.y, st.o[3] * corr);
    st.o[4] = fmaf(pr, (float)v.b02.x, st.o[4] * corr);
    st.o[5] = fmaf(pr, (float)v.b02.y, st.o[5] * corr);
    st.o[6] = fmaf(pr, (float)v.b13.x, st.o[6] * corr);
    st.o[7] = fmaf(pr, (float)v.b13.y, st.o[7] * corr);
}

template <int M>
struct StackCom {
    const StackParams &p;
    int id, n;
    int wave, lane, tid;                       // among the communicating waves
    uint32_t tag;                              // of the layer
    uint8_t *lds;
    Gates *gates;
    StackLds at;
    StackSpace sp;
    bool late;
    uint32_t met, sums_due;                    // counts of the gates
    Multiplier<M, 1, 0> mul;                      // of the first four waves
    int t_now;                                 // the step's suffix index and, of this lane's dims, its rotation
    half_t cos_l, sin_l;

    __device__ __forceinline__ void put(uint32_t off, uint32_t v, uint32_t tag_) const { st_u64(p.ws + off, u32x2{v, tag_}); }
    __device__ __forceinline__ void put_f(uint32_t off, float v, uint32_t tag_) const { put(off, __builtin_bit_cast(uint32_t, v), tag_); }
    __device__ __forceinline__ int first_step(const StackLinear &L, int task) const { const int r = task * L.run; return r - quotient(r, L.by_step) * L.steps; }
    // A workgroup one of whose waves has given up publishes nothing more.
    __device__ __forceinline__ void note_late() const {
        if (late && lane == 0) lds_store(&gates->gave_up, 1u);
    }
    __device__ __forceinline__ bool silent() const { return late || lds_load(&gates->gave_up) != 0u; }
    // Addresses of a phase are made in it: left alone the compiler makes all phases' in front of the loop over the layers and spills them.
    __device__ __forceinline__ void phase() {
        asm volatile("" : "+v"(lane), "+v"(tid));
        asm volatile("" : "+s"(id), "+s"(wave));
    }
    __device__ __forceinline__ void meet() {
        arrive(&gates->com, lane);
        met += DS_COM;
        wait_for(&gates->com, met);
    }
    __device__ __forceinline__ void hand_over() {          // the activations to the multiplying waves
        note_late();
        arrive(&gates->x, lane);
    }

    // activations of a run: pairs of columns of tagged words [M][K / 2], to LDS; NORM: RMSNorm with the row's sum of squares
    template <bool NORM>
    __device__ __forceinline__ void take(uint32_t src, uint32_t ss, const StackLinear &L, int K, int task, int len, const half_t *weight, float eps, int red_tasks) {
        constexpr int N = 2 * M, S = NORM ? (M * DS_SUMS + DS_COM_THREADS - 1) / DS_COM_THREADS : 0;
        const int per_row = len * 16, total = M * per_row, k_first = first_step(L, task) * 32;
        half_t *xs = reinterpret_cast<half_t *>(lds + at.x);
        for (int i0 = 0; i0 < total; i0 += N * DS_COM_THREADS) {
            uint32_t off[N + S], v[N + S], wv[N];
            int to[N], row[N];
#pragma unroll
            for (int i = 0; i < N; ++i) {
                const int idx = min(i0 + i * DS_COM_THREADS + tid, total - 1);         // (past the end: the last one again)
                const int m = (M > 1 && idx >= per_row) + (M > 2 && idx >= 2 * per_row) + (M > 3 && idx >= 3 * per_row), j = 2 * (idx - m * per_row);
                int k = k_first + j;
                k -= k >= K ? K : 0;
                off[i] = src + (uint32_t)(m * K + k) * 4u;
                wv[i] = NORM ? *reinterpret_cast<const uint32_t *>(weight + k) : 0u;
                to[i] = m * p.x_pitch + j;
                row[i] = m;
            }
#pragma unroll
            for (int i = 0; i < S; ++i) {                      // a row's sums of squares, 64 at a time
                const int idx = i * DS_COM_THREADS + tid;
                off[N + i] = ss + (uint32_t)(min(idx >> 8, M - 1) * DS_SUMS + min(idx & 255, red_tasks - 1)) * 8u;
            }
            get(p.ws, off, tag, v, late);
            if (NORM && i0 == 0) {
#pragma unroll
                for (int i = 0; i < S; ++i) {
                    const int idx = i * DS_COM_THREADS + tid;
                    const float sum = sum64((idx & 255) < red_tasks ? as_f(v[N + i]) : 0.f);
                    if (lane == 0 && (idx >> 8) < M) gates->row_sums[idx >> 8][(idx >> 6) & 3] = sum;
                }
                meet();
            }
            float r[M];
            if (NORM) {
#pragma unroll
                for (int m = 0; m < M; ++m) {
                    const float *four = gates->row_sums[m];
                    r[m] = rms_factor(((four[0] + four[1]) + four[2]) + four[3], K, eps);
                }
            }
#pragma unroll
            for (int i = 0; i < N; ++i) {
                uint32_t out = v[i];
                if (NORM) {
                    float f = r[0];
#pragma unroll
                    for (int m = 1; m < M; ++m) f = row[i] == m ? r[m] : f;
                    const h2 h = as_h2(v[i]), wt = as_h2(wv[i]);
                    const h2 y = {scale_to_half(h.x, f), scale_to_half(h.y, f)};
                    out = as_u32(y * wt);
                }
                *reinterpret_cast<uint32_t *>(xs + to[i]) = out;
            }
        }
        hand_over();
    }

    // the attention's output for the rows of a run of wo: the partials of a head added up
    __device__ __forceinline__ void take_attention(const StackLinear &L, int task, int len) {
        const int K = p.heads * 128, per_row = len * 32, total = M * per_row, splits = p.slices + 1, k_first = first_step(L, task) * 32;
        half_t *xs = reinterpret_cast<half_t *>(lds + at.x);
        for (int i0 = 0; i0 < total; i0 += DS_COM_THREADS) {
            const int idx = min(i0 + tid, total - 1);                      // (half a wave: the 32 rows of a tile, so of one head)
            const int m = (M > 1 && idx >= per_row) + (M > 2 && idx >= 2 * per_row) + (M > 3 && idx >= 3 * per_row), j = idx - m * per_row;
            int k = k_first + j;
            k -= k >= K ? K : 0;
            const uint32_t part = sp.part + (uint32_t)((m * p.heads + (k >> 7)) * splits * DS_PART) * 8u;
            uint32_t off[DS_MAX_SPLITS + 1], v[DS_MAX_SPLITS + 1];
#pragma unroll
            for (int i = 0; i < DS_MAX_SPLITS; ++i) off[i] = part + (uint32_t)(min(i, splits - 1) * DS_PART + (k & 127)) * 8u;
            off[DS_MAX_SPLITS] = part + (uint32_t)(min(lane & 15, splits - 1) * DS_PART + 128 + ((lane >> 4) & 1)) * 8u;
            get(p.ws, off, tag, v, late);
            float mx = -INFINITY, ms[DS_MAX_SPLITS], l = 0.f, o = 0.f;
#pragma unroll
            for (int i = 0; i < DS_MAX_SPLITS; ++i) {
                const float mi = as_f(__shfl((int)v[DS_MAX_SPLITS], (lane & 32) + i, 64));
                ms[i] = i < splits ? mi : -INFINITY;
                mx = fmaxf(mx, ms[i]);
            }
            const float m_ref = mx == -INFINITY ? 0.f : mx;
#pragma unroll
            for (int i = 0; i < DS_MAX_SPLITS; ++i) {
                const float li = as_f(__shfl((int)v[DS_MAX_SPLITS], (lane & 32) + 16 + i, 64));
                if (i < splits) {
                    const float f = __builtin_amdgcn_exp2f(ms[i] - m_ref);
                    l = fmaf(f, li, l);
                    o = fmaf(f, as_f(v[i]), o);
                }
            }
            const float inv = l > 0.f ? 1.0f / l : 0.f;
            xs[m * p.x_pitch + j] = (half_t)(o * inv);
        }
        hand_over();
    }

    // the multiplying waves' sums of a task
    __device__ __forceinline__ void publish(uint32_t slab, const StackLinear &L, int task, int len) {
        if (wave < 4) {
            __builtin_amdgcn_s_setprio(2);             // (its eight elders would leave it for last)
            mul.run(L, task, at);
            __builtin_amdgcn_s_setprio(0);
        }
        sums_due += 4 * DS_CLASSES;
        wait_for(&gates->sums, sums_due);
        if (silent()) return;
        const int pieces = L.steps - first_step(L, task) < len ? 2 : 1;
        const float *red = reinterpret_cast<const float *>(lds + at.red);
        const uint32_t dst = slab + (uint32_t)(task * 2 * M * 256) * 8u;
        for (int idx = tid; idx < pieces * M * 256; idx += DS_COM_THREADS) {
            const int in = idx + (idx >= M * 256 ? (DS_CLASSES - 1) * M * 256 : 0);
            put_f(dst + (uint32_t)idx * 8u, red[in] + (red[in + M * 256] + red[in + 2 * M * 256]), tag);
        }
    }

    // h += a linear's product (slab, or nothing before the first layer): wave m adds up row m of a task's columns, 16, 32 or 64
    // lanes side by side and as many parts of the product at a time as that leaves lanes for
    __device__ __forceinline__ void residual(int lin, bool first, bool last, uint32_t h_from, uint32_t h_to, uint32_t ss_to, uint32_t to_tag) {
        if (wave >= M) return;
        constexpr int U = 5;
        const StackLinear &L = p.lin[lin];
        const int m = wave, tasks = quotient(p.dim + p.red_cols - 1, p.by_red), wide = p.red_cols <= 16 ? 4 : p.red_cols <= 32 ? 5 : 6, groups = 64 >> wide;
        const int c_ = lane & ((1 << wide) - 1), grp = lane >> wide;
        for (int task = id; task < tasks; task += n) {
            const int col = min(task * p.red_cols + min(c_, p.red_cols - 1), p.dim - 1);
            const bool mine = c_ < p.red_cols && task * p.red_cols + c_ < p.dim && grp == 0;
            half_t h;
            if (first) {
                h = p.h_in[(size_t)m * p.dim + col];
            } else {
                const Slots at_ = slots_of(L, col >> 8);
                float sum = 0.f;
                uint32_t old = 0;
                for (int c0 = 0; c0 < DS_MAX_SLOTS; c0 += U * groups) {
                    uint32_t off[U + 1], v[U + 1];
#pragma unroll
                    for (int i = 0; i < U; ++i) off[i] = slab_word(sp.slab[lin], at_, c0 + i * groups + grp, M, m, col);
                    off[U] = h_from + (uint32_t)(m * p.dim + col) / 2u * 8u;
                    get(p.ws, off, tag, v, late);
#pragma unroll
                    for (int i = 0; i < U; ++i) sum += c0 + i * groups + grp < at_.count ? as_f(v[i]) : 0.f;
                    old = v[U];
                }
                if (groups >= 2) sum += __shfl_xor(sum, 32, 64);
                if (groups >= 4) sum += __shfl_xor(sum, 16, 64);
                const h2 pair = as_h2(old);
                h = (half_t)((float)((col & 1) ? pair.y : pair.x) + (float)(half_t)sum);
            }
            const float ss = sum64(mine ? (float)h * (float)h : 0.f);
            const uint32_t bits = __builtin_bit_cast(uint16_t, h), next = (uint32_t)__shfl_down((int)bits, 1, 64);
            uint32_t both = bits | next << 16;
            note_late();
            const bool bad = silent();
            if (last) {
                if (bad) both = 0x7e007e00u;                               // NaN
                if (mine && (lane & 1) == 0) *reinterpret_cast<uint32_t *>(p.h_out + (size_t)m * p.dim + col) = both;
            } else if (!bad) {
                if (mine && (lane & 1) == 0) put(h_to + (uint32_t)(m * p.dim + col) * 4u, both, to_tag);
                if (lane == 0) put_f(ss_to + (uint32_t)(m * DS_SUMS + task) * 8u, ss, to_tag);
            }
        }
    }

    // SiLU(gate) * up of a task's columns
    __device__ __forceinline__ void activate() {
        const bool two = p.act_cols > 64;                                  // waves a row
        const int m = two ? wave >> 1 : wave, part = two ? wave & 1 : 0;
        if (m >= M) return;
        const int tasks = quotient(p.ffn + p.act_cols - 1, p.by_act);
        for (int task = id; task < tasks; task += n) {
            const int in = 64 * part + lane, c0 = min(task * p.act_cols + min(in, p.act_cols - 1), p.ffn - 1);
            const bool mine = in < p.act_cols && task * p.act_cols + in < p.ffn;
            const int col[2] = {c0, p.ffn + c0};
            float sum[2];
            slab_columns<M, 5>(p.ws, sp.slab[2], p.lin[2], m, col, tag, sum, late);
            const float gf = (float)(half_t)sum[0];
            const half_t a = (half_t)(gf / (1.0f + expf(-gf))) * (half_t)sum[1];
            const uint32_t bits = __builtin_bit_cast(uint16_t, a), next = (uint32_t)__shfl_down((int)bits, 1, 64);
            note_late();
            const bool bad = silent();
            if (mine && (lane & 1) == 0 && !bad) put(sp.act + (uint32_t)(m * p.ffn + c0) * 4u, bits | next << 16, tag);
        }
    }

    // q, k or v of one head and branch, rotated (lane: dims lane and lane + 64)
    __device__ __forceinline__ void head_row(int m, int col0, half_t &x1, half_t &x2) {
        const int col[2] = {col0 + lane, col0 + 64 + lane};
        float sum[2];
        slab_columns<M, 7>(p.ws, sp.slab[0], p.lin[0], m, col, tag, sum, late);
        x1 = (half_t)sum[0];
        x2 = (half_t)sum[1];
    }

    // One attention task: a slice of the prompt for all branches' queries of a head, or a branch's own rows and its new token.
    // A row belongs to 16 lanes (attn_rows.hpp); the waves take four rows each in turn.  The first rows are requested while the
    // multiplying waves are at wq|wk|wv (request).
    static constexpr int PASSES = 4, STEP = 4 * DS_COM;        // passes over the waves whose rows wait in registers; rows of a pass
    struct Row { u32x2 kl, kh, vl, vh; };                      // own rows: kl bytes of k and v, kh their scales
    struct Rows { Row r0, r1, r2, r3; };
    struct Task { bool prefix; int hk, b, split, t0, rows; };  // b: of an own-rows task
    __device__ __forceinline__ Task att_task(int task) const {
        const int hk = quotient(task, p.by_att), js = task - hk * (p.slices + M);
        const bool prefix = js < p.slices;
        const int t0 = js * p.slice_rows;
        return Task{prefix, hk, js - p.slices, prefix ? js : p.slices, prefix ? t0 : 0, max(0, prefix ? min(p.slice_rows, p.P - t0) : min(t_now, p.smax))};
    }
    __device__ __forceinline__ Row att_row(const StackLayer &Y, const Task &T, int pass) const {
        const int c = lane & 15, g = lane >> 4, t = min(STEP * pass + 4 * wave + g, T.rows - 1);
        Row r;
        if (T.prefix) {
            const size_t off = ((size_t)(T.t0 + t) * p.heads + T.hk) * 128 + 4 * c;
            r.kl = *reinterpret_cast<const u32x2 *>(Y.prompt_k + off);
            r.kh = *reinterpret_cast<const u32x2 *>(Y.prompt_k + off + 64);
            r.vl = *reinterpret_cast<const u32x2 *>(Y.prompt_v + off);
            r.vh = *reinterpret_cast<const u32x2 *>(Y.prompt_v + off + 64);
        } else {
            long row = (long)T.b * p.smax + t;
            if (p.pages != nullptr) row = min(max((long)p.pages[(long)T.b * p.pages_stride + t], 0L), p.cache_rows - 1);
            const size_t at_ = (size_t)row * p.heads + T.hk;
            r.kl = u32x2{*reinterpret_cast<const uint32_t *>(Y.cache_k + at_ * 64 + 4 * c), *reinterpret_cast<const uint32_t *>(Y.cache_v + at_ * 64 + 4 * c)};
            r.kh = u32x2{*reinterpret_cast<const uint32_t *>(Y.cache_ks + at_ * 2), *reinterpret_cast<const uint32_t *>(Y.cache_vs + at_ * 2)};
            r.vl = r.vh = u32x2{0, 0};
        }
        return r;
    }
    // (one by one: in a loop the rows end up in memory)
    __device__ __forceinline__ void request(const StackLayer &Y, const Task &T, int first, Rows &r) const {
        if (STEP * first >= T.rows) return;
        r.r0 = att_row(Y, T, first);
        r.r1 = att_row(Y, T, first + 1);
        r.r2 = att_row(Y, T, first + 2);
        r.r3 = att_row(Y, T, first + 3);
    }
    __device__ __forceinline__ void att_use(const Task &T, int pass, Row r, const RowRegs (&q)[M], SoftState (&st)[M]) const {
        if (STEP * pass >= T.rows) return;                                     // (uniform)
        const bool in = STEP * pass + 4 * wave + (lane >> 4) < T.rows;         // a repeated row weighs nothing, also where it is infinite
        RowRegs k, v;
        if (T.prefix) {
            if (!in) r.vl = r.vh = u32x2{0, 0};
            k.a02 = as_h2(pack_lo16(r.kl[0], r.kl[1])); k.a13 = as_h2(pack_hi16(r.kl[0], r.kl[1]));
            k.b02 = as_h2(pack_lo16(r.kh[0], r.kh[1])); k.b13 = as_h2(pack_hi16(r.kh[0], r.kh[1]));
            v.a02 = as_h2(pack_lo16(r.vl[0], r.vl[1])); v.a13 = as_h2(pack_hi16(r.vl[0], r.vl[1]));
            v.b02 = as_h2(pack_lo16(r.vh[0], r.vh[1])); v.b13 = as_h2(pack_hi16(r.vh[0], r.vh[1]));
        } else {
            // us a step of the 7B architecture behind 128 rows, 60 of their own, masks in registers and as literals: 3 branches 1751 and 1775, 4 2045 and 2030
            if constexpr (M == 4) {
                k = row_from_q40(r.kl[0], r.kh[0]);
                v = row_from_q40(r.kl[1], r.kh[1]);
            } else {
                const RowCodes codes;
                k = row_from_q40(r.kl[0], r.kh[0], codes);
                v = row_from_q40(r.kl[1], r.kh[1], codes);
            }
            if (!in) v.a02 = v.a13 = v.b02 = v.b13 = h2{(half_t)0.f, (half_t)0.f};
        }
#pragma unroll
        for (int m = 0; m < M; ++m)
            if (m == 0 || T.prefix) {
                const float sc = dot_row(k, q[m]) * SCALE_LOG2;
                soft_row(st[m], in ? sc : -INFINITY, v);
            }
    }
    static constexpr float SCALE_LOG2 = 1.4426950408889634f * 0.08838834764831845f;
    __device__ __forceinline__ void attention(const StackLayer &Y, const Task &T, Rows &cur) {
        const int H = p.heads, hk = T.hk, b = T.b;
        const int c = lane & 15, g = lane >> 4;
        const bool prefix = T.prefix;
        float *fold = reinterpret_cast<float *>(lds + at.red);                                        // [M][waves][16][10]
        half_t *sq = reinterpret_cast<half_t *>(lds + at.q);                                          // [M] queries, k, v
        half_t *skv = sq + DS_MAX_M * 128;
        SoftState st[M];
#pragma unroll
        for (int m = 0; m < M; ++m) {
            st[m].m = -INFINITY;
            st[m].l = 0.f;
#pragma unroll
            for (int j = 0; j < 8; ++j) st[m].o[j] = 0.f;
        }
        // the new token's rows: the branches' queries, or one branch's query, k and v
        if (wave < (prefix ? M : 3)) {
            half_t x1, x2;
            head_row(prefix ? wave : b, prefix ? hk * 128 : (wave * H + hk) * 128, x1, x2);
            if (prefix || wave < 2) rope_pair2(x1, x2, cos_l, sin_l);
            half_t *dst = prefix || wave == 0 ? sq + wave * 128 : skv + (wave - 1) * 128;
            dst[lane] = x1;
            dst[64 + lane] = x2;
            if (!prefix && wave > 0 && t_now >= 0 && t_now < p.smax && !late) {
                const size_t row = ((size_t)b * p.smax + t_now) * H + hk;
                kv_store_row2(x1, x2, (wave == 1 ? Y.cache_k : Y.cache_v) + row * 64, (wave == 1 ? Y.cache_ks : Y.cache_vs) + row * 2, lane);
            }
        }
        note_late();
        meet();
        const int nq = prefix ? M : 1;
        RowRegs q[M];
#pragma unroll
        for (int m = 0; m < M; ++m) q[m] = row_from_fp16(sq + m * 128, c);
        for (int i = 0; i * STEP < T.rows; i += PASSES) {
            if (i > 0) request(Y, T, i, cur);
            att_use(T, i, cur.r0, q, st);
            att_use(T, i + 1, cur.r1, q, st);
            att_use(T, i + 2, cur.r2, q, st);
            att_use(T, i + 3, cur.r3, q, st);
        }
        if (!prefix && wave == 0) {                                        // the new token itself, by one of the wave's groups
            const float sc = dot_row(row_from_fp16(skv, c), q[0]) * SCALE_LOG2;
            if (g == 0) soft_row(st[0], sc, row_from_fp16(skv + 128, c));
        }
        // the four groups of a wave, then the waves
#pragma unroll
        for (int m = 0; m < M; ++m)
            if (m < nq) {
#pragma unroll
                for (int sh = 16; sh <= 32; sh <<= 1) {
                    const float m2 = __shfl_xor(st[m].m, sh, 64), l2 = __shfl_xor(st[m].l, sh, 64);
                    float o2[8];
#pragma unroll
                    for (int j = 0; j < 8; ++j) o2[j] = __shfl_xor(st[m].o[j], sh, 64);
                    soft_fold(st[m].m, st[m].l, st[m].o, partial_max(m2, l2), l2, o2);
                }
                if (g == 0) {
                    float *dst = fold + ((m * DS_COM + wave) * 16 + c) * 10;
                    dst[0] = partial_max(st[m].m, st[m].l);
                    dst[1] = st[m].l;
#pragma unroll
                    for (int j = 0; j < 8; ++j) dst[2 + j] = st[m].o[j];
                }
            }
        meet();
        if (wave < nq) {
            // group g: waves g and, where there is one, g + 4
            float mm, l, o[8];
            const float *src = fold + ((wave * DS_COM + g) * 16 + c) * 10;
            mm = src[0]; l = src[1];
#pragma unroll
            for (int j = 0; j < 8; ++j) o[j] = src[2 + j];
            if (g + 4 < DS_COM) {
                src += 4 * 160;
                const float o4[8] = {src[2], src[3], src[4], src[5], src[6], src[7], src[8], src[9]};
                soft_fold(mm, l, o, src[0], src[1], o4);
            }
#pragma unroll
            for (int sh = 16; sh <= 32; sh <<= 1) {
                const float m2 = __shfl_xor(mm, sh, 64), l2 = __shfl_xor(l, sh, 64);
                float o2[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) o2[j] = __shfl_xor(o[j], sh, 64);
                soft_fold(mm, l, o, partial_max(m2, l2), l2, o2);
            }
            if (!silent()) {
                const int row = prefix ? wave : b, split = T.split;
                const uint32_t dst = sp.part + (uint32_t)(((row * H + hk) * (p.slices + 1) + split) * DS_PART) * 8u;
                // every group has the merged state: group g leaves o[2 g], o[2 g + 1] (dims 4 c + g', 4 c + g' + 2, the upper half's for g >= 2)
                const float a = g == 0 ? o[0] : g == 1 ? o[2] : g == 2 ? o[4] : o[6], b_ = g == 0 ? o[1] : g == 1 ? o[3] : g == 2 ? o[5] : o[7];
                const uint32_t d = dst + (uint32_t)((g >> 1) * 64 + 4 * c + (g & 1)) * 8u;
                put_f(d, a, tag);
                put_f(d + 16, b_, tag);
                if (lane < 2) put_f(dst + (uint32_t)(128 + lane) * 8u, lane == 0 ? partial_max(mm, l) : l, tag);
            }
        }
    }

    __device__ __forceinline__ void run(uint32_t epoch) {
        const int red_tasks = quotient(p.dim + p.red_cols - 1, p.by_red), att_tasks = p.heads * (p.slices + M);
        const int pos = *p.pos_dev;
        t_now = *p.t_dev;
        cos_l = p.cos_tab[(size_t)pos * 64 + lane];
        sin_l = p.sin_tab[(size_t)pos * 64 + lane];
        tag = epoch + 1;
        residual(3, true, false, 0, sp.h[0], sp.ss[0], tag);
        for (int layer = 0; layer < p.layers; ++layer) {
            const StackLayer &Y = p.layer[layer];
            tag = epoch + 1 + (uint32_t)layer;
            Rows ahead;
            phase();
            for (int task = id; task * p.lin[0].run < p.lin[0].tiles; task += n) {
                const int len = run_len(p.lin[0], task);
                take<true>(sp.h[0], sp.ss[0], p.lin[0], p.dim, task, len, Y.att_norm, p.att_eps, red_tasks);
                phase();
                if (task == id && id < att_tasks) request(Y, att_task(id), 0, ahead);
                publish(sp.slab[0], p.lin[0], task, len);
            }
            phase();
            for (int task = id; task < att_tasks; task += n) {
                const Task T = att_task(task);
                if (task != id || id * p.lin[0].run >= p.lin[0].tiles) request(Y, T, 0, ahead);
                attention(Y, T, ahead);
            }
            phase();
            for (int task = id; task * p.lin[1].run < p.lin[1].tiles; task += n) {
                const int len = run_len(p.lin[1], task);
                take_attention(p.lin[1], task, len);
                phase();
                publish(sp.slab[1], p.lin[1], task, len);
            }
            phase();
            residual(1, false, false, sp.h[0], sp.h[1], sp.ss[1], tag);
            phase();
            for (int task = id; task * p.lin[2].run < p.lin[2].tiles; task += n) {
                const int len = run_len(p.lin[2], task);
                take<true>(sp.h[1], sp.ss[1], p.lin[2], p.dim, task, len, Y.ffn_norm, p.ffn_eps, red_tasks);
                phase();
                publish(sp.slab[2], p.lin[2], task, len);
            }
            phase();
            activate();
            phase();
            for (int task = id; task * p.lin[3].run < p.lin[3].tiles; task += n) {
                const int len = run_len(p.lin[3], task);
                take<false>(sp.act, 0, p.lin[3], p.ffn, task, len, nullptr, 0.f, 0);
                phase();
                publish(sp.slab[3], p.lin[3], task, len);
            }
            phase();
            residual(3, false, layer + 1 == p.layers, sp.h[1], sp.h[0], sp.ss[0], tag + 1);
        }
    }
};

template <int M>
__global__ __launch_bounds__(DS_THREADS) void decode_stack_kernel(StackParams p) {
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const StackLds at = stack_lds(M, p.x_pitch);
    uint32_t *ctl = reinterpret_cast<uint32_t *>(p.ws);         // [0] the list: count, closed at (<< 12), closed (bit 31); [64] left; [128] epoch
    Gates *gates = reinterpret_cast<Gates *>(lds + at.misc);
    const int tid = threadIdx.x;
    constexpr uint32_t CLOSED = 1u << 31;
    if (tid < (int)(sizeof(Gates) / 4)) reinterpret_cast<uint32_t *>(gates)[tid] = 0u;
    __syncthreads();
    if (tid == 0) {
        const uint32_t old = __hip_atomic_fetch_add(ctl, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if ((old & CLOSED) == 0) {
            const uint64_t since = ticks();
            uint32_t v = ld_u32(ctl);
            while ((v & CLOSED) == 0) {
                if ((v & 0xfff) == (uint32_t)p.workgroups || ticks() - since > (uint64_t)p.join_ticks) {
                    const uint32_t closed = v | CLOSED | (v & 0xfff) << 12;
                    uint32_t want = v;
                    if (__hip_atomic_compare_exchange_strong(ctl, &want, closed, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) v = closed;
                    else v = want;
                } else {
                    v = ld_u32(ctl);
                }
            }
            const int n = (int)((v >> 12) & 0xfff);
            gates->n = n;
            gates->id = n == p.workgroups ? (int)blockIdx.x : (int)(old & 0xfff);
            gates->epoch = ld_u32(ctl + 128);
        }
    }
    __syncthreads();
    const int n = __builtin_amdgcn_readfirstlane(gates->n), id = __builtin_amdgcn_readfirstlane(gates->id);
    const uint32_t epoch = (uint32_t)__builtin_amdgcn_readfirstlane((int)gates->epoch);
    if (n > 0) {
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        if (wave < DS_MUL) {
            multiply_waves<M>(StackWave{p, id, n, wave, tid & 63}, lds, gates);
        } else if (wave < DS_MUL + DS_DMA) {
            load_wave(StackWave{p, id, n, wave - DS_MUL, tid & 63}, lds, gates);
        } else {
            constexpr int first = DS_MUL + DS_DMA;
            StackCom<M> com{p, id, n, wave - first, tid & 63, tid - first * 64, 0u, lds, gates, at, stack_space(M, p.dim, p.ffn, p.heads), false, 0u, 0u,
                            Multiplier<M, 1, 0>{p, lds, gates, (wave - first) & 3, 2, tid & 63, 0u, 0u, 0u, 0u}, 0, (half_t)0.f, (half_t)0.f};
            com.run(epoch);
        }
    }
    __syncthreads();
    if (tid == 0 && __hip_atomic_fetch_add(ctl + 64, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (uint32_t)p.workgroups - 1) {
        // the last one out: nobody reads these any more, and the next launch starts behind this one
        const uint32_t e = ld_u32(ctl + 128);
        st_u32(ctl, 0u);
        st_u32(ctl + 64, 0u);
        st_u32(ctl + 128, e + (uint32_t)p.layers + 1u);
    }
}

// ---- host -------------------------------------------------------------------------------------------------------------
static uint32_t divisor(int d) { return (uint32_t)(((1ull << 32) + d - 1) / d); }      // exact for x * d < 2^32
static bool stack_linear(int K, int weights, int columns, StackLinear &L) {
    L.steps = K / 32;
    L.part = columns / 256 * L.steps;
    L.tiles = weights * L.part;
    const int tiles = L.tiles;
    L.run = (tiles + DS_WGS - 1) / DS_WGS;
    const int least = (L.steps + DS_MAX_SLOTS - 2) / (DS_MAX_SLOTS - 1);      // a unit's tiles in at most DS_MAX_SLOTS runs
    if (L.run < least) L.run = least;
    if (L.run < 2) L.run = 2;                                                 // (quotients by 1 do not fit the word)
    L.by_run = divisor(L.run);
    L.by_step = divisor(L.steps);
    return L.run <= L.steps;                                                  // a run touches two units at most
}
// Fills everything that follows from the sizes; false: this shape is not for the kernel.
static bool stack_plan(const smh_layer &L, int M, StackParams &p) {
    if (M < 1 || M > DS_MAX_M || L.heads != L.kv_heads || L.heads % 2 != 0 || L.dim % 256 != 0 || L.ffn % 256 != 0 || L.heads < 1 || L.dim < 256 || L.ffn < 256)
        return false;
    const int nq = L.heads * 128;
    if (!stack_linear(L.dim, 3, nq, p.lin[0]) || !stack_linear(nq, 1, L.dim, p.lin[1]) || !stack_linear(L.dim, 2, L.ffn, p.lin[2]) ||
        !stack_linear(L.ffn, 1, L.dim, p.lin[3]))
        return false;
    p.dim = L.dim;
    p.ffn = L.ffn;
    p.heads = L.heads;
    p.red_cols = ((L.dim + DS_WGS - 1) / DS_WGS + 1) & ~1;
    p.act_cols = ((L.ffn + DS_WGS - 1) / DS_WGS + 1) & ~1;
    if (p.red_cols > 64 || p.act_cols > 128 || M * (p.act_cols > 64 ? 2 : 1) > DS_COM) return false;
    int longest = 0;
    for (const StackLinear &l : p.lin) longest = l.run > longest ? l.run : longest;
    p.x_pitch = longest * 32 + 8;
    if (stack_lds(M, p.x_pitch).bytes > DS_LDS) return false;
    p.P = L.prompt_len;
    int slices = DS_WGS / L.heads - M;
    if (slices > DS_MAX_SPLITS - 1) slices = DS_MAX_SPLITS - 1;
    if (slices < 1) return false;
    if (slices > (p.P + 31) / 32) slices = p.P > 0 ? (p.P + 31) / 32 : 1;
    p.slices = slices;
    p.slice_rows = (p.P + slices - 1) / slices;
    p.by_att = divisor(slices + M);
    p.by_red = divisor(p.red_cols);
    p.by_act = divisor(p.act_cols);
    return true;
}

}  // namespace smh

using namespace smh;

extern "C" size_t smh_decode_stack_workspace_bytes(const smh_layer *layer, int rows) {
    static_assert(sizeof(StackParams) <= 4096, "kernel arguments");
    StackParams p;
    if (layer == nullptr || !stack_plan(*layer, rows, p)) return 0;
    return stack_space(rows, layer->dim, layer->ffn, layer->heads).bytes;
}

// Why a pass over these layers is not for the kernel, null: it is.  Alignments are those of its loads (the weights' of the DMA into LDS),
// looked at layer by layer, for tensors may be views: the layers' own launches take what is refused here.
static const char *stack_refuses(const smh_layer *const *layers, int n_layers, int rows, StackParams &p) {
    if (layers == nullptr || n_layers < 1) return "no layers";
    for (int i = 0; i < n_layers; ++i)
        if (layers[i] == nullptr) return "a layer is null";
    const smh_layer &L0 = *layers[0];
    if (!stack_plan(L0, rows, p)) return "its rows, heads or widths are not for this call";
    for (int i = 0; i < n_layers; ++i) {
        const smh_layer &L = *layers[i];
        if (L.dim != L0.dim || L.ffn != L0.ffn || L.heads != L0.heads || L.kv_heads != L0.kv_heads) return "layers of different sizes";
        if (L.prompt_len < 0) return "a negative prompt length";
        auto bad = [](const void *q, int align) { return q == nullptr || (uintptr_t)q % align != 0; };
        for (const void *q : {L.wq, L.wk, L.wv, L.wo, L.w1, L.w2, L.w3})
            if (bad(q, 16)) return "a weight is null or not 16-byte aligned";
        for (const void *q : {L.prompt_k, L.prompt_v})
            if (L.prompt_len > 0 && bad(q, 8)) return "a prompt cache is null or not 8-byte aligned";
        for (const void *q : {(const void *)L.cache_k, (const void *)L.cache_v, (const void *)L.cache_ks, (const void *)L.cache_vs, L.att_norm, L.ffn_norm})
            if (bad(q, 4)) return "a cache or the weight of a norm is null or not 4-byte aligned";
    }
    return nullptr;
}

extern "C" int smh_decode_stack_fits(const smh_layer *const *layers, int n_layers, int rows) {
    StackParams p;
    return stack_refuses(layers, n_layers, rows, p) == nullptr ? 1 : 0;
}

extern "C" int smh_decode_stack(const smh_layer *const *layers, int n_layers, smh_pass *pass, void *ws, size_t ws_bytes, smh_stream_t stream) {
    return smh_decode_stack_of(layers, n_layers, pass, ws, ws_bytes, DS_WGS, DS_JOIN_US, stream);
}

extern "C" int smh_decode_stack_of(const smh_layer *const *layers, int n_layers, smh_pass *pass, void *ws, size_t ws_bytes, int workgroups, int join_us,
                                   smh_stream_t stream) {
    const char *who = "smh_decode_stack";
    SMH_REQUIRE(workgroups >= 1 && workgroups <= DS_WGS && join_us >= 0 && join_us <= 1000000, "%s: workgroups=%d (1 .. %d) join_us=%d (up to a second)", who,
                workgroups, DS_WGS, join_us);
    SMH_REQUIRE(pass && pass->h && ws, "%s: null pointer", who);
    StackParams p;
    const char *why = stack_refuses(layers, n_layers, pass->rows, p);
    SMH_REQUIRE(why == nullptr, "%s: %s (%d rows)", who, why, pass->rows);
    const smh_layer &L0 = *layers[0];
    SMH_REQUIRE(pass->pos_dev && pass->t_dev && pass->cos_tab && pass->sin_tab && pass->smax >= 1, "%s: the step's tables and counters are missing", who);
    const size_t need = stack_space(pass->rows, p.dim, p.ffn, p.heads).bytes;
    SMH_REQUIRE(ws_bytes >= need, "%s: workspace %zu < %zu bytes", who, ws_bytes, need);
    const size_t rows_bytes = ((size_t)pass->rows * p.dim * 2 + 255) & ~(size_t)255;
    SMH_REQUIRE(pass->scratch && pass->scratch_bytes >= 2 * rows_bytes, "%s: scratch %zu < %zu bytes", who, pass->scratch_bytes, 2 * rows_bytes);
    SMH_REQUIRE(pass->pending == 0, "%s: a product is pending", who);
    SMH_REQUIRE(pass->pages == nullptr || (pass->pages_stride >= pass->smax && pass->cache_rows >= 1), "%s: pages_stride=%ld must cover the %d rows of a branch",
                who, (long)pass->pages_stride, pass->smax);
    p.cos_tab = (const half_t *)pass->cos_tab;
    p.sin_tab = (const half_t *)pass->sin_tab;
    p.pos_dev = pass->pos_dev;
    p.t_dev = pass->t_dev;
    p.pages = pass->pages;
    p.pages_stride = pass->pages_stride;
    p.cache_rows = pass->cache_rows;
    p.smax = pass->smax;
    p.ws = (uint8_t *)ws;
    p.workgroups = workgroups;
    p.join_ticks = join_us * 100;
    // more than 64 KB of dynamic LDS has to be allowed once (not stream work: fine under graph capture)
    static void (*const kernels[DS_MAX_M])(StackParams) = {decode_stack_kernel<1>, decode_stack_kernel<2>, decode_stack_kernel<3>, decode_stack_kernel<4>};
    static const hipError_t lds_ok = [] {
        hipError_t e = hipSuccess;
        for (auto *k : kernels)
            if (e == hipSuccess) e = hipFuncSetAttribute((const void *)k, hipFuncAttributeMaxDynamicSharedMemorySize, DS_LDS);
        return e;
    }();
    if (lds_ok != hipSuccess) {
        set_error("%s: the kernel's LDS could not be reserved: %s", who, hipGetErrorString(lds_ok));
        return (int)lds_ok;
    }
    for (int l0 = 0; l0 < n_layers;) {
        const smh_layer &A = *layers[l0];
        int count = 0;
        while (l0 + count < n_layers && count < DS_LAYERS) {
            const smh_layer &L = *layers[l0 + count];
            // (the first one always: a NaN differs from itself)
            if (count > 0 && (L.att_eps != A.att_eps || L.ffn_eps != A.ffn_eps || L.prompt_len != A.prompt_len)) break;
            p.layer[count++] = StackLayer{{(const uint8_t *)L.wq, (const uint8_t *)L.wk, (const uint8_t *)L.wv, (const uint8_t *)L.wo, (const uint8_t *)L.w1,
                                           (const uint8_t *)L.w3, (const uint8_t *)L.w2}, (const half_t *)L.att_norm, (const half_t *)L.ffn_norm,
                                          (const half_t *)L.prompt_k, (const half_t *)L.prompt_v, (uint8_t *)L.cache_k, (uint8_t *)L.cache_v,
                                          (half_t *)L.cache_ks, (half_t *)L.cache_vs};
        }
        if (!stack_plan(A, pass->rows, p)) return -1;           // (the prompt's slices)
        char *out = (char *)pass->scratch + (pass->h == pass->scratch ? rows_bytes : 0);
        p.h_in = (const half_t *)pass->h;
        p.h_out = (half_t *)out;
        p.att_eps = A.att_eps;
        p.ffn_eps = A.ffn_eps;
        p.layers = count;
        hipLaunchKernelGGL(kernels[pass->rows - 1], dim3((unsigned)workgroups), dim3(DS_THREADS), (size_t)stack_lds(pass->rows, p.x_pitch).bytes, (hipStream_t)stream, p);
        if (int st = launch_status()) return st;
        pass->h = out;
        l0 += count;
    }
    return 0;
}
