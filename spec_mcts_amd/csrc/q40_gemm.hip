// Q4_0 dequant + matmul for large batches (decode at B = 100, prefill): c[M,N] = a[M,K] . deq(W)[K,N].
//
// A workgroup of 4 waves (8 plus two that only issue DMA in launches with one workgroup per compute unit, and 8 on tiled weights,
// see the kernel) owns 128 rows of A, two adjacent 128-column blocks of the weight (one full 128-byte line of
// packed nibbles per k) and a slice of K - or, under a range cut, a run of steps that may end one column unit and begin
// the next; up to two workgroups share a compute unit.  Everything a 32-row step needs - 4 KB of nibbles, 256 B of scales, the 128 x 32 tile of A -
// goes global -> LDS by DMA (global_load_lds) into a 6-slot ring shared by the workgroup; one bare s_barrier
// per TWO steps both publishes stages and frees the oldest ones.  (__syncthreads() would wait for every
// outstanding DMA first, because they write LDS, and so empty the ring at every barrier.)
//   * wave w decodes TWO byte positions of ONE block (block w/2, bytes 2(w%2) and 2(w%2)+1 of every
//     dword): perm pairs the byte of two consecutive rows, and-or drops the nibbles into fp16
//     mantissas, one packed op recovers the exact code and one packed multiply applies the scales -
//     the value the reference's dequantiser produces, born in the B-operand layout of
//     v_mfma_f32_16x16x32_f16, so dequantised weights never travel through LDS or HBM;
//   * it multiplies its four B operands (2 byte positions x high / low nibbles = columns c and c+64)
//     with all TILES 16-row tiles of A, read from LDS through an XOR swizzle (GS_A): one read of the A tile feeds four MFMAs;
//   * the step is software-pipelined inside the wave: while the matrix pipe works through step i,
//     the vector ALU decodes the B operands of step i+1 (one basic block, no branches: the number of
//     row tiles and the ragged-K handling are template parameters), and the DMA addresses are a
//     scalar base per step plus lane offsets that never change, so issuing a stage costs no VALU work;
//   * the accumulators leave through LDS one row tile at a time, so global stores are 64-byte
//     contiguous per lane; K-slices are written as fp32 slabs and added by the consuming kernel.
//
// At M = 100 the work sits on the ridge of the roofline: 2*M*N*K flops against
// N*K*0.53125 + 2*M*(K+N) bytes.
#include <type_traits>
#include <utility>

#include "q40_warm.hpp"

namespace smh {

// most K-slices of a launch = GEMM_KSCAP / rows (every slice leaves an fp32 slab of rows x columns)
constexpr int GEMM_KSCAP = 1600;
constexpr int GEMM_BM = 128;
constexpr int GEMM_WAVES = 4;                  // ragged K, and the checkpoint layout where workgroups share compute units; the rest runs GEMM_TILED_WAVES
constexpr int GEMM_TILED_WAVES = 8;
constexpr int GEMM_THREADS = GEMM_WAVES * 64;
// slots of the DMA ring (with a barrier per step, four slots measured 2 % faster per launch at M=100 than six; with a
// barrier per two steps, six slots are 3 % faster than that)
constexpr int GEMM_STAGES = 6;
// slots of the ring in the variant with DMA waves, by row tiles, and the most workgroups of a launch that takes it (one per
// compute unit).  Up to 48 rows a step is over before its successors have come from memory: wq|wk|wv at 37 rows of the 7B shape takes 13.6 us with
// six slots, 12.8 with eight and with twelve.  At 64 rows and more six are as good or better (wo, w2 at 512 rows 36.9, 37.4 and 37.7 us with six, eight and ten).
constexpr int gemm_dma_slots(int tiles) { return tiles <= 3 ? 8 : 6; }
// slots of the kernels whose stages hold two steps: up to `most`, as many as fit.  w1|w3 at 37 rows of the 7B shape 25.5 us with six, 21.6 with eight,
// 22.0 with twelve; at 100 rows 30.0, 29.6.  The K-sliced kernel: at 37 rows 9.2 and 9.0, at 100 rows, where a slice has few stages, 16.6 and 17.0;
// nine to twelve slots are within 0.3 % of eight from 5 to 48 rows.
constexpr int gemm_slots(int stage, int most) { return 160 * 1024 / stage < most ? 160 * 1024 / stage : most; }
constexpr int GEMM_DMA_WAVE_MAX_WGS = 256;
constexpr int GS_WBLOCK = 8 * 128 + 64;        // the 8 rows one wave fetches, padded by 16 banks: the four row groups a
                                               // ds_read_b32 touches (lanes 16g..16g+15 read row 8g+r) then sit in different banks
constexpr int GS_W = 4 * GS_WBLOCK;            // nibbles
constexpr int GS_S = 32 * 8;                   // scales
// A tile, 64 B per row; the 16-byte chunk k of row r lies at k ^ ((r / 2) % 4): a wave's 16 rows x 64 B by k-octet then reach 480 - 520 GB/s
// a compute unit, with (r / 4) % 4 280 - 295.  (In turn: eight steps of 100 branches 33.67 -> 32.98 ms, prefill of 512 rows 9.44 -> 9.35 ms,
// of 2047 rows 31.16 -> 30.86, 100 x 11008 x 4096 25.7 -> 25.3 us.)
constexpr int GS_A = GEMM_BM * 64;
constexpr int GS_BYTES = GS_W + GS_S + GS_A;               // 12800
constexpr int GEMM_LDS = GEMM_STAGES * GS_BYTES;           // 76800
constexpr int GEMM_COLS = 256;

typedef const __attribute__((address_space(1))) void *gptr_t;
typedef __attribute__((address_space(3))) void *lptr_t;


// Waits until at most N DMA instructions of this wave are still in flight (the counter has six bits).
template <int N>
__device__ __forceinline__ void gemm_wait_vm() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N < 63 ? N : 63) : "memory"); }
// ... at most `stages` younger stages of PER DMA instructions each (4 with four waves, 2 with eight, 5 + row tiles in
// a DMA wave at most).  A ring of eight slots asks for MOST = 5, one of eleven for eight.
template <int PER, int MOST = 5>
__device__ __forceinline__ void gemm_wait_dma(int stages) {
    if constexpr (MOST > 5) {
        static_assert(MOST <= 8, "a case each");
        switch (stages) {
            case 8: return gemm_wait_vm<8 * PER>();
            case 7: return gemm_wait_vm<7 * PER>();
            case 6: return gemm_wait_vm<6 * PER>();
        }
    }
    switch (stages) {
        case 5: gemm_wait_vm<5 * PER>(); break;
        case 4: gemm_wait_vm<4 * PER>(); break;
        case 3: gemm_wait_vm<3 * PER>(); break;
        case 2: gemm_wait_vm<2 * PER>(); break;
        case 1: gemm_wait_vm<1 * PER>(); break;
        default: gemm_wait_vm<0>(); break;              // (waits for more than asked)
    }
}

// A bare workgroup barrier.  Every LDS read this wave has issued has returned (lgkmcnt), so after the
// barrier no wave still reads the stage that is refilled next.
__device__ __forceinline__ void gemm_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// A DMA wave: it issues PER instructions of each of n stages (issue(slot): the next stage's) into a ring of SLOTS slots, waits for them and meets
// the multiplying waves at their barriers, one per pair of stages (the protocol: gemm_piece).
// A workgroup has GEMM_DMA_WAVES of these, each with a share of every stage.  One wave gets an instruction (1 KB) out every 32 - 40 cycles, two or more
// together every 16, whatever rows the pieces lie in (measured from L2): with one, 22 instructions a stage of w1|w3 at 100 rows of
// the 7B shape took 885 cycles, the same with the products taken out; with two 815, and 52 200 cycles for the 64 stages instead of 56 600.
constexpr int GEMM_DMA_WAVES = 2;
template <int PER, int SLOTS, class Issue>
__device__ __forceinline__ void gemm_feed(int n, Issue issue) {
    if (n <= 0) return;
#pragma unroll 1
    for (int i = 0; i < min(SLOTS - 2, n); ++i) issue(i);
    gemm_wait_dma<PER, SLOTS - 3>(min(SLOTS - 3, n - 1));
    gemm_barrier();
    int slot = 0;
    auto back = [&](int k) { return slot >= k ? slot - k : slot + SLOTS - k; };
    int i = 0;
#pragma unroll 1
    for (; i + SLOTS - 1 < n; i += 2) {
        gemm_wait_vm<PER * (SLOTS - 5)>();
        gemm_barrier();
        issue(back(2));
        issue(back(1));
        slot = slot + 2 >= SLOTS ? slot + 2 - SLOTS : slot + 2;
    }
#pragma unroll 1
    for (; i < n; i += 2) {
        gemm_wait_dma<PER, SLOTS - 3>(max(0, min(n - 1, i + SLOTS - 3) - (i + 2)));      // stages issued past stage i + 2
        gemm_barrier();
        if (i + SLOTS - 2 < n) issue(back(2));
        if (i + SLOTS - 1 < n) issue(back(1));
        slot = slot + 2 >= SLOTS ? slot + 2 - SLOTS : slot + 2;
    }
}
template <int N> using int_constant = std::integral_constant<int, N>;
// f(int_constant<0>) .. f(int_constant<N - 1>)
template <int N, class F>
__device__ __forceinline__ void static_for(F f) {
    if constexpr (N > 0) {
        static_for<N - 1>(f);
        f(int_constant<N - 1>{});
    }
}

// What a multiplying wave reads of a stage's weights, and its operands out of that (gemm_decode): rows (2 j, 2 j + 1) of the piece's first
// (o = 0) or second byte, the nibble (high: hh = 0, low) as fp16 code * scale.
struct NibbleConsts {
    uint32_t mask, magic;
    h2 mul, off;
    // flip: bits that turn a two's complement nibble into code + 8
    __device__ __forceinline__ NibbleConsts(int hh, uint32_t flip)
        : mask(hh == 0 ? 0x00F000F0u : 0x000F000Fu), magic(MAGIC_1024 ^ flip),
          mul(hh == 0 ? h2{(half_t)0.0625f, (half_t)0.0625f} : h2{(half_t)1.0f, (half_t)1.0f}),
          off(hh == 0 ? h2{(half_t)-72.0f, (half_t)-72.0f} : h2{(half_t)-1032.0f, (half_t)-1032.0f}) {
        asm volatile("" : "+v"(magic));        // in a register the compiler cannot see through: (bits & mask) | magic is then ONE
    }                                          // v_and_or_b32 (no literal operands there), not an AND and an OR
    __device__ __forceinline__ h2 code(uint32_t bits) const { return __builtin_elementwise_fma(as_h2(bits), mul, off); }
};
struct TiledWeights {
    static constexpr int READS = 2;            // LDS instructions of a load
    NibbleConsts nib;
    int w_off, s_off;
    __device__ __forceinline__ TiledWeights(int hh, int w, int s) : nib(hh, 0), w_off(w), s_off(s) {}
    struct Regs { u32x4 w, scales; };
    __device__ __forceinline__ Regs load(const uint8_t *st, int) const {
        return Regs{*reinterpret_cast<const u32x4 *>(st + w_off), *reinterpret_cast<const u32x4 *>(st + s_off)};
    }
    __device__ __forceinline__ uint32_t bits(const Regs &r, int j, int o) const {
        const uint32_t w = r.w[(j & 1) + 2 * o], pr = j < 2 ? w : w >> 8;
        return (pr & nib.mask) | nib.magic;
    }
    __device__ __forceinline__ h2 scale(const Regs &r, int j) const { return as_h2(r.scales[j]); }
};
// Checkpoint layout: row 8 g + r of a stage (GS_WBLOCK) and its scales (of the block's first, second 64 columns in a dword).
// RAGGED: stage `last` is the end of K, where `dead` says that this lane's rows lie past it (their scales become zero).
// BLOCK (q40_gemm_kg_kernel): rows of 64 bytes in the order (r, g), so that the four rows of a read lie in different banks; scales row by row.
// (With reads that were waited for where they were issued, in us, before and now: 42 / 75 / 100 rows x 26880 x 9704 61.2 / 81.8 / 76.8 and 52.0 / 63.7 / 75.9,
// 75 x 4096 x 11008 21.5 and 19.9, 100 x 11008 x 4096 23.9 and 23.2, 300 x 11008 x 4096 59 and 46.)
template <bool RAGGED, bool BLOCK = false>
struct RowWeights {
    static constexpr int READS = BLOCK ? 6 : 8;            // (pairs of dwords; a block's scales: four dwords)
    static constexpr int PITCH = BLOCK ? 256 : 128;
    NibbleConsts nib;
    int w_off, s_off;
    uint32_t sel, half;                        // picks the first byte of two rows; the scales of the nibble
    int last;
    bool dead;
    __device__ __forceinline__ RowWeights(int hh, int w, int s, uint32_t byte, int last_, bool dead_)
        : nib(hh, hh == 0 ? 0x00800080u : 0x00080008u), w_off(w), s_off(s), sel(byte), half(hh == 0 ? 0x05040100u : 0x07060302u), last(last_), dead(dead_) {}
    struct Regs { uint32_t w[8], s[8], keep; };
    __device__ __forceinline__ Regs load(const uint8_t *st, int stage) const {
        Regs x;
        x.keep = RAGGED && stage == last && dead ? 0u : ~0u;
#pragma unroll
        for (int r = 0; r < 8; ++r) x.w[r] = *reinterpret_cast<const uint32_t *>(st + w_off + r * PITCH);
        if constexpr (BLOCK) {
            const u32x4 lo = *reinterpret_cast<const u32x4 *>(st + s_off), hi = *reinterpret_cast<const u32x4 *>(st + s_off + 16);
#pragma unroll
            for (int r = 0; r < 4; ++r) { x.s[r] = lo[r]; x.s[4 + r] = hi[r]; }
        } else {
#pragma unroll
            for (int r = 0; r < 8; ++r) x.s[r] = *reinterpret_cast<const uint32_t *>(st + s_off + r * 8);
        }
        return x;
    }
    __device__ __forceinline__ uint32_t bits(const Regs &x, int j, int o) const {
        const uint32_t pr = __builtin_amdgcn_perm(x.w[2 * j + 1], x.w[2 * j], o == 0 ? sel : sel + 0x00010001u);
        return (pr & nib.mask) ^ nib.magic;
    }
    __device__ __forceinline__ h2 scale(const Regs &x, int j) const {
        const uint32_t pair = __builtin_amdgcn_perm(x.s[2 * j + 1], x.s[2 * j], half);
        return as_h2(RAGGED ? pair & x.keep : pair);
    }
};

// A stage's B operands, one kind of instruction after the other: a packed product that reads the result of the packed fma before it waits (the compiler puts
// an s_nop between them), and a row pair at a time had one such wait each.  The checkpoint layout's, whose sixteen dwords of rows arrive one after the other, go
// as the compiler orders them (like the others 37 x 11008 x 4096 16.9 us and 16.5, 48 rows 17.6 and 17.2, 80 rows 21.3 and 20.9).
template <class Weights, class Regs>
__device__ __forceinline__ void gemm_decode(const Weights &weights, const Regs &w, u32x4 (&b)[2]) {
    if constexpr (Weights::READS > 2) {
#pragma unroll
        for (int u = 0; u < 8; ++u) b[u & 1][u >> 1] = as_u32(weights.nib.code(weights.bits(w, u >> 1, u & 1)) * weights.scale(w, u >> 1));
        return;
    }
    uint32_t bits[8];
    h2 scale[4], code[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) bits[u] = weights.bits(w, u >> 1, u & 1);
#pragma unroll
    for (int j = 0; j < 4; ++j) scale[j] = weights.scale(w, j);
    // (all of them, not one by one where the fma needs it)
    asm volatile("" : "+v"(bits[0]), "+v"(bits[1]), "+v"(bits[2]), "+v"(bits[3]), "+v"(bits[4]), "+v"(bits[5]), "+v"(bits[6]), "+v"(bits[7]));
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < 8; ++u) code[u] = weights.nib.code(bits[u]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < 8; ++u) b[u & 1][u >> 1] = as_u32(code[u] * scale[u >> 1]);
}

// The products of one multiplying wave of the kernels below: n stages of a ring of SLOTS slots, B operands (one nibble of one piece, 16 columns of either
// byte) x TILES row tiles.  A wave keeps the A rows and the B operands of ONE stage in registers.  As soon as a row tile's two products are
// issued its registers take the next stage's rows, and the next nibbles, read first, are decoded behind the last product: no read is waited for where it
// was issued.  Left to the compiler each pair of products waited for its own read - with the products 780 cycles a stage of 112 rows x 128 columns x 64,
// 448 of them on the matrix pipe.  (Decoded between the products, row pair by row pair, us before and now: tiled weights, 512 x 4096 x 11008 45.6 and 43.9,
// 2047 rows 155 and 149, SwiGLU at 2047 rows 339 and 335, wo at 100 rows 9.16 and 8.95.  In the middle of the products in half of the waves, so that some
// decode while others multiply: level or up to 6 % slower.)
// PRIO: GEMM_PRODUCTS_FIRST where two waves a SIMD share it, GEMM_DECODE_FIRST where three do (us without and with: SwiGLU at 128 rows 32.7 and 31.6, at 100
// 29.5 and 28.9; at 512 rows 91.6 and 90.0, at 2047 353 and 349; the 256-column units are level).
// Stages go in pairs, one barrier a pair (gemm_feed): at the barrier before stages i, i + 1 the stages up to i + 2 have landed, whose rows
// and nibbles stage i + 1 reads; past the last stage stale bytes are read, decoded and never used.
// Not AHEAD: a stage's rows are read in it, and the compiler puts reads and decode where it likes.
enum { GEMM_EVEN, GEMM_PRODUCTS_FIRST, GEMM_DECODE_FIRST };
template <int TILES, int SLOTS, int STAGE, int PRIO = GEMM_EVEN, bool AHEAD = true, class Weights>
__device__ __forceinline__ void gemm_multiply(const uint8_t *lds, int n, const Weights &weights, int a_off, f4 (&acc)[2][TILES]) {
#pragma unroll
    for (int o = 0; o < 2; ++o)
#pragma unroll
        for (int t = 0; t < TILES; ++t) acc[o][t] = f4{0.f, 0.f, 0.f, 0.f};
    if (n <= 0) return;
    h8 av[TILES];
    u32x4 bq[2];
    gemm_barrier();
    {
        const auto w = weights.load(lds, 0);
        if constexpr (AHEAD) {
#pragma unroll
            for (int t = 0; t < TILES; ++t) av[t] = *reinterpret_cast<const h8 *>(lds + a_off + t * 1024);
        }
        gemm_decode(weights, w, bq);
    }
    if constexpr (PRIO == GEMM_PRODUCTS_FIRST) __builtin_amdgcn_s_setprio(1);
    int slot = 0;
    auto one_stage = [&](int next) {
        const uint8_t *here = lds + slot * STAGE;
        slot = slot == SLOTS - 1 ? 0 : slot + 1;
        const uint8_t *st = lds + slot * STAGE;                // of the next stage
        if constexpr (!AHEAD) {
            u32x4 bn[2];
#pragma unroll
            for (int t = 0; t < TILES; ++t) av[t] = *reinterpret_cast<const h8 *>(here + a_off + t * 1024);
            const auto w = weights.load(st, next);
#pragma unroll
            for (int t = 0; t < TILES; ++t)
#pragma unroll
                for (int o = 0; o < 2; ++o) acc[o][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av[t], __builtin_bit_cast(h8, bq[o]), acc[o][t], 0, 0, 0);
            gemm_decode(weights, w, bn);
            bq[0] = bn[0];
            bq[1] = bn[1];
            return;
        }
        const auto w = weights.load(st, next);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
#pragma unroll
            for (int o = 0; o < 2; ++o) acc[o][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av[t], __builtin_bit_cast(h8, bq[o]), acc[o][t], 0, 0, 0);
            av[t] = *reinterpret_cast<const h8 *>(st + a_off + t * 1024);
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (PRIO != GEMM_EVEN) __builtin_amdgcn_s_setprio(PRIO == GEMM_DECODE_FIRST ? 1 : 0);
        gemm_decode(weights, w, bq);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (PRIO != GEMM_EVEN) __builtin_amdgcn_s_setprio(PRIO == GEMM_DECODE_FIRST ? 0 : 1);
    };
    // The slots that are refilled behind a barrier were read a stage ago, by reads older than the last stage's TILES + READS
    auto meet = [] {
        if constexpr (!AHEAD) return gemm_barrier();
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_waitcnt lgkmcnt(%0)\n\ts_barrier" ::"n"(TILES + Weights::READS < 15 ? TILES + Weights::READS : 15) : "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    int i = 0;
#pragma unroll 1
    for (; i + 1 < n; i += 2) {
        meet();
        one_stage(i + 1);
        one_stage(i + 2);
    }
    if (i < n) {
        meet();
        one_stage(i + 1);
    }
}

// TILED: the weights are in the tiled layout (q40_matmul.hpp).  Wave w then moves and decodes piece w of a
// tile (its two byte positions of its block, already paired by rows): one 16-byte LDS read instead of eight
// dword reads, shifts instead of byte permutes, the scales already in operand order; rows past K hold zeros.
// WAVES = 8: waves w and w + 4 share piece w of a tile; wave w multiplies the columns of its HIGH
// nibbles, wave w + 4 those of the low nibbles (two B operands and half the accumulators each, the same A tiles), so
// that every SIMD holds two waves of the workgroup and the decode of one runs under the MFMAs of the other.
//
// One piece of a workgroup's work: steps [step0, step1) of column unit `unit` (row block mb), accumulated and left as slab
// `slice`.  zero_rest: the piece ends its unit, and the slabs past `slice` (the unit has no piece for them) are written as
// zeros.  more: another piece follows in this workgroup (one more barrier, after which the ring may be refilled).
// tid_bias: zero (a range cut passes one the compiler cannot see, see there).
// SWIGLU (eight waves, tiled): unit j is 128-column block j of the gate weight (seg[0], pieces 0 and 1 of a stage) next to block
// j of the up weight (seg[1], pieces 2 and 3); all of K; the epilogue stores fp16(silu(fp16(gate))) * fp16(up).
// ROTATE (direct products): p.rope_cos.
template <int TILES, bool RAGGED, bool TILED, int WAVES, int SLOTS, bool PRODUCER, bool SWIGLU = false, bool ROTATE = false>
__device__ __forceinline__ void gemm_piece(const MatmulParams &p, int unit, int mb, int slice, int step0, int step1, bool zero_rest, bool more,
                                           int tid_bias) {
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    constexpr int NB = WAVES == 8 ? 2 : 4;     // B operands (16 columns each) per wave
    constexpr int DMA_PER = WAVES == 8 ? 2 : 4;

    const int tid = threadIdx.x + tid_bias;
    const int wave8 = tid >> 6;                // 0 .. WAVES-1
    const int wave = wave8 & 3;                // piece of the tile / rows of the ring this wave serves
    const int hh = wave8 >> 2;                 // eight waves: 0 = high nibbles (columns c), 1 = low nibbles (columns c + 64)
    const int lane = tid & 63;
    const int c = lane & 15;
    const int g = lane >> 4;
    int sg = 0;
    if (!SWIGLU && p.nseg > 1 && unit >= p.seg[1].unit0) sg = 1;
    if (!SWIGLU && p.nseg > 2 && unit >= p.seg[2].unit0) sg = 2;
    const MatmulSegment seg = segment_at<true>(p, sg);
    const int pair = SWIGLU ? unit >> 1 : unit - seg.unit0;
    const int col0 = SWIGLU ? unit * 128 : pair * GEMM_COLS;
    const bool two_blocks = SWIGLU || col0 + 128 < seg.N;
    const int m0 = mb * p.block_rows;
    const int blk = wave >> 1;                 // block of the pair this wave decodes
    const int bp = wave & 1;                   // ... and its pair of byte positions
    const uint32_t sel0 = 0x0c000c00u | (uint32_t)(2 * bp) | ((uint32_t)(4 + 2 * bp) << 16);
    const uint32_t sel1 = sel0 + 0x00010001u;

    const long w_row = seg.N / 2;              // bytes per k of the nibbles
    const long s_row = seg.N / 32;             // bytes per k of the scales
    // ---- this wave's four DMA instructions per stage ----
    //  rows 8w .. 8w+7 of the nibbles; their scales (lanes 0..15); rows 32w .. 32w+31 of the A tile.
    //  Address = uniform base of the step (scalar arithmetic) + a lane offset fixed for the whole kernel.
    const uint8_t *w_base = TILED ? seg.w + (long)pair * tiled_steps(p.K) * TILE_BYTES : seg.w + (long)pair * 128;
    const uint8_t *s_base = reinterpret_cast<const uint8_t *>(seg.s) + (long)pair * 8;
    // SWIGLU: bytes from the gate weight's tiles to the up weight's, the gate's first piece and its first scale group in a tile
    const long up = SWIGLU ? (long)((uintptr_t)p.seg[1].w - (uintptr_t)p.seg[0].w) : 0;
    const int sw_piece = SWIGLU ? 2 * (unit & 1) : 0;
    // ... and where lane l's dword of a step's 64 scale bytes of k-octet `oct` lies (groups 0, 1: gate, 2, 3: up)
    auto scale_off = [&](int oct, int l) -> long {
        if (!SWIGLU) return TILE_W_BYTES + (16 * oct + l) * 4;
        const int grp = l >> 2;
        return TILE_W_BYTES + oct * 64 + (2 * (unit & 1) + (grp & 1)) * 16 + (l & 3) * 4 + (grp >= 2 ? up : 0L);
    };
    auto piece_off = [&](int q) -> long { return SWIGLU ? (sw_piece + (q & 1)) * 1024L + (q >= 2 ? up : 0L) : q * 1024L; };
    const uint8_t *a_base = reinterpret_cast<const uint8_t *>(p.a);
    const int w_lrow = 8 * wave + (lane >> 3), w_lcol = 16 * (two_blocks ? (lane & 7) : (lane & 3));
    const int s_lrow = 8 * wave + ((lane & 15) >> 1), s_lcol = 4 * (two_blocks ? (lane & 1) : 0);
    const int a_chunk = (lane & 3) ^ ((lane >> 3) & 3);                   // logical 16-byte chunk stored in slot lane&3
    const long a_r0 = (long)min(m0 + (WAVES == 8 ? 16 * wave8 : 32 * wave) + (lane >> 2), p.M - 1) * p.lda * 2;
    const long a_r1 = (long)min(m0 + 32 * wave + 16 + (lane >> 2), p.M - 1) * p.lda * 2;
    const uint32_t w_voff = (uint32_t)(w_lrow * w_row + w_lcol);
    const uint32_t s_voff = (uint32_t)(s_lrow * s_row + s_lcol);
    const uint32_t a_voff0 = (uint32_t)(a_r0 + 16 * a_chunk), a_voff1 = (uint32_t)(a_r1 + 16 * a_chunk);

    // eight waves: the two DMA instructions of a wave and stage separately, so that the A rows' (no branch around it)
    // can go between the MFMAs of a step
    auto issue_ws8 = [&](int step, int slot_) {
        uint8_t *st = lds + slot_ * GS_BYTES;
        const uint8_t *tile = w_base + (long)step * TILE_BYTES;
        if (hh == 0) __builtin_amdgcn_global_load_lds((gptr_t)(tile + piece_off(wave) + lane * 16), (lptr_t)(st + wave * 1024), 16, 0, 0);
        else if (lane < 16) __builtin_amdgcn_global_load_lds((gptr_t)(tile + scale_off(wave, lane)), (lptr_t)(st + GS_W + wave * 64), 4, 0, 0);
    };
    auto issue_a8 = [&](int step, int slot_) {
        __builtin_amdgcn_global_load_lds((gptr_t)(a_base + (long)step * 64 + a_voff0), (lptr_t)(lds + slot_ * GS_BYTES + GS_W + GS_S + wave8 * 1024), 16, 0, 0);
    };
    auto issue = [&](int step, int slot_) {
        uint8_t *st = lds + slot_ * GS_BYTES;
        const long k0 = (long)step * 32;
        if (WAVES == 8) {
            // two DMA instructions a wave: waves 0-3 their piece of the nibbles, waves 4-7 its scales; every wave 16 rows of A
            issue_ws8(step, slot_);
            issue_a8(step, slot_);
        } else if (TILED) {
            const uint8_t *tile = w_base + (long)step * TILE_BYTES;
            __builtin_amdgcn_global_load_lds((gptr_t)(tile + wave * 1024 + lane * 16), (lptr_t)(st + wave * 1024), 16, 0, 0);
            if (lane < 16)
                __builtin_amdgcn_global_load_lds((gptr_t)(tile + TILE_W_BYTES + (16 * wave + lane) * 4), (lptr_t)(st + GS_W + wave * 64), 4, 0, 0);
            if (!RAGGED) {
                __builtin_amdgcn_global_load_lds((gptr_t)(a_base + k0 * 2 + a_voff0), (lptr_t)(st + GS_W + GS_S + wave * 2048), 16, 0, 0);
                __builtin_amdgcn_global_load_lds((gptr_t)(a_base + k0 * 2 + a_voff1), (lptr_t)(st + GS_W + GS_S + wave * 2048 + 1024), 16, 0, 0);
            } else {
                const long ac = min(k0 + 8 * a_chunk, (long)p.K - 8) * 2;
                __builtin_amdgcn_global_load_lds((gptr_t)(a_base + a_r0 + ac), (lptr_t)(st + GS_W + GS_S + wave * 2048), 16, 0, 0);
                __builtin_amdgcn_global_load_lds((gptr_t)(a_base + a_r1 + ac), (lptr_t)(st + GS_W + GS_S + wave * 2048 + 1024), 16, 0, 0);
            }
        } else if (!RAGGED) {
            __builtin_amdgcn_global_load_lds((gptr_t)(w_base + k0 * w_row + w_voff), (lptr_t)(st + wave * GS_WBLOCK), 16, 0, 0);
            if (lane < 16)
                __builtin_amdgcn_global_load_lds((gptr_t)(s_base + k0 * s_row + s_voff), (lptr_t)(st + GS_W + wave * 64), 4, 0, 0);
            __builtin_amdgcn_global_load_lds((gptr_t)(a_base + k0 * 2 + a_voff0), (lptr_t)(st + GS_W + GS_S + wave * 2048), 16, 0, 0);
            __builtin_amdgcn_global_load_lds((gptr_t)(a_base + k0 * 2 + a_voff1), (lptr_t)(st + GS_W + GS_S + wave * 2048 + 1024), 16, 0, 0);
        } else {
            // rows past K repeat row K-1 (their products are masked out below); the A columns stay inside the row
            const long wr = min(k0 + w_lrow, (long)p.K - 1), sr = min(k0 + s_lrow, (long)p.K - 1);
            const long ac = min(k0 + 8 * a_chunk, (long)p.K - 8) * 2;
            __builtin_amdgcn_global_load_lds((gptr_t)(w_base + wr * w_row + w_lcol), (lptr_t)(st + wave * GS_WBLOCK), 16, 0, 0);
            if (lane < 16)
                __builtin_amdgcn_global_load_lds((gptr_t)(s_base + sr * s_row + s_lcol), (lptr_t)(st + GS_W + wave * 64), 4, 0, 0);
            __builtin_amdgcn_global_load_lds((gptr_t)(a_base + a_r0 + ac), (lptr_t)(st + GS_W + GS_S + wave * 2048), 16, 0, 0);
            __builtin_amdgcn_global_load_lds((gptr_t)(a_base + a_r1 + ac), (lptr_t)(st + GS_W + GS_S + wave * 2048 + 1024), 16, 0, 0);
        }
    };

    f4 acc[NB][TILES];
#pragma unroll
    for (int h = 0; h < NB; ++h)
#pragma unroll
        for (int t = 0; t < TILES; ++t) acc[h][t] = f4{0.f, 0.f, 0.f, 0.f};

    const int n_steps = max(step1 - step0, 0);
    // workgroups that share a K-slice read the same A tiles; each starts at a different step of the
    // slice (and wraps) so that they do not all pull the same L2 lines at the same time
    const int rot = n_steps > 0 ? uniform_divmod(unit * 5, n_steps).r : 0;
    int fetch = step0 + rot;                   // next step to fetch
    auto fetch_next = [&](int slot_) {
        issue(fetch, slot_);
        fetch = fetch + 1 == step1 ? step0 : fetch + 1;
    };
    if constexpr (PRODUCER) {
        if (wave8 >= 8) {
            // ---- the DMA waves: 5 + TILES instructions a stage (four pieces of nibbles, the scales, one per 16 rows of A) ----
            constexpr int A_FIRST = TILES > 5 ? (TILES - 5) / 2 : 0;   // row tiles that go with the weights, so that the two have as many to issue
            __builtin_amdgcn_s_setprio(3);      // their few instructions first: the others wait for what they request (3 % of a launch)
            uint32_t a_voff[TILES];
#pragma unroll
            for (int t = 0; t < TILES; ++t)
                a_voff[t] = (uint32_t)((long)min(m0 + 16 * t + (lane >> 2), p.M - 1) * p.lda * 2 + 16 * a_chunk);
            // checkpoint layout: lane l moves 16 bytes of row l / 8 of a piece and the dword l % 2 of row l / 2 of the scales.
            // RAGGED: the last step has `left` = 8, 16 or 24 rows of k; what lies past them repeats valid ones (masked when decoded)
            const int last = RAGGED ? (p.K - 1) / 32 : -1, left = p.K - 32 * last;
            const uint32_t raw_w = (uint32_t)((lane >> 3) * w_row + w_lcol), raw_s = (uint32_t)((lane >> 1) * s_row + s_lcol);
            const uint32_t raw_s_last = RAGGED ? (uint32_t)(min(lane >> 1, left - 1) * s_row + s_lcol) : 0;
            const uint32_t a_back = RAGGED ? (uint32_t)(2 * (8 * a_chunk - min(8 * a_chunk, left - 8))) : 0;
            auto feed = [&](auto which) {
            constexpr bool WEIGHTS = decltype(which)::value == 0;
            constexpr int T0 = WEIGHTS ? 0 : A_FIRST, T1 = WEIGHTS ? A_FIRST : TILES;
            gemm_feed<(WEIGHTS ? 5 : 0) + T1 - T0, SLOTS>(n_steps, [&](int slot_) {
                uint8_t *st = lds + slot_ * GS_BYTES;
                const uint8_t *arow = a_base + (long)fetch * 64;
                if constexpr (!WEIGHTS) {
                } else if (TILED) {
                    const uint8_t *tile = w_base + (long)fetch * TILE_BYTES;
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        __builtin_amdgcn_global_load_lds((gptr_t)(tile + piece_off(q) + lane * 16), (lptr_t)(st + q * 1024), 16, 0, 0);
                    __builtin_amdgcn_global_load_lds((gptr_t)(tile + scale_off(lane >> 4, lane & 15)), (lptr_t)(st + GS_W), 4, 0, 0);
                } else {
                    const uint8_t *rows = w_base + (long)fetch * 32 * w_row;
                    const bool at_end = RAGGED && fetch == last;
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        __builtin_amdgcn_global_load_lds((gptr_t)(rows + (at_end && 8 * q >= left ? 0 : 8 * q) * w_row + raw_w),
                                                         (lptr_t)(st + q * GS_WBLOCK), 16, 0, 0);
                    __builtin_amdgcn_global_load_lds((gptr_t)(s_base + (long)fetch * 32 * s_row + (at_end ? raw_s_last : raw_s)), (lptr_t)(st + GS_W), 4, 0, 0);
                }
#pragma unroll
                for (int t = T0; t < T1; ++t)
                    __builtin_amdgcn_global_load_lds((gptr_t)(arow + (RAGGED && fetch == last ? a_voff[t] - a_back : a_voff[t])),
                                                     (lptr_t)(st + GS_W + GS_S + t * 1024), 16, 0, 0);
                fetch = fetch + 1 == step1 ? step0 : fetch + 1;
            });
            };
            if (wave8 == 8) feed(int_constant<0>{});
            else feed(int_constant<1>{});
            // the barriers of the epilogue: one that frees the ring, one per row tile
#pragma unroll 1
            for (int t = 0; t < 1 + TILES + (more ? 1 : 0); ++t) gemm_barrier();
            return;
        }
    } else {
#pragma unroll
        for (int i = 0; i < SLOTS - 2; ++i)
            if (i < n_steps) fetch_next(i);
    }

    // the eight dwords of this lane's column bytes and of their scales, for one step
    auto load_ws = [&](const uint8_t *st, uint32_t (&wv)[8], uint32_t (&sv)[8]) {
        if (TILED) {
            // wv[0..3] = (x, x2) of byte 2bp, (x, x2) of byte 2bp+1; sv[0..3] / sv[4..7] = the row pairs' scales of the
            // block's first / second 64 columns
            const u32x4 wq = *reinterpret_cast<const u32x4 *>(st + wave * 1024 + lane * 16);
            if (WAVES == 8) {                  // the scales of this wave's nibble only
                const u32x4 sc = *reinterpret_cast<const u32x4 *>(st + GS_W + g * 64 + (2 * blk + hh) * 16);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    wv[r] = wq[r];
                    wv[4 + r] = 0;
                    sv[r] = sc[r];
                    sv[4 + r] = 0;
                }
                return;
            }
            const u32x4 sh = *reinterpret_cast<const u32x4 *>(st + GS_W + g * 64 + (2 * blk) * 16);
            const u32x4 sl = *reinterpret_cast<const u32x4 *>(st + GS_W + g * 64 + (2 * blk + 1) * 16);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                wv[r] = wq[r];
                wv[4 + r] = 0;
                sv[r] = sh[r];
                sv[4 + r] = sl[r];
            }
            return;
        }
#pragma unroll
        for (int r = 0; r < 8; ++r) {
            wv[r] = *reinterpret_cast<const uint32_t *>(st + g * GS_WBLOCK + r * 128 + 64 * blk + 4 * c);
            sv[r] = *reinterpret_cast<const uint32_t *>(st + GS_W + (8 * g + r) * 8 + 4 * blk);
        }
    };
    // exact fp16 code * scale, as the four B operands (byte 2bp high / low, byte 2bp+1 high / low)
    // eight waves (tiled weights; the checkpoint layout's have the DMA waves and RowWeights): the nibble this wave decodes, as constants of one
    // and-or + one packed fma (code = fp16 bits * mul + off)
    const uint32_t nib_mask = hh == 0 ? 0x00F000F0u : 0x000F000Fu;
    uint32_t nib_magic = MAGIC_1024;                             // in a register the compiler cannot see through: (bits & mask) | magic is
    asm volatile("" : "+v"(nib_magic));                       // then ONE v_and_or_b32 (no literal operands there), not an AND and an OR
    const h2 nib_mul = hh == 0 ? h2{(half_t)0.0625f, (half_t)0.0625f} : h2{(half_t)1.0f, (half_t)1.0f};
    const h2 nib_off = hh == 0 ? h2{(half_t)-72.0f, (half_t)-72.0f} : h2{(half_t)-1032.0f, (half_t)-1032.0f};
    auto decode = [&](const uint32_t (&wv)[8], const uint32_t (&sv)[8], bool dead, h8 (&b)[NB]) {
        u32x4 v0h, v0l, v1h, v1l;
        if (TILED && WAVES == 8) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint32_t pr0 = j < 2 ? wv[j] : wv[j - 2] >> 8;           // rows (2j, 2j+1) of byte 2bp, codes + 8
                const uint32_t pr1 = j < 2 ? wv[2 + j] : wv[j] >> 8;           // ... of byte 2bp+1
                const h2 sc = as_h2(sv[j]);
                v0h[j] = as_u32(__builtin_elementwise_fma(as_h2((pr0 & nib_mask) | nib_magic), nib_mul, nib_off) * sc);
                v1h[j] = as_u32(__builtin_elementwise_fma(as_h2((pr1 & nib_mask) | nib_magic), nib_mul, nib_off) * sc);
            }
            b[0] = __builtin_bit_cast(h8, v0h);
            b[1] = __builtin_bit_cast(h8, v1h);
            return;
        }
        if (TILED) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint32_t pr0 = j < 2 ? wv[j] : wv[j - 2] >> 8;           // rows (2j, 2j+1) of byte 2bp, codes + 8
                const uint32_t pr1 = j < 2 ? wv[2 + j] : wv[j] >> 8;           // ... of byte 2bp+1
                const h2 s_hi = as_h2(sv[j]), s_lo = as_h2(sv[4 + j]);
                v0h[j] = as_u32(codes_high(pr0) * s_hi);
                v0l[j] = as_u32(codes_low(pr0) * s_lo);
                v1h[j] = as_u32(codes_high(pr1) * s_hi);
                v1l[j] = as_u32(codes_low(pr1) * s_lo);
            }
            if constexpr (NB == 4) {
                b[0] = __builtin_bit_cast(h8, v0h);
                b[1] = __builtin_bit_cast(h8, v0l);
                b[2] = __builtin_bit_cast(h8, v1h);
                b[3] = __builtin_bit_cast(h8, v1l);
            }
            return;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint32_t pr0 = __builtin_amdgcn_perm(wv[2 * j + 1], wv[2 * j], sel0) ^ 0x00880088u;
            const uint32_t pr1 = __builtin_amdgcn_perm(wv[2 * j + 1], wv[2 * j], sel1) ^ 0x00880088u;
            const h2 s_hi = as_h2(pack_lo16(sv[2 * j], sv[2 * j + 1]));
            const h2 s_lo = as_h2(pack_hi16(sv[2 * j], sv[2 * j + 1]));
            v0h[j] = as_u32(codes_high(pr0) * s_hi);
            v0l[j] = as_u32(codes_low(pr0) * s_lo);
            v1h[j] = as_u32(codes_high(pr1) * s_hi);
            v1l[j] = as_u32(codes_low(pr1) * s_lo);
        }
        if (RAGGED && dead) v0h = v0l = v1h = v1l = u32x4{0u, 0u, 0u, 0u};     // k >= K: no contribution
        if constexpr (NB == 4) {
            b[0] = __builtin_bit_cast(h8, v0h);
            b[1] = __builtin_bit_cast(h8, v0l);
            b[2] = __builtin_bit_cast(h8, v1h);
            b[3] = __builtin_bit_cast(h8, v1l);
        }
    };
    auto k_dead = [&](int step) { return step * 32 + 8 * g >= p.K; };      // only in the last step when K % 32 != 0
    // While the matrix pipe multiplies step i (A tile read from stage i, B operands decoded one iteration
    // earlier), the wave reads the nibbles of step i+1 from LDS and decodes them.  After the barrier of
    // iteration i every wave has finished iteration i-1, so the slot of stage i-1 is refilled with step i+5.
    auto load_a = [&](const uint8_t *st, h8 (&av)[TILES]) {
        const uint8_t *at = st + GS_W + GS_S;
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
            const int r = 16 * t + c;
            av[t] = *reinterpret_cast<const h8 *>(at + r * 64 + ((g ^ ((r >> 1) & 3)) << 4));
        }
    };
    auto multiply = [&](const h8 (&av)[TILES], const h8 (&b)[NB]) {
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
#pragma unroll
            for (int o = 0; o < NB; ++o) acc[o][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av[t], b[o], acc[o][t], 0, 0, 0);
        }
    };
    // Steps go in pairs: ONE wait + barrier per two steps.  With S slots (six; more only with the DMA waves): at the barrier
    // before steps i, i+1 the stages of steps i .. i+2 have landed (the B operands of step i+2 are decoded during step i+1),
    // steps i+3 .. i+S-3 may be in flight, and the slots of steps i-2, i-1 are refilled with steps i+S-2, i+S-1.  A stage has the same two steps of time to land as
    // with a barrier per step; the waves meet half as often.
    if constexpr (PRODUCER) {
        // (the end of K, the last step of a slice that has it, is fetched as stage at_end: rot < n_steps)
        const int at_end = RAGGED && step1 > (p.K - 1) / 32 ? n_steps - 1 - rot : -1;
        const auto weights = [&] {
            if constexpr (TILED) return TiledWeights(hh, wave * 1024 + lane * 16, GS_W + g * 64 + (2 * blk + hh) * 16);
            else return RowWeights<RAGGED>(hh, g * GS_WBLOCK + 64 * blk + 4 * c, GS_W + 64 * g + 4 * blk, sel0, at_end, (p.K - 1) / 32 * 32 + 8 * g >= p.K);
        }();
        gemm_multiply<TILES, SLOTS, GS_BYTES>(lds, n_steps, weights, GS_W + GS_S + c * 64 + ((g ^ ((c >> 1) & 3)) << 4), acc);
    } else if (n_steps > 0) {
        h8 bq[NB];
        int cur = step0 + rot;                 // step being multiplied
        int slot = 0;                          // its ring slot
        {
            gemm_wait_dma<DMA_PER>(min(SLOTS - 3, n_steps - 1));
            gemm_barrier();
            uint32_t wv[8], sv[8];
            load_ws(lds, wv, sv);
            decode(wv, sv, k_dead(cur), bq);
        }
        // multiply the step in `slot` with bq while the B operands of the next step are decoded
        auto one_step = [&]() {
            const uint8_t *st = lds + slot * GS_BYTES;
            slot = slot == SLOTS - 1 ? 0 : slot + 1;
            cur = cur + 1 == step1 ? step0 : cur + 1;
            // past the last step the next slot holds stale bytes: read, decoded and never used
            uint32_t wv[8], sv[8];
            h8 av[TILES], bn[NB];
            load_a(st, av);
            load_ws(lds + slot * GS_BYTES, wv, sv);
            multiply(av, bq);
            decode(wv, sv, k_dead(cur), bn);
#pragma unroll
            for (int o = 0; o < NB; ++o) bq[o] = bn[o];
        };
        auto back = [&](int k) { return slot >= k ? slot - k : slot + SLOTS - k; };
        int i = 0;
#pragma unroll 1
        for (; i + SLOTS - 1 < n_steps; i += 2) {      // both refills exist: the body is one basic block
            gemm_wait_vm<DMA_PER * (SLOTS - 5)>();
            gemm_barrier();
            if constexpr (WAVES == 8 && TILES < 8) {       // (with all 8 row tiles, the prefill, this form measured 5-8 % slower)
                // the nibbles and scales of the two refills now, their A rows from inside the steps: the address unit takes
                // 16 cycles per instruction, and between MFMAs the wave has them to spare (2 % off a launch at 100 rows;
                // the nibbles and scales too from inside the steps, behind their branches: 4 % slower)
                const int sa = back(2), sb = back(1);
                const int fa = fetch, fb = fetch + 1 == step1 ? step0 : fetch + 1;
                fetch = fb + 1 == step1 ? step0 : fb + 1;
                issue_ws8(fa, sa);
                issue_ws8(fb, sb);
                for (int half = 0; half < 2; ++half) {
                    const uint8_t *st = lds + slot * GS_BYTES;
                    slot = slot == SLOTS - 1 ? 0 : slot + 1;
                    cur = cur + 1 == step1 ? step0 : cur + 1;
                    uint32_t wv[8], sv[8];
                    h8 av[TILES], bn[NB];
                    load_a(st, av);
                    load_ws(lds + slot * GS_BYTES, wv, sv);
                    constexpr int T0 = TILES / 2;
#pragma unroll
                    for (int t = 0; t < T0; ++t)
#pragma unroll
                        for (int o = 0; o < NB; ++o) acc[o][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av[t], bq[o], acc[o][t], 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                    issue_a8(half == 0 ? fa : fb, half == 0 ? sa : sb);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int t = T0; t < TILES; ++t)
#pragma unroll
                        for (int o = 0; o < NB; ++o) acc[o][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av[t], bq[o], acc[o][t], 0, 0, 0);
                    decode(wv, sv, k_dead(cur), bn);
#pragma unroll
                    for (int o = 0; o < NB; ++o) bq[o] = bn[o];
                }
            } else {
                fetch_next(back(2));
                fetch_next(back(1));
                one_step();
                one_step();
            }
        }
#pragma unroll 1
        for (; i < n_steps; i += 2) {
            gemm_wait_dma<DMA_PER>(max(0, min(n_steps - 1, i + SLOTS - 3) - (i + 2)));      // stages issued past step i + 2
            gemm_barrier();
            if (i + SLOTS - 2 < n_steps) fetch_next(back(2));
            if (i + SLOTS - 1 < n_steps) fetch_next(back(1));
            one_step();
            if (i + 1 < n_steps) one_step();
        }
    }

    // ---- results leave one 16-row tile at a time through LDS: [16][256 + 4] floats, two buffers in turn ----
    // accumulator element r of acc[o][t] is row 16t + 4g + r, column 128*blk + 64*(o&1) + 4c + 2*bp + (o>>1).
    // Bare barriers again: __syncthreads() would wait for the global stores of the previous tile to be
    // acknowledged, one memory round trip per tile.  A buffer is rewritten two tiles later, after a barrier
    // that every wave reaches only when its reads of that buffer have returned.
    constexpr int OP = GEMM_COLS + 4;
    constexpr int OTILE_BYTES = 16 * OP * 4;
    static_assert(2 * OTILE_BYTES <= SLOTS * GS_BYTES, "two output tiles must fit in the ring");
    float *slab = p.partial + (long)slice * p.M * p.n_total;
    const int o_row = (tid & 255) >> 4;         // 0..15
    const int o_half = tid >> 8;                // eight waves: the second 256 threads store the second half of the columns
    const int o_lane = tid & 15;                // store q of this lane: columns 64q + 4*o_lane .. (fp16: 128q + 8*o_lane ..),
                                                // so that one store instruction writes whole contiguous rows
    // RoPE: the factors of this thread's eight dims, of three row tiles ahead
    static_assert(!ROTATE || (TILED && WAVES == 8 && !SWIGLU), "heads in whole runs of eight columns");
    const bool rotate = ROTATE && seg.col0 < p.rope_cols;
    constexpr int FAR = 3;
    h8 cs[ROTATE ? TILES : 1], sn[ROTATE ? TILES : 1];
    auto factors = [&](auto at) {
        constexpr int T = decltype(at)::value;
        if constexpr (ROTATE && T < TILES) {
            const uint32_t at_ = (uint32_t)(min(m0 + 16 * T + o_row, p.M - 1) * 128 + 16 * (o_lane & 7));
            cs[T] = *reinterpret_cast<const h8 *>(reinterpret_cast<const uint8_t *>(p.rope_cos) + at_);
            sn[T] = *reinterpret_cast<const h8 *>(reinterpret_cast<const uint8_t *>(p.rope_sin) + at_);
        }
    };
    if (rotate) {
        factors(int_constant<0>{});
        factors(int_constant<1>{});
        factors(int_constant<2>{});
    }
    gemm_barrier();                             // every wave has left the main loop: the ring is free
    static_for<TILES>([&](auto at) {
        constexpr int t = decltype(at)::value;
        if (rotate) factors(int_constant<t + FAR>{});
        float *otile = reinterpret_cast<float *>(lds + (t & 1) * OTILE_BYTES);
        // operands o and o + 2 are neighbouring columns: one 8-byte LDS store for the pair
        if constexpr (WAVES == 8) {
#pragma unroll
            for (int r = 0; r < 4; ++r)
                *reinterpret_cast<f2 *>(&otile[(4 * g + r) * OP + 128 * blk + 64 * hh + 4 * c + 2 * bp]) = f2{acc[0][t][r], acc[1][t][r]};
        } else {
#pragma unroll
            for (int o = 0; o < 2; ++o)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    *reinterpret_cast<f2 *>(&otile[(4 * g + r) * OP + 128 * blk + 64 * o + 4 * c + 2 * bp]) = f2{acc[o][t][r], acc[o + 2][t][r]};
        }
        gemm_barrier();
        const int m = m0 + 16 * t + o_row;
        if (SWIGLU || m < p.M) {
            if constexpr (SWIGLU) {
                // rows of 128 gate columns and the same 128 up columns: four of them a thread, with partial_silu_mul_kernel's roundings
                const int cq = 4 * (tid & 31), row = (tid >> 5) & 15, mr = m0 + 16 * t + row;
                if (mr < p.M) {
                    const f4 gv = *reinterpret_cast<const f4 *>(otile + row * OP + cq), uv = *reinterpret_cast<const f4 *>(otile + row * OP + 128 + cq);
                    h4 o;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float gf = (float)(half_t)gv[e];
                        o[e] = (half_t)(gf / (1.0f + expf(-gf))) * (half_t)uv[e];
                    }
                    *reinterpret_cast<h4 *>(seg.c + (long)mr * seg.ldc + col0 + cq) = o;
                }
            } else if (ROTATE || p.direct) {
#pragma unroll
                for (int q = (WAVES == 8 ? o_half : 0); q < (WAVES == 8 ? o_half + 1 : 2); ++q) {
                    const int n_seg = col0 + 128 * q + 8 * o_lane;
                    if (n_seg < seg.N) {
                        const int n = seg.col0 + n_seg;
                        const f4 v0 = *reinterpret_cast<const f4 *>(otile + o_row * OP + 128 * q + 8 * o_lane);
                        const f4 v1 = *reinterpret_cast<const f4 *>(otile + o_row * OP + 128 * q + 8 * o_lane + 4);
                        h8 o;
                        if (rotate && n < p.rope_cols) {
                            if constexpr (ROTATE) {
                                const float *there = otile + o_row * OP + 128 * q + 8 * (o_lane ^ 8);
                                const f4 u0 = *reinterpret_cast<const f4 *>(there), u1 = *reinterpret_cast<const f4 *>(there + 4);
                                o = rope_eight(v0, v1, u0, u1, o_lane >= 8, cs[t], sn[t]);
                            }
                        } else {
#pragma unroll
                            for (int e = 0; e < 4; ++e) {
                                o[e] = matmul_epilogue(p, v0[e], m, n + e);
                                o[4 + e] = matmul_epilogue(p, v1[e], m, n + 4 + e);
                            }
                        }
                        *reinterpret_cast<h8 *>(seg.c + (long)m * seg.ldc + n_seg) = o;
                    }
                }
            } else {
                float *dst = slab + (long)m * p.n_total + seg.col0 + col0;
#pragma unroll
                for (int q = (WAVES == 8 ? 2 * o_half : 0); q < (WAVES == 8 ? 2 * o_half + 2 : 4); ++q) {
                    const int cq = 64 * q + 4 * o_lane;
                    if (col0 + cq < seg.N) *reinterpret_cast<f4 *>(dst + cq) = *reinterpret_cast<const f4 *>(otile + o_row * OP + cq);
                }
            }
        }
    });
    if (zero_rest) {
        for (int sl = slice + 1; sl < p.ksplit; ++sl) {
            float *zslab = p.partial + (long)sl * p.M * p.n_total;
            for (int t = 0; t < TILES; ++t) {
                const int m = m0 + 16 * t + o_row;
                if (m < p.M) {
                    float *dst = zslab + (long)m * p.n_total + seg.col0 + col0;
#pragma unroll
                    for (int q = (WAVES == 8 ? 2 * o_half : 0); q < (WAVES == 8 ? 2 * o_half + 2 : 4); ++q) {
                        const int cq = 64 * q + 4 * o_lane;
                        if (col0 + cq < seg.N) *reinterpret_cast<f4 *>(dst + cq) = f4{0.f, 0.f, 0.f, 0.f};
                    }
                }
            }
        }
    }
    if (more) gemm_barrier();                   // the next piece refills the ring the last row tile left through
}

// PRODUCER (eight waves only): two more waves issue every DMA instruction of the workgroup and wait for them; the eight
// others only meet them at the barriers.  The compute unit's address unit takes 16 cycles per DMA instruction, during which
// the issuing wave stands still: ~0.28 us per pair of steps off the multiplying waves' path.  For launches with one
// workgroup per compute unit (more waves on a SIMD that already holds four would cap the registers below
// what the kernel needs).  SLOTS: slots of the ring.
// RANGE (p.chunk > 0): the steps of all column units, laid end to end, are dealt in runs of p.chunk to the workgroups, one
// workgroup per compute unit, so a workgroup may finish one unit and begin the next: up to two pieces, one after the other.
template <int TILES, bool RAGGED, bool TILED, int WAVES, int SLOTS = GEMM_STAGES, bool PRODUCER = false, bool RANGE = false, bool SWIGLU = false, bool ROTATE = false>
// (SWIGLU without the DMA waves: at most 128 registers, so that two workgroups of eight waves fit a compute unit)
__global__ __launch_bounds__(64 * (WAVES + (PRODUCER ? GEMM_DMA_WAVES : 0)), WAVES == 8 ? (SWIGLU && !PRODUCER ? 4 : 1) : 2) void q40_gemm_kernel(MatmulParams p) {
    static_assert(WAVES == 4 || (WAVES == 8 && (TILED ? !RAGGED : PRODUCER)), "eight waves: K a multiple of 32, or the checkpoint layout with the DMA waves");
    static_assert(SLOTS >= 6 && SLOTS <= 8 && (SLOTS == GEMM_STAGES || PRODUCER) && (!PRODUCER || WAVES == 8), "ring depth");
    args_ahead<sizeof(MatmulParams)>();
    const int steps_total = (p.K + 31) / 32;
    if constexpr (RANGE) {
        int run0 = (int)blockIdx.x * p.chunk;                  // (units x steps is far below 2^31)
        const int run1 = min(run0 + p.chunk, p.units * steps_total);
#pragma unroll 1
        for (bool more = true; more;) {                        // (a loop, not two calls: the second piece runs code that is warm)
            const int unit = run0 / steps_total;
            const int s0 = run0 - unit * steps_total;
            const int s1 = min(steps_total, s0 + (run1 - run0));
            const int first = (unit * steps_total) / p.chunk;  // the workgroup that holds the unit's first piece
            run0 += s1 - s0;
            more = run0 < run1;
            // a zero the compiler cannot see keeps everything derived from the thread index inside the piece: hoisted out of
            // this loop those values stay live through it and the kernel spills
            int opaque_zero;
            asm volatile("s_mov_b32 %0, 0" : "=s"(opaque_zero));
            gemm_piece<TILES, RAGGED, TILED, WAVES, SLOTS, PRODUCER>(p, unit, 0, (int)blockIdx.x - first, s0, s1, s1 == steps_total, more, opaque_zero);
        }
    } else {
        // blockIdx.x -> unit: each XCD (workgroups are dealt to them in turn) takes a contiguous run of column units, which share scale lines
        const int slot = blockIdx.x;
        const int unit = (slot & 7) * (p.units_pad >> 3) + (slot >> 3);
        if (unit >= p.units) return;
        const int mb = p.mb0 + (int)blockIdx.y;
        const int slice = blockIdx.z;
        const int s0 = slice * p.steps_per_slice;
        gemm_piece<TILES, RAGGED, TILED, WAVES, SLOTS, PRODUCER, SWIGLU, ROTATE>(p, unit, mb, slice, s0, min(s0 + p.steps_per_slice, steps_total), false, false, 0);
    }
}

// ---- two K-groups in one workgroup (tiled weights with K a multiple of 64, or the checkpoint layout; one workgroup per compute unit) ----------------
// A workgroup owns ONE 128-column block (pieces 2 blk, 2 blk + 1 of the unit's tiles), a block of rows and a K-slice, and
// its eight multiplying waves form two groups: group kk takes the steps 2 i + kk of the slice.  Wave (kk, hh, bp)
// multiplies the columns of nibble hh of piece 2 blk + bp of its group's steps with all row tiles of A - the same two B
// operands and 14 MFMAs per step as in q40_gemm_kernel - so a ring stage holds TWO steps: both pieces of the block and the
// scales of either step, and either step's rows of A.  The groups' accumulators are added through LDS at the end (group 0
// + group 1, a fixed order), and all eight waves write the slab.  Against q40_gemm_kernel's 256-column units this
// fills the GPU with half as many K-slices, i.e. half the slab bytes written here and read back by the consumer; the
// price is that a row of A is staged for 128 columns instead of 256.
// Checkpoint layout (gemm_blocks_fit): a step is 32 rows of 64 bytes, fetched in the order that RowWeights reads; K may end anywhere in the last stage
// (RAGGED), and a workgroup that has all of K stores the fp16 product itself.
constexpr int KG_W = 4096;                     // [group kk][piece bp] x 1024
constexpr int KG_S = 512;                      // [group kk] x 256 (the whole scale block of the step)
template <int TILES> struct KgShape {
    static constexpr int STAGE = KG_W + KG_S + 2 * TILES * 1024;
    static constexpr int SLOTS = gemm_slots(STAGE, TILES <= 4 ? 8 : 6);
    static constexpr int RING = SLOTS * STAGE;
    static constexpr int PER = 3 + TILES;                          // DMA instructions of a step
    static constexpr int OP = 128 + 4;                             // floats per row of a group's sums in LDS
    static constexpr int SUMS = TILES * 16 * OP * 4;               // one K-group's sums: [row][OP] fp32
    static constexpr int LDS = RING > 2 * SUMS ? RING : 2 * SUMS;
    static_assert(PER * (SLOTS - 5) <= 63 && LDS <= 160 * 1024, "ring");
};

template <int TILES, bool TILED, bool RAGGED>
__global__ __launch_bounds__(64 * (8 + GEMM_DMA_WAVES), 1) void q40_gemm_kg_kernel(MatmulParams p) {
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    typedef KgShape<TILES> S;
    constexpr int SLOTS = S::SLOTS, PER = S::PER, STAGE = S::STAGE;
    const int tid = threadIdx.x;
    const int wave8 = __builtin_amdgcn_readfirstlane(tid >> 6);       // 0..7 multiply, the others issue the DMA
    const int lane = tid & 63, c = lane & 15, g = lane >> 4;
    args_ahead<sizeof(MatmulParams)>();
    // blockIdx -> (128-column block, row block, K-slice).  Tiled weights: blocks of one unit are neighbours (same XCD every 8).  Checkpoint layout: the
    // blocks of a unit are the halves of its 128-byte lines and go to one XCD, one after the other, in step.
    const int hb = blockIdx.x;
    const int slot_u = hb >> 1, raw_b = (hb & 7) * (p.units_pad >> 2) + (hb >> 3);
    const int blk = TILED ? hb & 1 : raw_b & 1;
    const int unit = TILED ? (slot_u & 7) * (p.units_pad >> 3) + (slot_u >> 3) : raw_b >> 1;
    if (unit >= p.units) return;
    const int mb = blockIdx.y, slice = blockIdx.z;
    int sg = 0;
    if (p.nseg > 1 && unit >= p.seg[1].unit0) sg = 1;
    if (p.nseg > 2 && unit >= p.seg[2].unit0) sg = 2;
    const MatmulSegment seg = segment_at<true>(p, sg);
    const int pair = unit - seg.unit0;
    const int col0 = pair * GEMM_COLS + 128 * blk;
    if (col0 >= seg.N) return;                                         // a weight with an odd number of 128-column blocks
    const int m0 = mb * p.block_rows;
    const int steps_total = RAGGED ? (p.K + 31) / 32 : p.K / 32;
    const int step0 = slice * p.steps_per_slice, step1 = min(step0 + p.steps_per_slice, steps_total);
    // stages (two steps each; slices are even).  RAGGED: the last one of the slice that ends K may have a step that lies past it
    const int n_st = (max(step1 - step0, 0) + (RAGGED ? 1 : 0)) / 2;
    const bool ends = RAGGED && step1 == steps_total;
    const long w_row = seg.N / 2, s_row = seg.N / 32;                  // checkpoint layout: bytes per k of the nibbles, of the scales
    const uint8_t *w_base = TILED ? seg.w + (long)pair * tiled_steps(p.K) * TILE_BYTES + (long)step0 * TILE_BYTES : seg.w + (long)step0 * 32 * w_row + (long)pair * 128 + 64 * blk;
    const uint8_t *s_base = reinterpret_cast<const uint8_t *>(seg.s) + (long)step0 * 32 * s_row + (long)pair * 8 + 4 * blk;
    const uint8_t *a_base = reinterpret_cast<const uint8_t *>(p.a) + (long)step0 * 64;
    // workgroups of a K-slice start at different stages, above 128 rows in K's order (with the RMSNorm behind, 512 x 4096 x 4096 30.5 us and 28.8, fewer rows level)
    const int rot = n_st > 0 && p.M <= GEMM_BM ? uniform_divmod((TILED ? hb : unit) * 5, n_st).r : 0;

    if (wave8 >= 8) {
        // ---- the DMA waves: a K-group's steps each ----
        __builtin_amdgcn_s_setprio(3);
        const int a_chunk = (lane & 3) ^ ((lane >> 3) & 3);
        uint32_t a_voff[TILES];
#pragma unroll
        for (int t = 0; t < TILES; ++t)
            a_voff[t] = (uint32_t)((long)min(m0 + 16 * t + (lane >> 2), p.M - 1) * p.lda * 2 + 16 * a_chunk);
        int fetch = rot;
        const int kk = wave8 - 8;
        // checkpoint layout: lane l of instruction q moves 16 bytes of row 8 ((l / 4) % 4) + 4 q + l / 16 of a step (RowWeights), and row l % 32's scales (64 rows'
        // in one of the two waves: 1 % slower).  `left` rows of the last stage's step lie before the end of K (none, if it is all past it): what is read in the
        // place of others repeats valid ones.
        const int left = RAGGED && ends ? p.K - 32 * (step0 + 2 * (n_st - 1) + kk) : 32;
        const int raw_r = 8 * ((lane >> 2) & 3) + (lane >> 4), raw_c = 16 * (lane & 3);
        const uint32_t raw_w[2] = {(uint32_t)(raw_r * w_row + raw_c), (uint32_t)((raw_r + 4) * w_row + raw_c)}, raw_s = (uint32_t)((lane & 31) * s_row);
        auto back = [&](int r) { return r - min(r, left - 1); };           // rows to go back
        const uint32_t back_w[2] = {(uint32_t)(back(raw_r) * w_row), (uint32_t)(back(raw_r + 4) * w_row)}, back_s = (uint32_t)(back(lane & 31) * s_row);
        const uint32_t back_a = (uint32_t)(2 * (8 * a_chunk - min(8 * a_chunk, left - 8)));
        gemm_feed<PER, SLOTS>(n_st, [&](int slot_) {
            uint8_t *st = lds + slot_ * STAGE;
            {
                const long step = 2 * fetch + kk;
                const uint8_t *arow = a_base + step * 64;
                const bool at_end = RAGGED && ends && fetch == n_st - 1;
                if constexpr (TILED) {
                    const uint8_t *tile = w_base + step * TILE_BYTES;
#pragma unroll
                    for (int bp = 0; bp < 2; ++bp)
                        __builtin_amdgcn_global_load_lds((gptr_t)(tile + (2 * blk + bp) * 1024 + lane * 16), (lptr_t)(st + (2 * kk + bp) * 1024), 16, 0, 0);
                    __builtin_amdgcn_global_load_lds((gptr_t)(tile + TILE_W_BYTES + lane * 4), (lptr_t)(st + KG_W + kk * 256), 4, 0, 0);
                } else {
                    const uint8_t *rows = w_base + step * 32 * w_row;
#pragma unroll
                    for (int q = 0; q < 2; ++q)
                        __builtin_amdgcn_global_load_lds((gptr_t)(rows + raw_w[q] - (at_end ? back_w[q] : 0u)), (lptr_t)(st + (2 * kk + q) * 1024), 16, 0, 0);
                    __builtin_amdgcn_global_load_lds((gptr_t)(s_base + step * 32 * s_row + raw_s - (at_end ? back_s : 0u)), (lptr_t)(st + KG_W + kk * 256), 4, 0, 0);
                }
#pragma unroll
                for (int t = 0; t < TILES; ++t)
                    __builtin_amdgcn_global_load_lds((gptr_t)(arow + a_voff[t] - (at_end ? back_a : 0u)), (lptr_t)(st + KG_W + KG_S + (kk * TILES + t) * 1024), 16, 0, 0);
            }
            fetch = fetch + 1 == n_st ? 0 : fetch + 1;
        });
        gemm_barrier();                                        // the epilogue's two barriers: ring free, sums in place
        gemm_barrier();
        return;
    }

    const int kk = wave8 >> 2, hh = (wave8 >> 1) & 1, bp = wave8 & 1;
    f4 acc[2][TILES];
    const auto weights = [&] {
        if constexpr (TILED) return TiledWeights(hh, (2 * kk + bp) * 1024 + lane * 16, KG_W + kk * 256 + g * 64 + (2 * blk + hh) * 16);
        else return RowWeights<RAGGED, true>(hh, kk * 2048 + g * 64 + 4 * c, KG_W + kk * 256 + g * 32, 0x0c000c00u | (uint32_t)(2 * bp) | ((uint32_t)(4 + 2 * bp) << 16),
                                             ends ? n_st - 1 - rot : -1, 32 * (step0 + 2 * (n_st - 1) + kk) + 8 * g >= p.K);     // (the end of K is that stage: rot < n_st)
    }();
    gemm_multiply<TILES, SLOTS, STAGE, GEMM_PRODUCTS_FIRST>(lds, n_st, weights, KG_W + KG_S + kk * TILES * 1024 + c * 64 + ((g ^ ((c >> 1) & 3)) << 4), acc);

    // ---- both groups' sums as rows of 128 floats in LDS; then every thread adds group 0 + group 1 (a fixed order) for
    // 16-byte runs of whole rows and writes the slab: one pass, two barriers, all eight waves storing ----
    gemm_barrier();                                            // every wave has left the loop: the ring is free
    constexpr int OP = S::OP;
    {
        float *sums = reinterpret_cast<float *>(lds + kk * S::SUMS);
#pragma unroll
        for (int t = 0; t < TILES; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                *reinterpret_cast<f2 *>(&sums[(16 * t + 4 * g + r) * OP + 64 * hh + 4 * c + 2 * bp]) = f2{acc[0][t][r], acc[1][t][r]};
    }
    gemm_barrier();
    const float *sum0 = reinterpret_cast<const float *>(lds), *sum1 = reinterpret_cast<const float *>(lds + S::SUMS);
    float *slab = p.partial + (long)slice * p.M * p.n_total + seg.col0 + col0;
#pragma unroll
    for (int it = 0; it < TILES; ++it) {
        const int idx = tid + 512 * it;                        // tid < 512 here: (row, run of four columns)
        const int row = idx >> 5, cq = 4 * (idx & 31);
        const int m = m0 + row;
        if (m < p.M && row < p.block_rows) {
            const f4 v = *reinterpret_cast<const f4 *>(sum0 + row * OP + cq) + *reinterpret_cast<const f4 *>(sum1 + row * OP + cq);
            if (!TILED && p.direct) {
                const int n = col0 + cq;
                const h4 o = {matmul_epilogue(p, v[0], m, n), matmul_epilogue(p, v[1], m, n + 1), matmul_epilogue(p, v[2], m, n + 2), matmul_epilogue(p, v[3], m, n + 3)};
                *reinterpret_cast<h4 *>(seg.c + (long)m * seg.ldc + n) = o;
            } else {
                *reinterpret_cast<f4 *>(slab + (long)m * p.n_total + cq) = v;
            }
        }
    }
}

// ---- SwiGLU inside the launch of w1|w3 (tiled weights, up to 128 rows, all of K in one workgroup) -----------------------
// q40_gemm_kg_kernel with the roles of a workgroup's waves changed: instead of the two pieces of one 128-column block, a
// workgroup takes piece bp of block j of the GATE weight and the same piece of the UP weight (64 columns each, the same
// columns), so its wave (kk, hh, gu) holds, after the K-groups are added, gate or up for exactly the columns its neighbour
// holds the other for.  The epilogue forms fp16(silu(fp16(gate))) * fp16(up) with the roundings of partial_silu_mul_kernel
// and stores the activations of w2: no slab leaves the launch and the SiLU launch is gone.  Ask = WarmWeights: workgroups past the columns ask for w2 (q40_warm.hpp).
// (A kernel of its own: calls that ask for nothing took 19.04 us at 33 rows of 4096 -> 2 x 11008 before there were such workgroups, 19.32 with them, 19.04 so.)
template <int TILES> struct SwigluShape {
    static constexpr int SC = 1024;                                  // scales: [group kk][gate | up] x 256
    static constexpr int STAGE = KG_W + SC + 2 * TILES * 1024;
    // One row tile: eleven slots, steps behind 300 rows of the 7B model 1918, 2023 and 2046 us at 5, 10 and 16 branches with eight, 1895, 2001
    // and 2038 with eleven (ten: the same).  Two and three: seven to eleven within 1.2 % of eight either way, by the card; from four on they are as good.
    static constexpr int SLOTS = gemm_slots(STAGE, TILES == 1 ? 11 : 8);
    static constexpr int LDS = SLOTS * STAGE;
    static constexpr int PER = 4 + TILES;                            // DMA instructions of a step
    static constexpr int OP = 128 + 4;                               // floats per row of a group's sums in LDS
    static constexpr int SUMS = TILES * 16 * OP * 4;                 // one K-group's sums: [row][gate | up] fp32
    static_assert(2 * SUMS <= LDS, "both groups' sums must fit in the ring");
    static_assert(PER * (SLOTS - 5) <= 63 && LDS <= 160 * 1024, "ring");
};

template <int TILES, class... Ask>
__global__ __launch_bounds__(64 * (8 + GEMM_DMA_WAVES), 1) void q40_gemm_swiglu_kernel(MatmulParams p, Ask... next) {
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    typedef SwigluShape<TILES> S;
    constexpr int SLOTS = S::SLOTS, PER = S::PER, STAGE = S::STAGE;
    const int tid = threadIdx.x;
    const int wave8 = __builtin_amdgcn_readfirstlane(tid >> 6);       // 0..7 multiply, the others issue the DMA
    const int lane = tid & 63, c = lane & 15, g = lane >> 4;
    args_ahead<sizeof(MatmulParams)>();
    // blockIdx -> (128-column block j of the gate and of the up weight, piece bp of that block)
    const int hb = blockIdx.x;
    const int blockj = hb >> 1, bp = hb & 1;
    const int pair = blockj >> 1, blk = blockj & 1;
    const int n_half = p.seg[0].N;
    if constexpr (sizeof...(Ask) > 0) {
        if (__builtin_expect(128 * blockj >= n_half, 0)) return warm_weights(next..., hb & 7, (hb - n_half / 64) >> 3, tid, 64 * (8 + GEMM_DMA_WAVES));
    } else if (128 * blockj >= n_half) return;
    constexpr int m0 = 0;
    const int n_st = p.K / 64;                                         // stages (two steps each), all of K
    const uint8_t *w_gate = p.seg[0].w + (long)pair * tiled_steps(p.K) * TILE_BYTES;
    const uint8_t *w_up = p.seg[1].w + (long)pair * tiled_steps(p.K) * TILE_BYTES;
    const uint8_t *a_base = reinterpret_cast<const uint8_t *>(p.a);
    const int rot = n_st > 0 ? uniform_divmod(hb * 5, n_st).r : 0;             // workgroups of a K-slice start at different stages

    if (wave8 >= 8) {
        // ---- the DMA waves: a K-group's steps each ----
        __builtin_amdgcn_s_setprio(3);
        const int a_chunk = (lane & 3) ^ ((lane >> 3) & 3);
        uint32_t a_voff[TILES];
#pragma unroll
        for (int t = 0; t < TILES; ++t)
            a_voff[t] = (uint32_t)((long)min(m0 + 16 * t + (lane >> 2), p.M - 1) * p.lda * 2 + 16 * a_chunk);
        int fetch = rot;
        const int kk = wave8 - 8;
        gemm_feed<PER, SLOTS>(n_st, [&](int slot_) {
            uint8_t *st = lds + slot_ * STAGE;
            {
                const long off = (long)(2 * fetch + kk) * TILE_BYTES;
                const uint8_t *arow = a_base + (long)(2 * fetch + kk) * 64;
#pragma unroll
                for (int gu = 0; gu < 2; ++gu) {
                    const uint8_t *tile = (gu == 0 ? w_gate : w_up) + off;
                    __builtin_amdgcn_global_load_lds((gptr_t)(tile + (2 * blk + bp) * 1024 + lane * 16), (lptr_t)(st + (2 * kk + gu) * 1024), 16, 0, 0);
                    __builtin_amdgcn_global_load_lds((gptr_t)(tile + TILE_W_BYTES + lane * 4), (lptr_t)(st + KG_W + (2 * kk + gu) * 256), 4, 0, 0);
                }
#pragma unroll
                for (int t = 0; t < TILES; ++t)
                    __builtin_amdgcn_global_load_lds((gptr_t)(arow + a_voff[t]), (lptr_t)(st + KG_W + S::SC + (kk * TILES + t) * 1024), 16, 0, 0);
            }
            fetch = fetch + 1 == n_st ? 0 : fetch + 1;
        });
        gemm_barrier();                                        // the epilogue's two barriers: ring free, sums in place
        gemm_barrier();
        return;
    }

    const int kk = wave8 >> 2, hh = (wave8 >> 1) & 1, gu = wave8 & 1;       // K-group, nibble, gate (0) or up (1)
    f4 acc[2][TILES];
    gemm_multiply<TILES, SLOTS, STAGE, GEMM_PRODUCTS_FIRST>(lds, n_st, TiledWeights(hh, (2 * kk + gu) * 1024 + lane * 16, KG_W + (2 * kk + gu) * 256 + g * 64 + (2 * blk + hh) * 16),
                                       KG_W + S::SC + kk * TILES * 1024 + c * 64 + ((g ^ ((c >> 1) & 3)) << 4), acc);

    // ---- both groups' sums as rows of 64 gate and 64 up columns in LDS, then every thread adds group 0 + group 1 (a fixed order) of four columns ----
    // local column 32 hh + 2 c + o is column 128 blockj + 64 hh + 4 c + 2 bp + o of the weights
    gemm_barrier();                                            // every wave has left the loop: the ring is free
    constexpr int OP = S::OP;
    {
        float *sums = reinterpret_cast<float *>(lds + kk * S::SUMS) + 64 * gu + 32 * hh + 2 * c;
#pragma unroll
        for (int t = 0; t < TILES; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) *reinterpret_cast<f2 *>(&sums[(16 * t + 4 * g + r) * OP]) = f2{acc[0][t][r], acc[1][t][r]};
    }
    gemm_barrier();
    const float *sum0 = reinterpret_cast<const float *>(lds), *sum1 = reinterpret_cast<const float *>(lds + S::SUMS);
    const int cq = 4 * (tid & 15), out_col = 128 * blockj + 64 * ((tid & 15) >> 3) + 4 * (2 * (tid & 7)) + 2 * bp;      // tid < 512 here
#pragma unroll
    for (int row = tid >> 4; row < 16 * TILES; row += 32) {
        if (row >= p.M) break;
        const int at = row * OP + cq;
        const f4 gv = *reinterpret_cast<const f4 *>(sum0 + at) + *reinterpret_cast<const f4 *>(sum1 + at);
        const f4 uv = *reinterpret_cast<const f4 *>(sum0 + at + 64) + *reinterpret_cast<const f4 *>(sum1 + at + 64);
        half_t ov[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {                          // the roundings of partial_silu_mul_kernel
            const float gf = (float)(half_t)gv[e];
            const half_t sl = (half_t)(gf / (1.0f + expf(-gf)));
            ov[e] = sl * (half_t)uv[e];
        }
        half_t *dst = p.c + (long)row * p.ldc + out_col;
        *reinterpret_cast<h2 *>(dst) = h2{ov[0], ov[1]};
        *reinterpret_cast<h2 *>(dst + 4) = h2{ov[2], ov[3]};
    }
}

// ---- above 128 rows, six slots of weights a workgroup (tiled weights, all of K, one workgroup per compute unit) -------------------
// A workgroup owns 64 .. 128 rows of A; its twelve multiplying waves - wave (nibble hh, slot s) has one piece's columns of one nibble, two
// B operands, as in q40_gemm_kernel - work on six pieces (64 columns x 32 rows) a stage:
//   * WIDE_SWIGLU: pieces 3 u .. 3 u + 2 of the gate weight and the same of the up weight: 384 columns, where q40_gemm_kernel has 256;
//   * WIDE_GROUPS: pieces 3 u .. 3 u + 2 of the weights laid end to end, of two steps: 192 columns and two K-groups, added through LDS;
//   * WIDE_SIX: pieces 6 u .. 6 u + 5, 384 columns.
// Bound by the matrix and vector pipes, which a third wave on each SIMD keeps busier (0.55 us a step of 128 rows x 384 columns,
// where 1.5 steps of the 256-column units take 0.63), and by how well its workgroups divide the compute units: w1|w3 of the 7B shape is
// 232 of them at 512 rows, one round, where 256-column units leave 344, two rounds; wq|wk|wv is 256, where those leave 192.
// In us, before and now: w1|w3 4096 -> 2 x 11008 at 512 rows 112.9 (818 TFLOP/s) and 90.1 (1025), at 300 rows 85.3 and 65.2, 1024 rows 201
// and 178, 2047 rows 375 (985) and 353 (1047); 8192 -> 2 x 28672 at 640 rows 609 and 515, 2047 rows 1834 and 1693.  wq|wk|wv 4096 -> 12288 at
// 512 rows 60.3 (855 TFLOP/s) and 53.2 (969), 1024 rows 119 and 106; 8192 -> 10240 at 512 rows 99.6 and 86.8; 5120 -> 5120 at 2047 rows
// 131 and 122.  With six pieces, against the faster of the others: 4096 -> 12288 at 1024 rows 101 and 93, 2047 rows 191 (1079) and 181 (1140);
// 5120 -> 15360 at 1300 rows 226 and 192; 5120 -> 5120 at 2047 rows 120 and 112.  The rules: gemm_swiglu_rows_launch and gemm_wide_fits.
enum { WIDE_SWIGLU, WIDE_GROUPS, WIDE_SIX };
template <int TILES, int MODE> struct WideShape {
    static constexpr int STEPS = MODE == WIDE_GROUPS ? 2 : 1;    // of a stage
    static constexpr int PIECES = MODE == WIDE_SIX ? 6 : 3;      // of an output row
    static constexpr int W = 6 * 1024, SC = 6 * 128;             // of the six slots: nibbles; scales [octet][nibble][8 rows]
    static constexpr int STAGE = W + SC + STEPS * TILES * 1024;
    static constexpr int SLOTS = 6;
    static constexpr int OP = 64 * PIECES + 4;
    static constexpr int OTILE = (MODE == WIDE_SWIGLU ? 2 : 1) * 16 * OP * 4;      // [16][OP] fp32; SwiGLU: [gate | up][16][OP]
    static constexpr int SUMS = TILES * 16 * OP * 4;             // two K-groups: [row][OP] fp32
    static constexpr int OUT = MODE == WIDE_GROUPS ? SUMS : 2 * OTILE;
    // RoPE: the rows' cosines, then their sines (128 bytes each), behind the sums, where the ring was, or (WIDE_SIX) behind the ring
    static constexpr int ROPE = MODE == WIDE_SIX ? SLOTS * STAGE : OUT, ROPE_END = MODE == WIDE_SWIGLU ? 0 : ROPE + TILES * 4096;
    static constexpr int LDS = SLOTS * STAGE > OUT ? (SLOTS * STAGE > ROPE_END ? SLOTS * STAGE : ROPE_END) : OUT > ROPE_END ? OUT : ROPE_END;
    static_assert(ROPE % 16 == 0 && 2 * OTILE <= SLOTS * STAGE, "factors are brought by DMA");
    static_assert(LDS <= 160 * 1024, "ring");
};
constexpr int WIDE_WAVES = 12;

template <int TILES, int MODE>
__global__ __launch_bounds__(64 * (WIDE_WAVES + GEMM_DMA_WAVES), 1) void q40_gemm_wide_kernel(MatmulParams p) {
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    typedef WideShape<TILES, MODE> S;
    constexpr int SLOTS = S::SLOTS, STAGE = S::STAGE, STEPS = S::STEPS, PIECES = S::PIECES;
    constexpr bool SWIGLU = MODE == WIDE_SWIGLU;
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63, c = lane & 15, g = lane >> 4;
    // blockIdx -> (unit of three or six pieces, row block): each XCD takes a contiguous run of units
    args_ahead<sizeof(MatmulParams)>();
    const int at = blockIdx.x, mb = p.mb0 + (int)blockIdx.y;
    const int unit = (at & 7) * (p.units_pad >> 3) + (at >> 3);
    if (unit >= p.units) return;
    const int m0 = mb * p.block_rows, pieces = (SWIGLU ? p.seg[0].N : p.n_total) / 64;
    const int n_st = p.K / (32 * STEPS);
    // a piece's weight and its number within the weight
    auto segment_of = [&](int &P) {
        int sg = 0;
        if (!SWIGLU && p.nseg > 1 && P >= p.seg[1].col0 / 64) sg = 1;
        if (!SWIGLU && p.nseg > 2 && P >= p.seg[2].col0 / 64) sg = 2;
        if (!SWIGLU) P -= p.seg[sg].col0 / 64;
        return sg;
    };

    if (wave >= WIDE_WAVES) {
        // ---- the DMA waves: the weights and the rows of A, or (WIDE_GROUPS) a step each ----
        __builtin_amdgcn_s_setprio(3);
        const int a_chunk = (lane & 3) ^ ((lane >> 3) & 3);
        uint32_t a_voff[TILES];
#pragma unroll
        for (int t = 0; t < TILES; ++t) a_voff[t] = (uint32_t)((long)min(m0 + 16 * t + (lane >> 2), p.M - 1) * p.lda * 2 + 16 * a_chunk);
        const uint8_t *w[6], *sc[3];
        int in_tile[6];
#pragma unroll
        for (int s = 0; s < 6; ++s) {
            int P = min(PIECES * unit + s % PIECES, pieces - 1);       // (past the end: the last one again, not stored)
            const int sg = SWIGLU ? s / 3 : segment_of(P);
            in_tile[s] = P & 3;
            w[s] = p.seg[sg].w + ((long)(P >> 2) * tiled_steps(p.K) + (MODE == WIDE_GROUPS ? s / 3 : 0)) * TILE_BYTES;
        }
#pragma unroll
        for (int i = 0; i < 3; ++i) {                                  // lanes 0 .. 31: slot 2 i's 128 bytes, the others slot 2 i + 1's
            const bool odd = lane >= 32;
            const int d = lane & 31;
            sc[i] = (odd ? w[2 * i + 1] : w[2 * i]) + TILE_W_BYTES + (d >> 3) * 64 + ((odd ? in_tile[2 * i + 1] : in_tile[2 * i]) >> 1) * 32 + (d & 7) * 4;
        }
#pragma unroll
        for (int s = 0; s < 6; ++s) w[s] += in_tile[s] * 1024;
        const uint8_t *a_base = reinterpret_cast<const uint8_t *>(p.a);
        int fetch = 0;                                                 // (in K's order: a start of its own for each unit gains nothing here)
        auto feed = [&](auto which) {
            constexpr int D = decltype(which)::value;
            constexpr bool GROUPS = MODE == WIDE_GROUPS;
            constexpr int W0 = GROUPS ? 3 * D : 6 * D, W1 = GROUPS ? W0 + 3 : 6;             // slots, pairs of slots' scales and steps of A of this wave
            constexpr int S0 = GROUPS ? 2 * D : 3 * D, S1 = GROUPS && D == 0 ? 2 : 3;
            constexpr int K0 = GROUPS || D == 1 ? (GROUPS ? D : 0) : STEPS, K1 = GROUPS ? D + 1 : STEPS;
            gemm_feed<W1 - W0 + S1 - S0 + (K1 - K0) * TILES, SLOTS>(n_st, [&](int slot_) {
                uint8_t *st = lds + slot_ * STAGE;
                const long off = (long)fetch * STEPS * TILE_BYTES;
                const uint8_t *arow = a_base + (long)fetch * STEPS * 64;
#pragma unroll
                for (int s = W0; s < W1; ++s) __builtin_amdgcn_global_load_lds((gptr_t)(w[s] + off + lane * 16), (lptr_t)(st + s * 1024), 16, 0, 0);
#pragma unroll
                for (int i = S0; i < S1; ++i) __builtin_amdgcn_global_load_lds((gptr_t)(sc[i] + off), (lptr_t)(st + S::W + i * 256), 4, 0, 0);
#pragma unroll
                for (int k = K0; k < K1; ++k)
#pragma unroll
                    for (int t = 0; t < TILES; ++t)
                        __builtin_amdgcn_global_load_lds((gptr_t)(arow + k * 64 + a_voff[t]), (lptr_t)(st + S::W + S::SC + (k * TILES + t) * 1024), 16, 0, 0);
                ++fetch;
            });
        };
        if (wave == WIDE_WAVES) feed(int_constant<0>{});
        else feed(int_constant<1>{});
        // RoPE: the factors of the workgroup's rows, cosines by one wave, sines by the other (eight rows an instruction)
        const bool rotate = !SWIGLU && p.rope_cos != nullptr;
        auto bring_factors = [&] {
            const uint8_t *tab = reinterpret_cast<const uint8_t *>(wave == WIDE_WAVES ? p.rope_cos : p.rope_sin);
            uint8_t *to = lds + S::ROPE + (wave == WIDE_WAVES ? 0 : TILES * 2048);
#pragma unroll
            for (int i = 0; i < 2 * TILES; ++i)
                __builtin_amdgcn_global_load_lds((gptr_t)(tab + (uint32_t)(min(m0 + 8 * i + (lane >> 3), p.M - 1) * 128 + 16 * (lane & 7))), (lptr_t)(to + i * 1024), 16, 0, 0);
        };
        // the barriers of the epilogue: ring free, one per row tile; ring free, the second group's sums in place, all sums
        if constexpr (MODE == WIDE_GROUPS) {
            gemm_barrier();
            if (rotate) bring_factors();
            gemm_barrier();
            gemm_wait_vm<0>();
            gemm_barrier();
        } else {
            if (MODE == WIDE_SIX && rotate) bring_factors();           // (under the last stages)
            gemm_wait_vm<0>();
#pragma unroll 1
            for (int t = 0; t < 1 + TILES; ++t) gemm_barrier();
        }
        return;
    }

    // nibble, slot; the slot's half - gate (0) or up (1), or K-group - and piece
    const int hh = wave >= 6 ? 1 : 0, s = wave - 6 * hh, half = s >= PIECES ? 1 : 0, k3 = s - 3 * half;
    f4 acc[2][TILES];
    // (Seven row tiles: reading ahead needs more than the 128 registers of four waves a SIMD, and does not gain what that costs.  In us, ahead and not:
    // w1|w3 and wq|wk|wv of the 7B shape at 400 rows 90.1, 52.9 and 86.2, 49.3, w1|w3 of the 70B shape at 540 rows 551 and 524.)
    gemm_multiply<TILES, SLOTS, STAGE, GEMM_DECODE_FIRST, TILES != 7>(lds, n_st, TiledWeights(hh, s * 1024 + lane * 16, S::W + s * 128 + g * 32 + hh * 16),
                                       S::W + S::SC + (MODE == WIDE_GROUPS ? half * TILES * 1024 : 0) + c * 64 + ((g ^ ((c >> 1) & 3)) << 4), acc);

    // rows of 64 PIECES columns: local column 64 k3 + 32 hh + 2 c + o is column 128 (P / 2) + 64 hh + 4 c + 2 (P % 2) + o, P the piece;
    // a thread stores local columns 4 o_lane .. + 3
    constexpr int OP = S::OP;
    const int o_row = tid / 48, o_lane = tid % 48, q = o_lane & 15;
    int P = PIECES * unit + (o_lane >> 4);
    const bool mine = P < pieces;
    const int sg = segment_of(P), out_col = 128 * (P >> 1) + 64 * (q >> 3) + 8 * (q & 7) + 2 * (P & 1);
    half_t *const out = (sg == 0 ? p.seg[0].c : sg == 1 ? p.seg[1].c : p.seg[2].c) + out_col;
    const long ldc = sg == 0 ? p.seg[0].ldc : sg == 1 ? p.seg[1].ldc : p.seg[2].ldc;
    const bool rotate = !SWIGLU && p.rope_cos != nullptr;
    // four sums of row r of the workgroup, with the residual or rotated, to columns n_, n_ + 1, n_ + 4 and n_ + 5 (dims 8 (q % 8) + 2 (piece % 2) + 0, 1, 4, 5)
    auto store = [&](const float *row_sums, int piece, int n_, int m, int r, half_t *dst) {
        const f4 v = *reinterpret_cast<const f4 *>(row_sums + 4 * o_lane);
        h2 lo, hi;
        if (rotate && n_ < p.rope_cols) {
            const f4 u = *reinterpret_cast<const f4 *>(row_sums + 4 * (o_lane ^ 8));
            const half_t *cs = reinterpret_cast<const half_t *>(lds + S::ROPE) + r * 64 + 8 * (q & 7) + 2 * (piece & 1), *sn = cs + TILES * 1024;
            rope_pairs(v, u, (q & 8) != 0, *reinterpret_cast<const h2 *>(cs), *reinterpret_cast<const h2 *>(cs + 4), *reinterpret_cast<const h2 *>(sn),
                       *reinterpret_cast<const h2 *>(sn + 4), lo, hi);
        } else {
            lo = h2{matmul_epilogue(p, v[0], m, n_), matmul_epilogue(p, v[1], m, n_ + 1)};
            hi = h2{matmul_epilogue(p, v[2], m, n_ + 4), matmul_epilogue(p, v[3], m, n_ + 5)};
        }
        *reinterpret_cast<h2 *>(dst) = lo;
        *reinterpret_cast<h2 *>(dst + 4) = hi;
    };
    gemm_barrier();                                            // every wave has left the loop: the ring is free
    if constexpr (SWIGLU) {
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
            float *otile = reinterpret_cast<float *>(lds + (t & 1) * S::OTILE);
#pragma unroll
            for (int r = 0; r < 4; ++r)
                *reinterpret_cast<f2 *>(&otile[half * 16 * OP + (4 * g + r) * OP + 64 * k3 + 32 * hh + 2 * c]) = f2{acc[0][t][r], acc[1][t][r]};
            gemm_barrier();
            const int m = m0 + 16 * t + o_row;
            if (m < p.M && mine) {
                const f4 gv = *reinterpret_cast<const f4 *>(otile + o_row * OP + 4 * o_lane);
                const f4 uv = *reinterpret_cast<const f4 *>(otile + 16 * OP + o_row * OP + 4 * o_lane);
                half_t ov[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {                  // the roundings of partial_silu_mul_kernel
                    const float gf = (float)(half_t)gv[e];
                    ov[e] = (half_t)(gf / (1.0f + expf(-gf))) * (half_t)uv[e];
                }
                *reinterpret_cast<h2 *>(out + (long)m * ldc) = h2{ov[0], ov[1]};
                *reinterpret_cast<h2 *>(out + (long)m * ldc + 4) = h2{ov[2], ov[3]};
            }
        }
    } else if constexpr (MODE == WIDE_SIX) {
        // two runs of four columns a thread: local columns 4 o_lane .. and 192 + 4 o_lane ..
        int P2 = 6 * unit + 3 + (o_lane >> 4);
        const bool mine2 = P2 < pieces;
        const int sg2 = segment_of(P2), out_col2 = 128 * (P2 >> 1) + 64 * (q >> 3) + 8 * (q & 7) + 2 * (P2 & 1);
        half_t *const out2 = (sg2 == 0 ? p.seg[0].c : sg2 == 1 ? p.seg[1].c : p.seg[2].c) + out_col2;
        const long ldc2 = sg2 == 0 ? p.seg[0].ldc : sg2 == 1 ? p.seg[1].ldc : p.seg[2].ldc;
        const int n = p.seg[sg].col0 + out_col, n2 = p.seg[sg2].col0 + out_col2;
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
            float *otile = reinterpret_cast<float *>(lds + (t & 1) * S::OTILE);
#pragma unroll
            for (int r = 0; r < 4; ++r) *reinterpret_cast<f2 *>(&otile[(4 * g + r) * OP + 64 * k3 + 32 * hh + 2 * c]) = f2{acc[0][t][r], acc[1][t][r]};
            gemm_barrier();
            const int m = m0 + 16 * t + o_row;
            if (m < p.M && mine) store(otile + o_row * OP, P, n, m, 16 * t + o_row, out + (long)m * ldc);
            if (m < p.M && mine2) store(otile + o_row * OP + 192, P2, n2, m, 16 * t + o_row, out2 + (long)m * ldc2);
        }
    } else {
        // the second K-group's sums, then both groups' (in their order), then whole rows
        float *sums = reinterpret_cast<float *>(lds) + 64 * k3 + 32 * hh + 2 * c;
        if (half == 1) {
#pragma unroll
            for (int t = 0; t < TILES; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) *reinterpret_cast<f2 *>(&sums[(16 * t + 4 * g + r) * OP]) = f2{acc[0][t][r], acc[1][t][r]};
        }
        gemm_barrier();
        if (half == 0) {
#pragma unroll
            for (int t = 0; t < TILES; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    f2 *at_ = reinterpret_cast<f2 *>(&sums[(16 * t + 4 * g + r) * OP]);
                    const f2 other = *at_;
                    *at_ = f2{acc[0][t][r] + other[0], acc[1][t][r] + other[1]};
                }
        }
        gemm_barrier();
        const int n = p.seg[sg].col0 + out_col;
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
            const int m = m0 + 16 * t + o_row;
            if (m < p.M && mine) store(reinterpret_cast<const float *>(lds) + (16 * t + o_row) * OP, P, n, m, 16 * t + o_row, out + (long)m * ldc);
        }
    }
}

// Row blocks and K-slices of a launch with more than 128 rows: the pair with the least estimated time.  Measured on the 7B shapes
// at 160 .. 2047 rows: a workgroup takes 0.18 us a step and 0.24 more at 128 rows (in proportion), 4 us around its loop; a launch
// takes as many of these as the workgroups of the busiest XCD need rounds over its 32 compute units (whole column units go to an
// XCD: of 20 units six XCDs get three, one two and one none), and at least 1.2 times its share of them when all
// compute units are busy (the clock drops: two workgroups that share a compute unit take as long as one behind the other).  A
// split's consumer reads 4 bytes an output and slice at ~4 TB/s.  Blocks are even (130 rows: two of 80, not 128 and 2).
// (Before, 128-row blocks and at most 1600 / M slices: w1|w3 at 300 rows 108 us, now 85; wo and w2 at 1024 rows 56 and 136, now
// 37 and 88; 700 rows of wq|wk|wv 108, now 89.  With rounds counted over the 256 compute units together: 5120 x 5120 at 1024 rows
// 128 us, now 77, 5120 x 13824 at 512 rows 138, now 101.)
// Against measurement at the 7B, 13B, 34B and 70B shapes, 160 .. 2047 rows: 0.87 to 1.17 times the estimate, 1.3 to 1.4 times it
// for square weights at 160 rows (15 and 19 us: launches).
// All of these figures and constants are of the loop with one DMA wave whose products waited for their own reads; with two and the read-ahead launches are
// faster (7B: w1|w3 at 512 rows 93.9 -> 90.6 us, at 2047 358.6 -> 346.8), and the constants have not been fitted again.
// (us a step, us more a step at 128 rows, us around the loop, that factor, and what the share of busy compute units adds to the rounds)
struct RowsCost { float step, per_rows, around, busy, more; };
constexpr RowsCost ROWS_256 = {0.18f, 0.24f, 4.0f, 1.2f, 0.0f};
// SwiGLU with three pieces a workgroup (384 columns): fitted to the shapes of 7B, 13B, 34B and 70B at 130 .. 2047 rows, within 4 % in
// the mean.  Taking it where its estimate is the smaller was never slower there than the 256-column units (0.72 .. 0.99 of their time).
constexpr RowsCost ROWS_384 = {0.21f, 0.37f, 4.0f, 1.15f, 0.0f};
// Three pieces and two K-groups a workgroup (192 columns), in the place of 256-column units without a K-split: fitted to wq|wk|wv, wo and
// w2 of 7B, 13B and 70B at 130 .. 2047 rows, within 7 % in the mean.  Taken where it promises 3 %, it took 0.85 .. 0.97 of the time (once
// 1.01: 300 rows of 4096 x 12288).  Where the 256-column units have a K-split they stay: launch and slabs are level or better.
constexpr RowsCost ROWS_192 = {0.11f, 0.21f, 4.0f, 1.2f, 0.0f};
// Six pieces of direct products (384 columns): the step of ROWS_384; with its `busy` a launch that nearly fills a round was estimated 10 to
// 15 % short (8192 x 10240 at 1024 rows 173 us, 3 % more than with 192 columns).  Taken where it promises 3 % more than the others:
// 0.85 .. 0.98 of their time, once 1.007 (1536 rows of 4096 x 12288).  Where that is between 3 and 6 % against 256 columns: 0.85 .. 0.96 (us,
// 4096 x 12288 at 1600 rows 179 -> 155, 5120 x 15360 at 1240 rows 222 -> 189, at 2047 305 -> 291, 4096 x 11008 at 1929 rows 186 -> 175).
constexpr RowsCost ROWS_SIX = {0.21f, 0.37f, 4.0f, 1.0f, 0.15f};
static float gemm_rows_us(const RowsCost &t, int units, long of_unit, int rows, int steps) {
    const float r = (float)(units * of_unit) / 256.0f, rounds = (float)(((units + 7) / 8 * of_unit + 31) / 32);
    return ((rounds > t.busy * r ? rounds : t.busy * r) + t.more * r) * ((float)steps * (t.step + t.per_rows * rows / GEMM_BM) + t.around);
}
// (p.units on entry; returns the estimate)
static float gemm_plan_rows(MatmulParams &p, int steps, int max_ks, const RowsCost &cost) {
    float best_us = -1.0f;
    int ksplit = 1;
    for (int mb = (p.M + GEMM_BM - 1) / GEMM_BM; mb <= p.M / 64; ++mb) {                // (blocks of 64 .. 128 rows)
        const int rows = ((p.M + mb - 1) / mb + 15) / 16 * 16;
        const int blocks = (p.M + rows - 1) / rows;
        const long tiles = (long)p.units * blocks;
        for (int ks = 1; ks <= max_ks && (ks == 1 || (tiles * ks <= 512 && steps / ks >= GEMM_STAGES)); ++ks) {
            const float us = gemm_rows_us(cost, p.units, (long)blocks * ks, rows, (steps + ks - 1) / ks) + (ks > 1 ? (float)ks * p.M * p.n_total * 4.0f / 4.0e6f : 0.0f);
            if (best_us < 0.0f || us < best_us) {
                best_us = us;
                ksplit = ks;
                p.block_rows = rows;
                p.mblocks = blocks;
            }
        }
    }
    p.steps_per_slice = (steps + ksplit - 1) / ksplit;
    p.ksplit = (steps + p.steps_per_slice - 1) / p.steps_per_slice;
    p.chunk = 0;
    return best_us;
}

void gemm_fill_plan(MatmulParams &p) {
    int unit0 = 0, col0 = 0;
    for (int i = 0; i < p.nseg; ++i) {
        p.seg[i].unit0 = unit0;
        p.seg[i].col0 = col0;
        unit0 += (p.seg[i].N + GEMM_COLS - 1) / GEMM_COLS;
        col0 += p.seg[i].N;
    }
    p.units = unit0;
    p.units_pad = (unit0 + 7) / 8 * 8;
    p.n_total = col0;
    p.block_rows = GEMM_BM;
    p.kgroups = 0;
    // Tiled weights, 17 .. 128 rows, K a multiple of 64: 128-column blocks with two K-groups a workgroup (q40_gemm_kg_kernel)
    // where they fill at least two thirds of the compute units in one round - half the K-slices, or fewer, of the 256-column
    // units below for the same number of workgroups.  Narrow matrices (at most 32 blocks: wo, w2) at any such row count, and
    // with two 64-row blocks per column block where K is short (wo at 65 .. 128 rows); wide ones (wq|wk|wv, w1|w3) above 64 rows,
    // and below where K is still cut at least once (wq|wk|wv) above 32 rows or with K up to 4096.  (A step in us, 256-column units and this: 7B architecture,
    // 24 branches 2349 and 2340, 32 2440 and 2414, 37 2523 and 2506, 48 2663 and 2618, 64 2926 and 2880; three layers of the 70B architecture, K = 8192,
    // 24 branches 557 and 561, 40 630 and 624, 48 644 and 638.)  K up to 16384
    // (a row of A is staged for 128 columns
    // instead of 256, which makes the loop ~12 % slower per step: with K = 28672 that outweighs the slabs).  Measured at 100
    // rows, launch + consumer: wo 15.8 against 17.5 us, w2 24.7 against 26.9, w1|w3 39.7 against 40.9; a decode step at 100
    // branches 4.06 against 4.29 ms.
    if (p.tiled && p.M <= 128 && p.K % 64 == 0 && p.K <= 16384) {
        int blocks = 0;
        for (int i = 0; i < p.nseg; ++i) blocks += p.seg[i].N / 128;
        const bool narrow = blocks <= 32;
        const int mblocks = (narrow && p.M > 64 && p.K <= 4096) ? 2 : 1;
        int ks = 256 / (blocks * mblocks);
        int cap = GEMM_KSCAP / p.M;
        if (cap > SMH_MAX_KSPLIT) cap = SMH_MAX_KSPLIT;
        if (ks > cap) ks = cap;
        const int steps = p.K / 32;
        if (ks > steps / 8) ks = steps / 8;                    // at least four stages (of two steps) a slice
        if (ks >= 1 && (narrow || p.M > 64 || (ks >= 2 && (p.M > 32 || p.K <= 4096))) && (long)blocks * mblocks * ks >= 170) {
            p.kgroups = 2;
            p.mblocks = mblocks;
            p.block_rows = mblocks == 2 ? 64 : GEMM_BM;
            p.chunk = 0;
            int sps = (steps + ks - 1) / ks;
            sps += sps & 1;                                    // a stage of the ring is two steps
            p.steps_per_slice = sps;
            p.ksplit = (steps + sps - 1) / sps;
            return;
        }
    }
    // 65 .. 128 rows of a matrix with few column units and a short K (wo at 100 branches): two 64-row blocks per unit take
    // half as many K-slices to fill the GPU, so half the slab bytes are written here and read by the consumer.  The blocks
    // of a unit read the same weights at the same time in the same XCD.  (Measured at 100 rows: wo and the RMSNorm behind
    // it 17.1 us against 19.8; with K = 11008 the launch itself loses what the consumer gains, 43 steps a workgroup.)
    if (p.M > 64 && p.M <= 128 && p.units <= 16 && p.K % 32 == 0 && p.K <= 4096) p.block_rows = 64;
    p.mblocks = (p.M + p.block_rows - 1) / p.block_rows;
    const int steps = (p.K + 31) / 32;
    if (p.M > GEMM_BM) {
        gemm_plan_rows(p, steps, SMH_MAX_KSPLIT, ROWS_256);
        // A plan that is cut along K: the same row blocks with 128-column blocks and two K-groups a workgroup, where they fill two thirds of the
        // compute units in one round with at least two slices of at most 48 stages (64 rows of K each) - about half the slabs.  48 launches of 129 .. 749 rows of
        // tiled weights that take it, with the RMSNorm behind them: 1.06 .. 1.23 times as fast (us, 512 x 4096 x 4096 32.4 and 30.2, 240 rows 21.7 and 19.9,
        // 144 rows 20.3 and 17.0, 221 x 4096 x 11008 32.8 and 29.5), 44 of the checkpoint layout 1.08 .. 1.24; of 86 stages 0.98 and 1.00 (300 and 512 x 4096 x
        // 11008), of one slice 0.81 .. 1.02.  Against 64 bits the slabs' sum errs 0.83 to 1.0 times as much.  Both layouts take it: above 128 rows their slabs
        // are the same bits.
        if (p.ksplit > 1 && p.K % 64 == 0 && p.K <= 16384) {
            const long blocks = p.n_total / 128, on_xcd = (long)p.units_pad / 4 * p.mblocks;
            const int ks = (int)min(min(256 / (blocks * p.mblocks), 32 / on_xcd), (long)p.ksplit), sps = ks > 0 ? ((steps + ks - 1) / ks + 1) / 2 * 2 : 0;
            if (ks >= 2 && blocks * p.mblocks * ks >= 170 && sps <= 96) {
                p.kgroups = 2;
                p.steps_per_slice = sps;
                p.ksplit = (steps + sps - 1) / sps;
            }
        }
        return;
    }
    const long tiles = (long)p.units * p.mblocks;
    // One round of workgroups.  One workgroup per compute unit when the column units divide the GPU well
    // (at least 200 of the 256 units busy): a second co-resident workgroup buys little there and doubles the
    // slabs the next kernel has to read.  Otherwise two per compute unit.  (At M = 100 matrices with few column
    // units still take up to 16 slices: idle compute units cost more than the slab traffic.)
    constexpr int capacity = 512;
    int ks = (int)(capacity / 2 / tiles);
    if (ks < 1 || tiles * ks < 200) ks = (int)(capacity / tiles);
    int cap = GEMM_KSCAP / (p.M > 0 ? p.M : 1);
    if (cap > SMH_MAX_KSPLIT) cap = SMH_MAX_KSPLIT;
    if (ks > cap) ks = cap;
    if (ks > steps / GEMM_STAGES) ks = steps / GEMM_STAGES;
    if (ks < 1) ks = 1;
    p.steps_per_slice = (steps + ks - 1) / ks;
    p.ksplit = (steps + p.steps_per_slice - 1) / p.steps_per_slice;
    // Range cut: a launch that would put two workgroups on some compute units and one on others (256 < workgroups <= 512)
    // deals runs of steps instead, one workgroup per compute unit, crossing unit boundaries.
    p.chunk = 0;
    const long wgs = tiles * p.ksplit;
    if (p.mblocks == 1 && p.K % 32 == 0 && wgs > 256 && wgs <= 512) {
        const long total = (long)p.units * steps;
        const int chunk = (int)((total + 255) / 256);
        if (chunk <= steps && chunk >= 2 * GEMM_STAGES) {
            int pieces = 0;
            for (int u = 0; u < p.units; ++u) {
                const int n = (int)(((long)u * steps + steps - 1) / chunk - ((long)u * steps) / chunk) + 1;
                if (n > pieces) pieces = n;
            }
            if (pieces <= p.ksplit) {           // never more slabs than the even split leaves
                p.chunk = chunk;
                p.ksplit = pieces;
                p.steps_per_slice = chunk;
            }
        }
    }
}

typedef void (*gemm_kernel_t)(MatmulParams);

// Grid (units, row blocks, K-slices), by rows of at most 65535 row blocks
static int gemm_launch_rows(gemm_kernel_t kern, MatmulParams p, int threads, int lds, hipStream_t stream) {
    for (int mb = 0; mb < p.mblocks; mb += 65535) {
        p.mb0 = mb;
        hipLaunchKernelGGL(kern, dim3((unsigned)p.units_pad, (unsigned)min(p.mblocks - mb, 65535), (unsigned)p.ksplit), dim3(threads), lds, stream, p);
    }
    return launch_status();
}

template <bool TILED>
static int gemm_launch_layout(const MatmulParams &p, hipStream_t stream) {
    // one instantiation per number of 16-row tiles (M <= 128) keeps the step free of branches; K % 32 != 0
    // takes the masked variant with all 8 tiles
    constexpr int W = TILED ? GEMM_TILED_WAVES : GEMM_WAVES;
    static const gemm_kernel_t exact[9] = {nullptr, q40_gemm_kernel<2, false, TILED, W>, q40_gemm_kernel<2, false, TILED, W>,
                                           q40_gemm_kernel<3, false, TILED, W>, q40_gemm_kernel<4, false, TILED, W>,
                                           q40_gemm_kernel<5, false, TILED, W>, q40_gemm_kernel<6, false, TILED, W>,
                                           q40_gemm_kernel<7, false, TILED, W>, q40_gemm_kernel<8, false, TILED, W>};
    // one workgroup per compute unit: eight waves and the DMA waves, on both layouts.  (Checkpoint layout, against four waves that
    // leave every SIMD one: 100 rows x 11008 x 4096 31.9 -> 27.2 us, x 32128 61 -> 51, 20 x 28672 x 8192 66 -> 51, 160 x 28672 x
    // 4096 96 -> 64.  Where two workgroups of four waves share a compute unit, eight re-read each nibble from LDS for nothing:
    // 512 x 28672 x 8192 312-324 us against 314, 512 x 20480 x 12288 412 against 389.)
    constexpr int WD = GEMM_TILED_WAVES;
    static const gemm_kernel_t with_dma_wave[9] = {
        nullptr, q40_gemm_kernel<2, false, TILED, WD, gemm_dma_slots(2), true>, q40_gemm_kernel<2, false, TILED, WD, gemm_dma_slots(2), true>,
        q40_gemm_kernel<3, false, TILED, WD, gemm_dma_slots(3), true>, q40_gemm_kernel<4, false, TILED, WD, gemm_dma_slots(4), true>,
        q40_gemm_kernel<5, false, TILED, WD, gemm_dma_slots(5), true>, q40_gemm_kernel<6, false, TILED, WD, gemm_dma_slots(6), true>,
        q40_gemm_kernel<7, false, TILED, WD, gemm_dma_slots(7), true>, q40_gemm_kernel<8, false, TILED, WD, gemm_dma_slots(8), true>};
    static const gemm_kernel_t range_cut[9] = {
        nullptr, q40_gemm_kernel<2, false, TILED, WD, gemm_dma_slots(2), true, true>, q40_gemm_kernel<2, false, TILED, WD, gemm_dma_slots(2), true, true>,
        q40_gemm_kernel<3, false, TILED, WD, gemm_dma_slots(3), true, true>, q40_gemm_kernel<4, false, TILED, WD, gemm_dma_slots(4), true, true>,
        q40_gemm_kernel<5, false, TILED, WD, gemm_dma_slots(5), true, true>, q40_gemm_kernel<6, false, TILED, WD, gemm_dma_slots(6), true, true>,
        q40_gemm_kernel<7, false, TILED, WD, gemm_dma_slots(7), true, true>, q40_gemm_kernel<8, false, TILED, WD, gemm_dma_slots(8), true, true>};
    // blocks of 64 .. 128 rows with RoPE (a kernel of its own: with the factors' registers in the others' epilogue three layers of a 70B shape took 1.2 % longer at 384 rows)
    static const gemm_kernel_t rotate[2][5] = {{q40_gemm_kernel<4, false, true, WD, GEMM_STAGES, false, false, false, true>, q40_gemm_kernel<5, false, true, WD, GEMM_STAGES, false, false, false, true>,
                                                q40_gemm_kernel<6, false, true, WD, GEMM_STAGES, false, false, false, true>, q40_gemm_kernel<7, false, true, WD, GEMM_STAGES, false, false, false, true>,
                                                q40_gemm_kernel<8, false, true, WD, GEMM_STAGES, false, false, false, true>},
                                               {q40_gemm_kernel<4, false, true, WD, gemm_dma_slots(4), true, false, false, true>, q40_gemm_kernel<5, false, true, WD, gemm_dma_slots(5), true, false, false, true>,
                                                q40_gemm_kernel<6, false, true, WD, gemm_dma_slots(6), true, false, false, true>, q40_gemm_kernel<7, false, true, WD, gemm_dma_slots(7), true, false, false, true>,
                                                q40_gemm_kernel<8, false, true, WD, gemm_dma_slots(8), true, false, false, true>}};
    // K not a multiple of 32: on tiled weights one kernel for all row counts, on the checkpoint layout the two forms from above with
    // a masked last step (against one four-wave kernel of eight row tiles: 33
    // rows x 11008 x 4072 29.7 -> 19.4 us, 100 rows 34.5 -> 27.6, 20 x 28672 x 8200 103 -> 53, 512 x 4096 x 4104 50 -> 40)
    static const gemm_kernel_t ragged = q40_gemm_kernel<8, true, TILED, 4>;
    static const gemm_kernel_t ragged_four[9] = {nullptr, q40_gemm_kernel<2, true, false, 4>, q40_gemm_kernel<2, true, false, 4>, q40_gemm_kernel<3, true, false, 4>,
                                                 q40_gemm_kernel<4, true, false, 4>, q40_gemm_kernel<5, true, false, 4>, q40_gemm_kernel<6, true, false, 4>,
                                                 q40_gemm_kernel<7, true, false, 4>, q40_gemm_kernel<8, true, false, 4>};
    static const gemm_kernel_t ragged_dma_wave[9] = {
        nullptr, q40_gemm_kernel<2, true, false, WD, gemm_dma_slots(2), true>, q40_gemm_kernel<2, true, false, WD, gemm_dma_slots(2), true>, q40_gemm_kernel<3, true, false, WD, gemm_dma_slots(3), true>,
        q40_gemm_kernel<4, true, false, WD, gemm_dma_slots(4), true>, q40_gemm_kernel<5, true, false, WD, gemm_dma_slots(5), true>, q40_gemm_kernel<6, true, false, WD, gemm_dma_slots(6), true>,
        q40_gemm_kernel<7, true, false, WD, gemm_dma_slots(7), true>, q40_gemm_kernel<8, true, false, WD, gemm_dma_slots(8), true>};
    // more than 64 KB of dynamic LDS has to be allowed once per kernel (the attribute is not stream work,
    // so a launch under graph capture is not affected)
    static const hipError_t lds_ok = [] {
        hipError_t e = hipFuncSetAttribute((const void *)ragged, hipFuncAttributeMaxDynamicSharedMemorySize, GEMM_LDS);
        for (int t = 2; t <= 8 && e == hipSuccess; ++t) {
            const std::pair<gemm_kernel_t, int> all[5] = {{exact[t], GEMM_LDS}, {ragged_four[t], GEMM_LDS}, {with_dma_wave[t], gemm_dma_slots(t) * GS_BYTES},
                                                          {range_cut[t], gemm_dma_slots(t) * GS_BYTES}, {ragged_dma_wave[t], gemm_dma_slots(t) * GS_BYTES}};
            for (int i = 0; i < 5 && e == hipSuccess; ++i)
                e = hipFuncSetAttribute((const void *)all[i].first, hipFuncAttributeMaxDynamicSharedMemorySize, all[i].second);
            for (int i = 0; TILED && t >= 4 && i < 2 && e == hipSuccess; ++i)
                e = hipFuncSetAttribute((const void *)rotate[i][t - 4], hipFuncAttributeMaxDynamicSharedMemorySize, i == 0 ? GEMM_LDS : gemm_dma_slots(t) * GS_BYTES);
        }
        return e;
    }();
    if (lds_ok != hipSuccess) {
        set_error("q40 gemm: the kernels' LDS could not be reserved: %s", hipGetErrorString(lds_ok));
        return (int)lds_ok;
    }
    SMH_REQUIRE((long)p.M * p.lda * 2 < (1L << 32), "q40 gemm: M x lda = %d x %ld exceeds the 32-bit lane offsets of A", p.M, p.lda);
    const int tiles = max(2, p.mblocks > 1 ? p.block_rows / 16 : (p.M + 15) / 16);
    const bool odd_k = p.K % 32 != 0;
    // (Whole column units go to an XCD, so with few of them an XCD can get more than its 32 workgroups although the launch has fewer than
    // 256: those wait for a second round unless they share a compute unit, which four-wave workgroups do.  Where they are short that is
    // the better way: 26 x 7168 x 1984 14.3 against 16.2 us, 93 x 5504 x 5792 26.1 against 29.1; from 25 steps on level or worse: 73 x
    // 4736 x 15840 43.7 against 41.4, 45 x 21120 x 18728 152 against 141.)
    const bool crowded = !TILED && (long)(p.units_pad / 8) * p.mblocks * p.ksplit > GEMM_DMA_WAVE_MAX_WGS / 8 && p.steps_per_slice <= 24;
    const bool one_each = !(TILED && odd_k) && (p.chunk > 0 || ((long)p.units * p.mblocks * p.ksplit <= GEMM_DMA_WAVE_MAX_WGS && !crowded));
    const bool four = odd_k ? !one_each : !TILED && !one_each;
    const gemm_kernel_t kern = p.rope_cos != nullptr ? rotate[one_each][p.block_rows / 16 - 4] : odd_k ? (TILED ? ragged : (one_each ? ragged_dma_wave : ragged_four)[tiles])
                                     : (p.chunk > 0 ? range_cut : one_each ? with_dma_wave : exact)[tiles];
    const long total_steps = (long)p.units * ((p.K + 31) / 32);
    const int lds = one_each ? gemm_dma_slots(tiles) * GS_BYTES : GEMM_LDS, threads = one_each ? 64 * (WD + GEMM_DMA_WAVES) : four ? GEMM_THREADS : 64 * W;
    if (p.chunk > 0) {
        hipLaunchKernelGGL(kern, dim3((unsigned)((total_steps + p.chunk - 1) / p.chunk)), dim3(threads), lds, stream, p);
        return launch_status();
    }
    return gemm_launch_rows(kern, p, threads, lds, stream);
}

// The checkpoint layout's plan for q40_gemm_kg_kernel in the place of p's: one weight, 17 rows and more, never more slabs than p's (whose workspace holds
// them), none where a workgroup has all of K.
// It has half the slabs for as many workgroups, or one workgroup a compute unit where p has two of half the waves, but fetches half a line of weights
// and as many lines of scales for half the columns: per 64 rows of K it takes 0.15 us more than two steps of the 256-column units, and up to 20 % more where
// rows lie a large power of two apart.  So it is taken
//   * where p has at most 256 workgroups, of which one XCD gets more than its 32 compute units hold at a time: 21 shapes 1.24 .. 1.85 times as fast;
//   * where p has one workgroup a compute unit: up to 20 stages (64 rows of K each) a workgroup, above 64 rows 24: 48 shapes 1.02 .. 1.41 times
//     (above that 0.76 .. 1.07: 37 x 4096 x 11008, 22 stages, 17.1 us and 18.0, 100 x 12288 x 4096, 32 stages, 26.0 and 28.3);
//   * where p's are more, or cut at runs of steps: up to 48 stages, above 64 rows 64: 10 shapes 1.05 .. 1.64 (20 x 24576 x 4096, 64 stages, 26.1 us and
//     32.0; 80 x 22400 x 15208 109.6 and 133);
//   * above 128 rows, on p's row blocks, where K is cut, p has not that form already and half the compute units get work: up to 40 stages, 46 shapes of 130 .. 512 rows 1.02 .. 1.52 times
//     (us, 512 x 4096 x 4096 32.1 and 28.3, 300 rows 24.1 and 22.0, 242 x 5888 x 1176 20.4 and 13.4; of 41 to 45 stages 0.99 .. 1.07, of 86 0.91 and 0.92, of 191 0.81).
// us of both launches, in turn: 100 x 4096 x 4096 18.8 and 15.5, 20 x 4096 x 4096 11.4 and 9.8, 100 x 5120 x 5120 28.5 and 17.9, 37 x 7168 x 7168 26.2 and
// 19.1, 100 x 6400 x 3000 26.7 and 18.5, 100 x 24064 x 1928 35.3 and 24.7.
bool gemm_blocks_fit(const MatmulParams &p, MatmulParams &b) {
    // (half a stage past a K that is a multiple of 32 would meet an infinite activation with a zero)
    if (p.tiled || p.kgroups == 2 || p.nseg != 1 || p.M <= SMH_GEMV_MAX_M || p.K > 16384 || p.K % 64 == 32) return false;
    const bool many = p.M > GEMM_BM;
    const int blocks = p.seg[0].N / 128, mblocks = many ? p.mblocks : blocks <= 32 && p.M > 64 && p.K <= 4096 ? 2 : 1, steps = (p.K + 31) / 32;
    if ((long)blocks * mblocks > 256) return false;
    const int on_xcd = p.units_pad / 4 * mblocks;              // workgroups of a K-slice on the busiest XCD
    const int ks = min(min(256 / (blocks * mblocks), 32 / on_xcd), min(p.ksplit, steps / 8));
    if (ks < 1 || blocks * mblocks * ks < (many ? 128 : 170)) return false;
    b = p;
    b.kgroups = 2;
    b.mblocks = mblocks;
    if (!many) b.block_rows = mblocks == 2 ? 64 : GEMM_BM;
    b.chunk = 0;
    b.steps_per_slice = ((steps + ks - 1) / ks + 1) / 2 * 2;   // a stage of the ring is two steps
    b.ksplit = (steps + b.steps_per_slice - 1) / b.steps_per_slice;
    if (many) return b.steps_per_slice <= 80;
    const bool one_round = p.chunk == 0 && (long)p.units * p.mblocks * p.ksplit <= 256;
    if (one_round && p.units_pad / 8 * p.mblocks * p.ksplit > 32) return true;
    return b.steps_per_slice / 2 <= (one_round ? (p.M <= 64 ? 20 : 24) : (p.M <= 64 ? 48 : 64));
}

typedef void (*gemm_kg_kernel_t)(MatmulParams);
static int gemm_kg_launch(const MatmulParams &p, hipStream_t stream) {
#define KG_KERNELS(one, ...) {nullptr, one, q40_gemm_kg_kernel<2, __VA_ARGS__>, q40_gemm_kg_kernel<3, __VA_ARGS__>, q40_gemm_kg_kernel<4, __VA_ARGS__>, \
                         q40_gemm_kg_kernel<5, __VA_ARGS__>, q40_gemm_kg_kernel<6, __VA_ARGS__>, q40_gemm_kg_kernel<7, __VA_ARGS__>, q40_gemm_kg_kernel<8, __VA_ARGS__>}
    static const gemm_kg_kernel_t kern[3][9] = {KG_KERNELS((q40_gemm_kg_kernel<1, true, false>), true, false), KG_KERNELS(nullptr, false, false), KG_KERNELS(nullptr, false, true)};
#undef KG_KERNELS
    static const int lds_bytes[9] = {0, KgShape<1>::LDS, KgShape<2>::LDS, KgShape<3>::LDS, KgShape<4>::LDS, KgShape<5>::LDS, KgShape<6>::LDS, KgShape<7>::LDS, KgShape<8>::LDS};
    static const hipError_t lds_ok = [] {
        hipError_t e = hipSuccess;
        for (int t = 1; t <= 8; ++t)
            for (int form = 0; form < 3 && e == hipSuccess; ++form)
                if (kern[form][t] != nullptr) e = hipFuncSetAttribute((const void *)kern[form][t], hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes[t]);
        return e;
    }();
    if (lds_ok != hipSuccess) {
        set_error("q40 gemm: the kernels' LDS could not be reserved: %s", hipGetErrorString(lds_ok));
        return (int)lds_ok;
    }
    SMH_REQUIRE((long)p.M * p.lda * 2 < (1L << 32), "q40 gemm: M x lda = %d x %ld exceeds the 32-bit lane offsets of A", p.M, p.lda);
    int tiles = p.mblocks > 1 ? p.block_rows / 16 : (p.M + 15) / 16;
    if (tiles < 2 && !p.tiled) tiles = 2;
    const int form = p.tiled ? 0 : p.K % 32 == 0 ? 1 : 2;
    hipLaunchKernelGGL(kern[form][tiles], dim3((unsigned)(2 * p.units_pad), (unsigned)p.mblocks, (unsigned)p.ksplit), dim3(64 * (8 + GEMM_DMA_WAVES)), lds_bytes[tiles], stream, p);
    return launch_status();
}

// Can w1|w3 of these dimensions run with SwiGLU inside the launch, and is it the faster way?  Above 128 rows always (K a multiple
// of 32; the two-launch form writes and reads 8 bytes of slabs per gate and up value: 62 of 426 us at 2047 rows of the 7B
// shape).  Up to 128 rows: K a multiple of
// 64, two weights of n_half columns (a multiple of 128) whose 2 * n_half / 128 workgroups fit the compute units in one round;
// `worth_it`: and fill at least half of them (narrower weights are faster as two kernels with a K-split; w1|w3 + SiLU of the 7B shape 38.1 against
// 44.9 us at 100 rows, 29.1 against 31.5 at 64, level at 32).  From how many rows on is for the caller: smh_q40_swiglu_fits says 33, layer calls behind a longer
// prompt 5 (as_blocks) and 17 (swiglu_inside).
bool gemm_swiglu_fits(int M, int K, int n_half, bool worth_it) {
    if (M < 1 || K <= 0 || n_half <= 0 || n_half % 128 != 0) return false;
    if (M > GEMM_BM) return K % 32 == 0;                        // gemm_swiglu_rows_launch
    if (K % 64 != 0) return false;
    const int wgs = 2 * (n_half / 128);
    return wgs <= 256 && (!worth_it || wgs >= 128);
}

int swiglu_idle(int n_half) { return n_half / 64 < 256 ? (256 - n_half / 64) / 8 * 8 : 0; }

int gemm_swiglu_launch(const MatmulParams &p, const WarmWeights &next, hipStream_t stream) {
#define SWIGLU_KERNELS(...) {nullptr, q40_gemm_swiglu_kernel<1 __VA_ARGS__>, q40_gemm_swiglu_kernel<2 __VA_ARGS__>, q40_gemm_swiglu_kernel<3 __VA_ARGS__>, \
                             q40_gemm_swiglu_kernel<4 __VA_ARGS__>, q40_gemm_swiglu_kernel<5 __VA_ARGS__>, q40_gemm_swiglu_kernel<6 __VA_ARGS__>, \
                             q40_gemm_swiglu_kernel<7 __VA_ARGS__>, q40_gemm_swiglu_kernel<8 __VA_ARGS__>}
    typedef void (*plain_t)(MatmulParams);
    typedef void (*ask_t)(MatmulParams, WarmWeights);
    static const plain_t plain[9] = SWIGLU_KERNELS();
    static const ask_t asking[9] = SWIGLU_KERNELS(, WarmWeights);
#undef SWIGLU_KERNELS
    static const int lds_bytes[9] = {0, SwigluShape<1>::LDS, SwigluShape<2>::LDS, SwigluShape<3>::LDS, SwigluShape<4>::LDS, SwigluShape<5>::LDS, SwigluShape<6>::LDS,
                                     SwigluShape<7>::LDS, SwigluShape<8>::LDS};
    static const hipError_t lds_ok = [] {
        hipError_t e = hipSuccess;
        for (int t = 1; t <= 8 && e == hipSuccess; ++t) {
            e = hipFuncSetAttribute((const void *)plain[t], hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes[t]);
            if (e == hipSuccess) e = hipFuncSetAttribute((const void *)asking[t], hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes[t]);
        }
        return e;
    }();
    if (lds_ok != hipSuccess) {
        set_error("q40 gemm: the kernels' LDS could not be reserved: %s", hipGetErrorString(lds_ok));
        return (int)lds_ok;
    }
    SMH_REQUIRE((long)p.M * p.lda * 2 < (1L << 32), "q40 gemm: M x lda = %d x %ld exceeds the 32-bit lane offsets of A", p.M, p.lda);
    const int tiles = (p.M + 15) / 16;
    const dim3 grid((unsigned)(2 * (p.seg[0].N / 128) + next.workgroups)), threads(64 * (8 + GEMM_DMA_WAVES));
    if (next.workgroups > 0) hipLaunchKernelGGL(asking[tiles], grid, threads, lds_bytes[tiles], stream, p, next);
    else hipLaunchKernelGGL(plain[tiles], grid, threads, lds_bytes[tiles], stream, p);
    return launch_status();
}

// More than 128 rows (a prefill) on tiled weights: without a K-split a launch stores fp16 results itself - no fp32 slabs (4 bytes
// an output and slice written here and read behind) and no kernel to add them.
bool gemm_direct_fits(const MatmulParams &p) { return p.tiled && p.M > GEMM_BM && p.K % 32 == 0 && p.ksplit == 1; }

// Both forms of SwiGLU above 128 rows planned: p in workgroups of two pieces of each weight, w of three; true: w promises more.
static bool gemm_swiglu_rows_plan(MatmulParams &p, MatmulParams &w) {
    p.units = p.seg[0].N / 128;
    p.units_pad = (p.units + 7) / 8 * 8;
    w.units = (p.seg[0].N / 64 + 2) / 3;
    w.units_pad = (w.units + 7) / 8 * 8;
    const float narrow_us = gemm_plan_rows(p, p.K / 32, 1, ROWS_256);
    return gemm_plan_rows(w, p.K / 32, 1, ROWS_384) < narrow_us;
}
int gemm_swiglu_columns(MatmulParams p) {
    if (p.M <= GEMM_BM) return 128;
    MatmulParams w = p;
    return gemm_swiglu_rows_plan(p, w) ? 384 : 256;
}

// w.units columns of workgroups of three pieces, w.mblocks row blocks, need rounds of which the last can be a poor one (w1|w3 of the 7B shape at 2047 rows: 928
// workgroups, 3.6 rounds): the units of a first launch where a second one of two pieces of each weight a workgroup (256 columns) for the columns behind
// them promises 3 % less, 0: none does.  Rounds on the busiest XCD, without what full ones cost in clock.  45 launches at 430 .. 2047 rows of the 7B, 13B, 34B and
// 70B shapes and of 4096 -> 2 x 14336, promised 0.82 .. 0.96 of one launch's time: 0.89 .. 0.99 (us, 4096 -> 2 x 11008 at 2047 rows 336 and 324, at 1720 317 and
// 302; 8192 -> 2 x 28672 at 430 rows 442 and 395, at 1965 1607 and 1564).
static int gemm_swiglu_split(const MatmulParams &w, int pieces, int steps) {
    auto rounds = [&](int units) { return ((units + 7) / 8 * w.mblocks + 31) / 32; };
    auto us = [&](const RowsCost &c) { return (float)steps * (c.step + c.per_rows * w.block_rows / GEMM_BM) + c.around; };
    const float wide = us(ROWS_384), narrow = us(ROWS_256);
    float least = 0.97f * rounds(w.units) * wide;
    int first = 0;
    for (int units = 8; units < w.units; units += 8) {
        const float t = rounds(units) * wide + rounds((pieces - 3 * units + 1) / 2) * narrow;
        if (t < least) {
            least = t;
            first = units;
        }
    }
    return first;
}

int gemm_swiglu_first_columns(MatmulParams p) {
    MatmulParams w = p;
    return p.M > GEMM_BM && gemm_swiglu_rows_plan(p, w) ? 192 * gemm_swiglu_split(w, p.seg[0].N / 64, p.K / 32) : 0;
}

int gemm_swiglu_rows_launch(MatmulParams p, hipStream_t stream) {
    // (blocks of 64 .. 128 rows)
    static const gemm_kernel_t plain[5] = {q40_gemm_kernel<4, false, true, 8, GEMM_STAGES, false, false, true>, q40_gemm_kernel<5, false, true, 8, GEMM_STAGES, false, false, true>, q40_gemm_kernel<6, false, true, 8, GEMM_STAGES, false, false, true>,
                                           q40_gemm_kernel<7, false, true, 8, GEMM_STAGES, false, false, true>, q40_gemm_kernel<8, false, true, 8, GEMM_STAGES, false, false, true>};
    static const gemm_kernel_t dma_wave[5] = {q40_gemm_kernel<4, false, true, 8, gemm_dma_slots(4), true, false, true>, q40_gemm_kernel<5, false, true, 8, gemm_dma_slots(5), true, false, true>, q40_gemm_kernel<6, false, true, 8, gemm_dma_slots(6), true, false, true>,
                                              q40_gemm_kernel<7, false, true, 8, gemm_dma_slots(7), true, false, true>, q40_gemm_kernel<8, false, true, 8, gemm_dma_slots(8), true, false, true>};
    static const gemm_kernel_t wide[5] = {q40_gemm_wide_kernel<4, WIDE_SWIGLU>, q40_gemm_wide_kernel<5, WIDE_SWIGLU>, q40_gemm_wide_kernel<6, WIDE_SWIGLU>,
                                          q40_gemm_wide_kernel<7, WIDE_SWIGLU>, q40_gemm_wide_kernel<8, WIDE_SWIGLU>};
    static const int wide_lds[5] = {WideShape<4, WIDE_SWIGLU>::LDS, WideShape<5, WIDE_SWIGLU>::LDS, WideShape<6, WIDE_SWIGLU>::LDS, WideShape<7, WIDE_SWIGLU>::LDS, WideShape<8, WIDE_SWIGLU>::LDS};
    static const hipError_t lds_ok = [] {
        hipError_t e = hipSuccess;
        for (int t = 0; t < 5 && e == hipSuccess; ++t) {
            e = hipFuncSetAttribute((const void *)wide[t], hipFuncAttributeMaxDynamicSharedMemorySize, wide_lds[t]);
            if (e == hipSuccess) e = hipFuncSetAttribute((const void *)plain[t], hipFuncAttributeMaxDynamicSharedMemorySize, GEMM_LDS);
            if (e == hipSuccess) e = hipFuncSetAttribute((const void *)dma_wave[t], hipFuncAttributeMaxDynamicSharedMemorySize, gemm_dma_slots(t + 4) * GS_BYTES);
        }
        return e;
    }();
    if (lds_ok != hipSuccess) {
        set_error("q40 gemm: the kernels' LDS could not be reserved: %s", hipGetErrorString(lds_ok));
        return (int)lds_ok;
    }
    SMH_REQUIRE((long)p.M * p.lda * 2 < (1L << 32), "q40 gemm: M x lda = %d x %ld exceeds the 32-bit lane offsets of A", p.M, p.lda);
    p.kgroups = 0;
    MatmulParams w = p;
    if (gemm_swiglu_rows_plan(p, w)) {
        const int t = w.block_rows / 16 - 4, pieces = p.seg[0].N / 64, first = gemm_swiglu_split(w, pieces, p.K / 32);
        w.ksplit = 1;
        if (first > 0) w.units = w.units_pad = first;
        const int st = gemm_launch_rows(wide[t], w, 64 * (WIDE_WAVES + GEMM_DMA_WAVES), wide_lds[t], stream);
        if (st || first == 0) return st;
        // the columns behind the first launch's: 3 pieces a unit, a multiple of 12 blocks of 128
        const int blocks = 3 * first / 2;
        for (int i = 0; i < 2; ++i) {
            p.seg[i].w += (long)(blocks / 2) * tiled_steps(p.K) * TILE_BYTES;
            p.seg[i].N -= 128 * blocks;
        }
        p.seg[0].c += 128 * blocks;
        p.units = p.seg[0].N / 128;
        p.units_pad = (p.units + 7) / 8 * 8;
        p.mblocks = w.mblocks;
        p.block_rows = w.block_rows;
    }
    const bool one_each = (long)p.units * p.mblocks <= GEMM_DMA_WAVE_MAX_WGS;
    const int t = p.block_rows / 16 - 4;
    p.ksplit = 1;
    return gemm_launch_rows((one_each ? dma_wave : plain)[t], p, 512 + (one_each ? 64 * GEMM_DMA_WAVES : 0), one_each ? gemm_dma_slots(t + 4) * GS_BYTES : GEMM_LDS, stream);
}

// The launch of a direct product whose plan has no K-split, with workgroups of three pieces and two K-groups or of six pieces where they
// promise more (slabs stay with gemm_fill_plan's kernel).  Returns the pieces, 0: neither.
static int gemm_wide_fits(const MatmulParams &p, MatmulParams &w) {
    if (!p.tiled || !p.direct || p.M <= GEMM_BM || p.ksplit != 1 || p.K % 32 != 0) return 0;
    int pieces = 0;
    w = p;
    float least = gemm_plan_rows(w, p.K / 32, 1, ROWS_256);
    for (int n = 3; n <= 6; n += 3) {
        if (n == 3 && p.K % 64 != 0) continue;
        MatmulParams t = p;
        t.units = (p.n_total / 64 + n - 1) / n;
        t.units_pad = (t.units + 7) / 8 * 8;
        const float us = gemm_plan_rows(t, p.K / 32, 1, n == 3 ? ROWS_192 : ROWS_SIX);
        if (us < 0.97f * least) {
            least = us;
            w = t;
            pieces = n;
        }
    }
    return pieces;
}
int gemm_direct_columns(MatmulParams p) {
    MatmulParams w;
    p.direct = 1;
    const int pieces = gemm_wide_fits(p, w);
    return pieces > 0 ? 64 * pieces : GEMM_COLS;
}
static int gemm_wide_launch(const MatmulParams &p, int pieces, hipStream_t stream) {
    static const gemm_kernel_t kern[2][5] = {{q40_gemm_wide_kernel<4, WIDE_GROUPS>, q40_gemm_wide_kernel<5, WIDE_GROUPS>, q40_gemm_wide_kernel<6, WIDE_GROUPS>,
                                              q40_gemm_wide_kernel<7, WIDE_GROUPS>, q40_gemm_wide_kernel<8, WIDE_GROUPS>},
                                             {q40_gemm_wide_kernel<4, WIDE_SIX>, q40_gemm_wide_kernel<5, WIDE_SIX>, q40_gemm_wide_kernel<6, WIDE_SIX>,
                                              q40_gemm_wide_kernel<7, WIDE_SIX>, q40_gemm_wide_kernel<8, WIDE_SIX>}};
    static const int lds_bytes[2][5] = {{WideShape<4, WIDE_GROUPS>::LDS, WideShape<5, WIDE_GROUPS>::LDS, WideShape<6, WIDE_GROUPS>::LDS,
                                         WideShape<7, WIDE_GROUPS>::LDS, WideShape<8, WIDE_GROUPS>::LDS},
                                        {WideShape<4, WIDE_SIX>::LDS, WideShape<5, WIDE_SIX>::LDS, WideShape<6, WIDE_SIX>::LDS, WideShape<7, WIDE_SIX>::LDS,
                                         WideShape<8, WIDE_SIX>::LDS}};
    static const hipError_t lds_ok = [] {
        hipError_t e = hipSuccess;
        for (int t = 0; t < 10 && e == hipSuccess; ++t)
            e = hipFuncSetAttribute((const void *)kern[t / 5][t % 5], hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes[t / 5][t % 5]);
        return e;
    }();
    if (lds_ok != hipSuccess) {
        set_error("q40 gemm: the kernels' LDS could not be reserved: %s", hipGetErrorString(lds_ok));
        return (int)lds_ok;
    }
    SMH_REQUIRE((long)p.M * p.lda * 2 < (1L << 32), "q40 gemm: M x lda = %d x %ld exceeds the 32-bit lane offsets of A", p.M, p.lda);
    const int six = pieces == 6 ? 1 : 0, t = p.block_rows / 16 - 4;
    return gemm_launch_rows(kern[six][t], p, 64 * (WIDE_WAVES + GEMM_DMA_WAVES), lds_bytes[six][t], stream);
}

int gemm_launch(const MatmulParams &p, hipStream_t stream) {
    MatmulParams w;
    if (const int pieces = gemm_wide_fits(p, w)) return gemm_wide_launch(w, pieces, stream);
    if (p.kgroups == 2) return gemm_kg_launch(p, stream);
    return p.tiled ? gemm_launch_layout<true>(p, stream) : gemm_launch_layout<false>(p, stream);
}

}  // namespace smh

