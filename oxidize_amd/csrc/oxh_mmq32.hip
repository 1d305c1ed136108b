/* oxh_mmq32.hip — the prefill matmul of the six 32-value formats (Q8_0, Q4_0, Q4_1, Q5_0, Q5_1, AL5_XS).
 *
 * Arithmetic.  Per (row, token, block) the reference adds (dw*dq)*(float)isum, for the _1 formats plus
 * (mw*dq)*(float)qsum, block after block (oxk.c:88-241).  A block is the K of one v_mfma_i32_16x16x32_i8; the
 * float step is the reference's, in its order, so every result has the single-vector dot's bits.  Codes with an
 * offset are staged as the signed values code - offset, so four formats share Q8_0's step exactly.
 *
 * What bounds it.  The float step: three vector instructions per result and block (seven for the _1 formats) beside a
 * 256th of an MFMA, at 2.6 cycles each on a SIMD of two or four waves.  So everything else has to stay off that port: a
 * block is fetched and taken apart ONCE per workgroup, by a lane that owns it (eight lanes along a row's consecutive
 * blocks, so that a wave's load touches some 24 cache lines and not 64), and goes to LDS as MFMA operands, int8 values and
 * scales; the inner loop issues MFMAs, the float step and little else but LDS reads.  The products of the scales come
 * from the matrix cores as well, four blocks to an instruction (`scales`): one of four vector instructions gone, and
 * three two-byte reads of LDS per sixteen tiles in the place of six of 16 bytes, on a pipe that was nearly as busy
 * (quantiser and matmul, us, in a run of that step alone: Q8_0 4096 x 4096 x 512 50.2 -> 48.4, 14336 x 4096 x 256 85.0 -> 81.1, Q4_0
 * 85.1 -> 81.7, AL5_XS 90.7 -> 87.6).  The _1 formats have two products and no registers for both: theirs stay vector
 * instructions.
 *
 * Shape.  A wave computes 16 rows x 32 tokens; eight waves, 64 rows x 64 tokens, to a workgroup and two workgroups to
 * a CU, or (WIDE) sixteen waves and 128 rows; four waves per SIMD either way, since one wave alone issues dependent
 * vector instructions 8.3 cycles apart and independent ones 4.7 to 5.4.  Steps of eight blocks, two stages in LDS, one
 * barrier per step; the next step's blocks go to LDS in the middle of a step and the ones after it are requested
 * then.  Of the Q8_0 tile's 92 % vector issue by counter, a third was not the float step: 64-bit addresses formed anew for
 * every block, the place within four bytes asked again, values cleared past the row's end.  With a wave's address in
 * scalar registers and 32-bit offsets, 269 of 317 instructions were left (in a run of that step: Q8_0 48.4 -> 45.3 and
 * 81.1 -> 75.5, Q4_0 81.7 -> 74.5, Q5_0 86.0 -> 79.4, AL5_XS 87.6 -> 80.7, Q4_1 112 -> 108, Q5_1 115 -> 113), and since
 * the wave's address moves and not the offsets, 262.  All steps of this comment and those beside the code in one run, us
 * before the first / now:
 *                       Q8_0       Q4_0       Q4_1        Q5_0       Q5_1        AL5_XS
 *   4096 x 4096 x 512   43.7/39.5  44.3/39.8  58.9/54.7   47.1/42.1  60.8/57.5   48.5/41.9
 *   900 x 8192 x 128    50.8/46.0  51.6/44.8  74.1/64.8   53.2/48.3  69.8/66.9   55.9/49.1
 *   333 x 14336 x 700   92.4/84.8  94.4/82.9  134.7/117.8 97.3/88.3  125.3/120.7 102.0/90.2
 * 128 x 64 tiles whose waves kept raw blocks in regions of their own, one workgroup to a CU, took 69 us where the kernel
 * before these steps took 41, eight waves of 32 x 32 42.5. */
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "oxhip.h"
#include "oxh_internal.h"
#include "oxh_device.inc"
#include "blocks32.inc"
#include "mmq_tiles.inc"

template <int LEG, bool WIDE> struct Mmq32Geom {
    static constexpr bool HAS_M = LEG == 2 || LEG == 4;
    static constexpr uint32_t BB = LEG == 0 ? 34u : LegGeom<LEG ? LEG : 1>::BYTES;
    static constexpr uint32_t RW = WIDE ? 8 : 4, TW = 2, RC = 1, TC = 2;   /* waves, 16-chunks of a wave */
    static constexpr uint32_t KP = 4, KB = 2u * KP;    /* pairs of blocks, blocks to a step */
    static constexpr uint32_t ROWS = RW * RC * 16u, TOK = TW * TC * 16u, THREADS = RW * TW * 64u;
    /* A stage.  Values: [pair][row or token][16-byte slot]: slot s of row r holds values 8k .. 8k+7 of the pair's
     * two blocks, k = s ^ mmq32_swizzle(r); a pair is skewed by a slot row.  Scales of rows [block][row], of tokens [four blocks][token][4]. */
    static constexpr uint32_t W_PAIR = ROWS * 64u, A_PAIR = TOK * 64u;
    static constexpr uint32_t D_PITCH = ROWS;
    static constexpr uint32_t A_OFF = KP * W_PAIR;
    static constexpr uint32_t DW_OFF = A_OFF + KP * A_PAIR;
    /* without minimums: the halves themselves, [row or token][block] */
    static constexpr uint32_t DQ_OFF = DW_OFF + (HAS_M ? KB * D_PITCH * 4u : ROWS * KB * 2u);
    static constexpr uint32_t MW_OFF = DQ_OFF + KB * TOK * (HAS_M ? 4u : 2u);
    static constexpr uint32_t QS_OFF = MW_OFF + (HAS_M ? KB * D_PITCH * 4u : 0u);
    static constexpr uint32_t STAGE_BYTES = QS_OFF + (HAS_M ? KB * TOK * 4u : 0u);
    static constexpr uint32_t LDS_BYTES = 2u * STAGE_BYTES;
    static_assert(THREADS == ROWS * KB && TOK * KB <= THREADS && TOK * KB % 64u == 0u && KP % 2u == 0u, "staging: a thread, a block of weights");
    static_assert((WIDE ? 1u : 2u) * LDS_BYTES <= 160u * 1024u, "workgroups to a CU");
};

/* Rows lie 64 bytes apart: eight aligned rows' slots of one k fall on the eight 16-byte pieces of 128 bytes, sixteen
 * rows' on the sixteen of 256. */
__device__ __forceinline__ uint32_t mmq32_swizzle(uint32_t row) { return ((row >> 1) & 3u) ^ ((row >> 3) & 1u); }

/* a half and three zeros: an operand of one K */
__device__ __forceinline__ v4h half_first(const uint8_t *p)
{
    uint32_t h = *reinterpret_cast<const uint16_t *>(p);
    asm("" : "+v"(h));          /* the load has cleared the upper half; seen as halves it would be cleared once more */
    return __builtin_bit_cast(v4h, make_uint2(h, 0u));
}

/* Where a lane's blocks lie: block `blk` of every step of eight, in row `row` of its wave's eight, as a 32-bit offset
 * (`first`) from the wave's base, which starts `lead` bytes below the wave's first row and moves on by a step at a time.  In
 * a last step that the row's end cuts short, lanes past the end stay on their block of the step before (`back`), in an
 * only step on the row's last one; `lead` leaves room for that and for an edge two bytes before a block.  So an offset
 * spans seven rows and two steps, which is below 2^32 in the longest rows oxh_mmq takes. */
struct Mmq32Walk {
    static constexpr uint32_t KB = 8u;
    static __host__ __device__ constexpr uint32_t lead(uint32_t bb) { return KB * bb + 2u; }
    static __host__ __device__ __forceinline__ uint32_t first(uint32_t row, uint32_t blk, uint32_t B, uint32_t bb)
    {
        return lead(bb) + (row * B + (blk < B ? blk : B - 1u)) * bb;
    }
    static __host__ __device__ __forceinline__ uint32_t back(uint32_t step, uint32_t blk, uint32_t B, uint32_t bb)
    {
        return step * KB + blk < B ? 0u : KB * bb;
    }
    static constexpr uint64_t reach(uint64_t B, uint32_t bb) { return lead(bb) + (7u * B + 2u * KB) * bb; }
};
static_assert(Mmq32Walk::reach(OXH_MMQ32_MAX_BLOCKS, 34u) <= 0xFFFFFFFFull, "a lane's offsets");

/* the byte of its wave's first row at which lane (row, blk) fetches its block of step `step` */
extern "C" uint64_t oxh_debug_mmq32_fetched(uint32_t block_bytes, uint32_t blocks, uint32_t row, uint32_t blk, uint32_t step)
{
    const uint32_t n_steps = (blocks + Mmq32Walk::KB - 1u) / Mmq32Walk::KB;
    const uint64_t base = (uint64_t)step * (Mmq32Walk::KB * block_bytes) - Mmq32Walk::lead(block_bytes);
    uint32_t off = Mmq32Walk::first(row, blk, blocks, block_bytes);
    if (step != 0u && step + 1u == n_steps) off -= Mmq32Walk::back(step, blk, blocks, block_bytes);
    return base + off;
}

template <int LEG> struct Mmq32Raw { LegRegs r; };
template <> struct Mmq32Raw<0> { Q80Regs r; };

template <int LEG, bool WIDE>
__global__ __launch_bounds__(WIDE ? 1024 : 512, 4) void
k_mmq_32(const uint8_t *__restrict__ w, uint32_t rows, uint32_t B, const uint8_t *__restrict__ acts, uint32_t nv,
         float *__restrict__ out, size_t out_stride, uint32_t n_row_tiles, uint32_t n_tok_tiles)
{
    typedef Mmq32Geom<LEG, WIDE> G;
    constexpr bool HAS_M = G::HAS_M;
    constexpr int RC = (int)G::RC, TC = (int)G::TC, KP = (int)G::KP;
    extern __shared__ __attribute__((aligned(16))) uint8_t mmq_lds[];
    /* workgroups whose numbers are equal modulo 8 share an XCD and its L2: the token tiles of a row tile get such
     * numbers, so a row tile's weights come from HBM once */
    const uint32_t place = blockIdx.x >> 3;
    const uint32_t row_tile = (place / n_tok_tiles) * 8u + (blockIdx.x & 7u), tok_tile = place % n_tok_tiles;
    if (row_tile >= n_row_tiles) return;
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t r16 = lane & 15u, kq = lane >> 4;
    const uint32_t row_first = row_tile * G::ROWS, tok_first = tok_tile * G::TOK;
    const uint32_t rows_here = min(rows - row_first, G::ROWS), toks_here = min(nv - tok_first, G::TOK);

    /* staging: this thread's blocks are block tid % KB of a step, rows (tokens) tid / KB and further ones */
    const uint32_t s_blk = tid % G::KB, s_row = tid / G::KB;
    uint32_t w_dst, a_dst;
    {
        const uint32_t k = (s_blk >> 1) & 3u;
        w_dst = (s_blk >> 1) * G::W_PAIR + s_row * 64u + 16u * (mmq32_swizzle(s_row) ^ k) + 8u * (s_blk & 1u);      /* ^ 16 k */
        a_dst = G::A_OFF + (s_blk >> 1) * G::A_PAIR + s_row * 64u + 16u * (mmq32_swizzle(s_row) ^ k) + 8u * (s_blk & 1u);
    }
    /* A wave stages eight rows (tokens).  Its base, in scalar registers, starts at the first one's address and goes a step
     * on at a time; a lane's block is a 32-bit offset from it, and so is its edge (Mmq32Walk).  Steps are a multiple of four
     * bytes in every format: a block's place within four is asked once. */
    static_assert(G::KB == Mmq32Walk::KB && G::KB * G::BB % 4u == 0u && G::KB * 34u % 4u == 0u, "blocks of a thread");
    const uint32_t wave_row = wave * (64u / G::KB);
    const uint32_t w_row0 = min(wave_row, rows_here - 1u), a_row0 = min(wave_row, toks_here - 1u);
    const uint8_t *w_base = w + (size_t)(row_first + w_row0) * B * G::BB - Mmq32Walk::lead(G::BB);
    const uint8_t *a_base = acts + (size_t)(tok_first + a_row0) * B * 34u - Mmq32Walk::lead(34u);
    uint32_t w_off = Mmq32Walk::first(min(s_row, rows_here - 1u) - w_row0, s_blk, B, G::BB);
    uint32_t a_off = Mmq32Walk::first(min(s_row, toks_here - 1u) - a_row0, s_blk, B, 34u);
    const uint32_t w_odd = block_odd(w_base + w_off), a_odd = block_odd(a_base + a_off);
    Mmq32Raw<LEG> w_raw;
    Q80Regs a_raw;
    constexpr bool W_EDGE = LEG == 0 || LegEdge<LEG ? LEG : 1>::ON;
    uint32_t w_edge = w_off + (w_odd ? 0u - 2u : G::BB - 4u), a_edge = a_off + (a_odd ? 0u - 2u : 30u);
    w_off += W_EDGE ? w_odd : 0u;
    a_off += a_odd;
    a_raw.shift = a_odd ? 0u : 16u;
    if constexpr (LEG == 0) w_raw.r.shift = w_odd ? 0u : 16u;
    else if (W_EDGE) w_raw.r.qh = w_odd ? 0u : 16u;
    /* on to step `step`, the steps in turn from 1; past the last it stays there */
    const uint32_t n_steps = (B + G::KB - 1u) / G::KB;
    uint32_t w_step = n_steps > 1u ? G::KB * G::BB : 0u, a_step = n_steps > 1u ? G::KB * 34u : 0u;
    auto advance = [&](uint32_t step) {
        w_base += w_step;
        a_base += a_step;
        if (__builtin_expect(step + 1u == n_steps, 0)) {
            asm volatile("");           /* once in a launch: a branch, and not selects in every step */
            const uint32_t w_back = Mmq32Walk::back(step, s_blk, B, G::BB), a_back = Mmq32Walk::back(step, s_blk, B, 34u);
            w_off -= w_back;
            w_edge -= w_back;
            a_off -= a_back;
            a_edge -= a_back;
            w_step = a_step = 0u;
        }
    };
    auto load = [&]() {
        if constexpr (LEG == 0) {
            w_raw.r.w0 = *reinterpret_cast<const U32x4a4g *>(w_base + w_off);
            w_raw.r.w1 = *reinterpret_cast<const U32x4a4g *>(w_base + w_off + 16);
            w_raw.r.edge = reinterpret_cast<const U32u2 *>(w_base + w_edge)->v;
        } else if constexpr (W_EDGE) {
            w_raw.r.qs = *reinterpret_cast<const U32x4a4g *>(w_base + w_off);
            w_raw.r.hdr = reinterpret_cast<const U32u2 *>(w_base + w_edge)->v;
        } else {
            leg_load_at<LEG>(w_raw.r, w_base + w_off, w_odd);
        }
        a_raw.w0 = *reinterpret_cast<const U32x4a4g *>(a_base + a_off);
        a_raw.w1 = *reinterpret_cast<const U32x4a4g *>(a_base + a_off + 16);
        a_raw.edge = reinterpret_cast<const U32u2 *>(a_base + a_edge)->v;
    };
    /* blocks past the row's end get zero scales (their values are another block's): their term is 0, which changes
     * nothing (a sum that starts at +0 never becomes -0) */
    auto put = [&](uint8_t *st, uint32_t dst, const uint32_t q[8]) {
#pragma unroll
        for (uint32_t k = 0; k < 4u; k++) *reinterpret_cast<uint2 *>(st + (dst ^ (16u * k))) = make_uint2(q[2 * k], q[2 * k + 1]);
    };
    auto store = [&](uint32_t step) {
        uint8_t *st = mmq_lds + (step & 1u) * G::STAGE_BYTES;
        const bool live = step * G::KB + s_blk < B;
        {
            const uint32_t r = s_row;
            uint32_t q[8], d;
            float m = 0.0f;
            if constexpr (LEG == 0) {
                d = q80_unpack(w_raw.r, q);
            } else {
                uint32_t lo[4], hi[4];
                d = leg_unpack<LEG>(w_raw.r, lo, hi);
                if (HAS_M) m = half_to_float_hw(w_raw.r.hdr >> 16);
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    /* code - offset as a signed byte: codes stay below 2 * offset, so no carry leaves a byte */
                    constexpr uint32_t UP = 0x01010101u * (128u - (uint32_t)LegGeom<LEG>::OFFSET);
                    q[k] = HAS_M ? lo[k] : (lo[k] + UP) ^ 0x80808080u;
                    q[4 + k] = HAS_M ? hi[k] : (hi[k] + UP) ^ 0x80808080u;
                }
            }
            put(st, w_dst, q);
            if (!HAS_M) reinterpret_cast<uint16_t *>(st + G::DW_OFF)[tid] = live ? (uint16_t)d : (uint16_t)0u;
            if (HAS_M) reinterpret_cast<float *>(st + G::DW_OFF)[s_blk * G::D_PITCH + r] = live ? half_to_float_hw(d) : 0.0f;
            if (HAS_M) reinterpret_cast<float *>(st + G::MW_OFF)[s_blk * G::D_PITCH + r] = live ? m : 0.0f;
        }
        if (!WIDE || wave < G::TOK * G::KB / 64u) {        /* the wide tile has more threads than token blocks */
            const uint32_t t = s_row;
            uint32_t q[8];
            const uint32_t d = q80_unpack(a_raw, q);
            put(st, a_dst, q);
            const uint32_t at = ((s_blk >> 2) * G::TOK + t) * 4u + (s_blk & 3u);
            if (!HAS_M) reinterpret_cast<uint16_t *>(st + G::DQ_OFF)[tid] = live ? (uint16_t)d : (uint16_t)0u;
            if (HAS_M) {
                reinterpret_cast<float *>(st + G::DQ_OFF)[at] = live ? half_to_float_hw(d) : 0.0f;
                int qs = 0;
#pragma unroll
                for (int k = 0; k < 8; k++) qs = dot4(0x01010101u, q[k], qs);
                reinterpret_cast<float *>(st + G::QS_OFF)[at] = (float)qs;
            }
        }
    };

    /* a wave's operands of one pair of blocks */
    struct Frag {
        u32x4 w[RC], a[TC];
        v4f dw[HAS_M ? 2 : 1][RC];
    };
    const uint32_t rw = wave % G::RW, tw = wave / G::RW;
    const uint32_t w_row = rw * (16u * G::RC) + r16, a_row = tw * (16u * G::TC) + r16;
    const uint32_t swz = 16u * (kq ^ mmq32_swizzle(r16));
    const uint32_t w_rd = w_row * 64u + swz, a_rd = G::A_OFF + a_row * 64u + swz;
    const uint32_t dw_rd = G::DW_OFF + (rw * (16u * G::RC) + 4u * kq) * 4u;
    const uint32_t dq_rd = G::DQ_OFF + a_row * 16u;
    const uint32_t dwh_rd = G::DW_OFF + w_row * (2u * G::KB) + 2u * kq;      /* halves: this lane's of four blocks is block kq's */
    auto fetch = [&](const uint8_t *st, int p) -> Frag {
        Frag f;
#pragma unroll
        for (int rc = 0; rc < RC; rc++) f.w[rc] = *reinterpret_cast<const u32x4 *>(st + (w_rd ^ (16u * ((uint32_t)p & 3u))) + (uint32_t)p * G::W_PAIR + 1024u * (uint32_t)rc);
#pragma unroll
        for (int tc = 0; tc < TC; tc++) f.a[tc] = *reinterpret_cast<const u32x4 *>(st + (a_rd ^ (16u * ((uint32_t)p & 3u))) + (uint32_t)p * G::A_PAIR + 1024u * (uint32_t)tc);
#pragma unroll
        for (int j = 0; j < (HAS_M ? 2 : 0); j++)
#pragma unroll
            for (int rc = 0; rc < RC; rc++) {
                const uint32_t at = ((2u * (uint32_t)p + (uint32_t)j) * G::D_PITCH + 16u * (uint32_t)rc) * 4u;
                f.dw[j][rc] = *reinterpret_cast<const v4f *>(st + dw_rd + at);
            }
        return f;
    };
    v4f acc[RC][TC];
#pragma unroll
    for (int rc = 0; rc < RC; rc++)
#pragma unroll
        for (int tc = 0; tc < TC; tc++) acc[rc][tc] = (v4f){ 0.0f, 0.0f, 0.0f, 0.0f };
    /* BIASED: the integer sums start at the bits of 1.5 * 2^23, as floats they are then that plus the sum, exactly (at most
     * 2^19 here in either direction), and a subtraction makes the sum of it, where a conversion takes nearly twice a
     * subtraction's time.  It costs four registers: AL5_XS 4096 x 4096 x 512 50.3 -> 47.9 us, Q4_0 46.0 -> 45.3, Q5_1 900 x
     * 8192 x 128 73.4 -> 71.0; Q5_0 as before; Q8_0 2048 x 2016 x 333 17.4 -> 18.3 and Q4_1 1000 x 2048 x 100 21.1 -> 21.4,
     * so not those three (all with a scheduling barrier between the pairs of a step, as it was then). */
    constexpr bool BIASED = LEG == 1 || LEG == 4 || LEG == 5;
    v4i start = { 0, 0, 0, 0 };
    if (BIASED) {
        start = (v4i){ 0x4B400000, 0x4B400000, 0x4B400000, 0x4B400000 };
        asm volatile("" : "+v"(start));         /* kept in registers, not made anew for every MFMA */
    }
    auto block_of = [](const u32x4 &v, int j) -> long {
        return (long)(((unsigned long)v[2 * j + 1] << 32) | (unsigned long)v[2 * j]);
    };
    /* dw * dq of four blocks: a product of two halves is an f32 exactly, and v_mfma_f32_16x16x4_4b_f16 is four outer
     * products side by side, block b from the operands of lanes 16 b .. 16 b + 15, the result where the integer
     * MFMA of the block has its own */
    auto scales = [&](const uint8_t *st, int q, v16f t[RC][TC]) {
        v4h a[RC], b[TC];
#pragma unroll
        for (int rc = 0; rc < RC; rc++)
            a[rc] = half_first(st + dwh_rd + 8u * (uint32_t)q + 16u * 2u * G::KB * (uint32_t)rc);
#pragma unroll
        for (int tc = 0; tc < TC; tc++)
            b[tc] = half_first(st + dq_rd + 2u * kq + 8u * (uint32_t)q + 16u * 2u * G::KB * (uint32_t)tc);
        const v16f none = {};
#pragma unroll
        for (int rc = 0; rc < RC; rc++)
#pragma unroll
            for (int tc = 0; tc < TC; tc++) t[rc][tc] = __builtin_amdgcn_mfma_f32_16x16x4f16(a[rc], b[tc], none, 0, 0, 0);
    };
    auto compute = [&](const Frag &f, const uint8_t *st, const v4f dq[TC], const v4f qs[TC], const v16f ts[RC][TC], int p) {
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const int bq = 2 * (p & 1) + j;
            v4i isum[RC][TC];
            v4f mw[RC];
#pragma unroll
            for (int rc = 0; rc < RC; rc++) {
#pragma unroll
                for (int tc = 0; tc < TC; tc++)
                    /* weights first: result i of a lane is row 4 kq + i against token r16 */
                    isum[rc][tc] = __builtin_amdgcn_mfma_i32_16x16x32_i8(block_of(f.w[rc], j), block_of(f.a[tc], j), start, 0, 0, 0);
                if (HAS_M)
                    mw[rc] = *reinterpret_cast<const v4f *>(st + dw_rd + (G::MW_OFF - G::DW_OFF) +
                                                            ((2u * (uint32_t)p + (uint32_t)j) * G::D_PITCH + 16u * (uint32_t)rc) * 4u);
            }
#pragma unroll
            for (int rc = 0; rc < RC; rc++)
#pragma unroll
                for (int tc = 0; tc < TC; tc++)
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const float t = HAS_M ? f.dw[HAS_M ? j : 0][rc][i] * dq[tc][bq] : ts[rc][tc][4 * bq + i];
                        const float sum = BIASED ? __int_as_float(isum[rc][tc][i]) - 12582912.0f : (float)isum[rc][tc][i];
                        const float up = t * sum;
                        if (HAS_M) {
                            const float tm = mw[rc][i] * dq[tc][bq];
                            const float off = tm * qs[tc][bq];
                            acc[rc][tc][i] += up + off;
                        } else {
                            acc[rc][tc][i] += up;
                        }
                    }
        }
    };

    load();
    store(0u);
    advance(1u);
    load();
    __syncthreads();
    for (uint32_t s = 0; s < n_steps; s++) {
        const uint8_t *st = mmq_lds + (s & 1u) * G::STAGE_BYTES;
        const uint32_t nb = min(B - s * G::KB, G::KB);
        advance(s + 2u);
        Frag cur = fetch(st, 0);
#pragma unroll
        for (int q = 0; q < KP / 2; q++) {
            if (4u * (uint32_t)q < nb) {
                v4f dq[TC], qs[TC];
                v16f ts[RC][TC];
                if (!HAS_M) scales(st, q, ts);
#pragma unroll
                for (int tc = 0; tc < TC; tc++) {
                    if (HAS_M) dq[tc] = *reinterpret_cast<const v4f *>(st + dq_rd + (uint32_t)q * G::TOK * 16u + 256u * (uint32_t)tc);
                    if (HAS_M) qs[tc] = *reinterpret_cast<const v4f *>(st + dq_rd + (G::QS_OFF - G::DQ_OFF) + (uint32_t)q * G::TOK * 16u + 256u * (uint32_t)tc);
                }
                /* (The compiler may mix this pair's reads with its sums.  Kept apart by a scheduling barrier, Q5_1 spilled three
                 * registers and Q4_1 and Q5_1 were slower, us: 900 x 8192 x 128 71.1 / 64.6 and 70.2 / 66.2, 4096 x 4096 x 512
                 * 62.9 / 61.2 and 65.8 / 63.3; the others within 1 %.) */
                const Frag nxt = fetch(st, 2 * q + 1);
                compute(cur, st, dq, qs, ts, 2 * q);
                if (q + 1 < KP / 2) cur = fetch(st, 2 * q + 2);
                __builtin_amdgcn_sched_barrier(0);
                compute(nxt, st, dq, qs, ts, 2 * q + 1);
            }
            if (q == 0 && s + 1u < n_steps) {
                store(s + 1u);
                load();
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        __syncthreads();
    }

    const bool wide = (out_stride & 3u) == 0u && ((uintptr_t)out & 15u) == 0u;
#pragma unroll
    for (int tc = 0; tc < TC; tc++) {
        const uint32_t tok = a_row + 16u * (uint32_t)tc;
        if (tok >= toks_here) continue;
        float *o = out + (size_t)(tok_first + tok) * out_stride + row_first;
#pragma unroll
        for (int rc = 0; rc < RC; rc++) {
            const uint32_t r = rw * (16u * G::RC) + 16u * (uint32_t)rc + 4u * kq;
            if (wide && r + 4u <= rows_here) {
                *reinterpret_cast<v4f *>(o + r) = acc[rc][tc];
            } else {
#pragma unroll
                for (int i = 0; i < 4; i++)
                    if (r + (uint32_t)i < rows_here) o[r + (uint32_t)i] = acc[rc][tc][i];
            }
        }
    }
}

template <int LEG> static hipError_t mmq32_raise(void)
{
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(k_mmq_32<LEG, false>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    if (e == hipSuccess)
        e = hipFuncSetAttribute(reinterpret_cast<const void *>(k_mmq_32<LEG, true>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    return e;
}

extern "C" int oxh_internal_mmq32_init(void)
{
    hipError_t e;
    if ((e = mmq32_raise<0>()) != hipSuccess || (e = mmq32_raise<1>()) != hipSuccess || (e = mmq32_raise<2>()) != hipSuccess ||
        (e = mmq32_raise<3>()) != hipSuccess || (e = mmq32_raise<4>()) != hipSuccess || (e = mmq32_raise<5>()) != hipSuccess)
        return (int)e;
    return (int)hipSuccess;
}

/* Workgroups: row tiles in runs of eight (one to an XCD) by token tiles. */
static uint64_t mmq32_tiles(size_t rows, size_t n_vec, uint32_t tile_rows)
{
    const uint64_t n_rt = (rows + tile_rows - 1u) / tile_rows, n_tt = (n_vec + 63u) / 64u;
    return (n_rt + 7u) / 8u * 8u * n_tt;
}

/* Which tile.  64 x 64, two to a CU, unless some XCD gets more of them than it has CUs and one round of 128 x 64 tiles, a
 * CU's worth of waves each, holds the launch on every XCD: then every CU gets the same and the smaller tiles' third more
 * staging shows (us, 64 / 128 rows: 4096 x 4096 x 512 42.7 / 42.2, Q5_1 60.3 / 57.7, 3072 x 2048 x 512 23.3 / 22.3).  With
 * fewer tiles a small one alone on its CU is done sooner (2048 x 2048 x 333 14.6 / 21.1), with more their rounds are finer
 * (5120 x 2048 x 512 33.0 / 41.2, 8192 rows 43.0 / 43.6, 14336 x 4096 x 512 136 / 149).  The XCD and not the device is what
 * fills: the row tiles are dealt to eight of them, and the first gets the odd ones with all their token tiles (4224 x 4096
 * under 448, 231 tiles of 128 rows, 35 of them on the first XCD's 32 CUs: 44.4 / 74.6; 2100 rows under 960 58.6 / 72.0).
 * Over 200 random launches near the lines the choice is 0.1 % above the faster tile, at most 5.5 % at 16 us; counted over
 * the whole device it was 4.3 %, at most 80 %. */
static bool mmq32_wide(size_t rows, size_t n_vec, size_t cus)
{
    const uint64_t xcd_cus = cus / 8u;
    auto busiest = [&](uint64_t tile_rows) { return mmq32_tiles(rows, n_vec, (uint32_t)tile_rows) / 8u; };
    return busiest(64u) > xcd_cus && busiest(128u) <= xcd_cus;
}

/* see oxh_internal.h */
extern "C" void oxh_internal_mmq32_tile(size_t rows, size_t n_vec, size_t cus, uint32_t tile[2])
{
    tile[0] = mmq32_wide(rows, n_vec, cus) ? Mmq32Geom<0, true>::ROWS : Mmq32Geom<0, false>::ROWS;
    tile[1] = Mmq32Geom<0, false>::TOK;
}

extern "C" int oxh_internal_mmq32_fits(size_t rows, size_t n_vec)
{
    return mmq32_tiles(rows, n_vec, Mmq32Geom<0, true>::ROWS) <= 0x7FFFFFFFull;
}

/* One launch, or several where the grid would reach the 2^32 threads that HIP takes in one dimension (8.4 million tiles:
 * 513 rows and 33.6 million tokens): row tiles first, then token tiles. */
template <int LEG, bool WIDE>
static void mmq32_launch(const void *d_w, size_t rows, size_t blocks, const void *d_acts, size_t n_vec, float *d_out,
                         size_t out_stride, hipStream_t st)
{
    typedef Mmq32Geom<LEG, WIDE> G;
    const size_t most = 0xFFFFFFFFull / G::THREADS / 8u * 8u;
    const size_t rows_each = rows < most * G::ROWS ? rows : most * G::ROWS;
    for (size_t r0 = 0; r0 < rows; r0 += rows_each) {
        const size_t r_here = rows - r0 < rows_each ? rows - r0 : rows_each;
        const uint32_t n_rt = (uint32_t)((r_here + G::ROWS - 1u) / G::ROWS);
        const size_t toks_each = most / ((n_rt + 7u) / 8u * 8u) * G::TOK;
        for (size_t t0 = 0; t0 < n_vec; t0 += toks_each) {
            const size_t t_here = n_vec - t0 < toks_each ? n_vec - t0 : toks_each;
            hipLaunchKernelGGL((k_mmq_32<LEG, WIDE>), dim3((uint32_t)mmq32_tiles(r_here, t_here, G::ROWS)), dim3(G::THREADS),
                               G::LDS_BYTES, st, (const uint8_t *)d_w + r0 * blocks * G::BB, (uint32_t)r_here, (uint32_t)blocks,
                               (const uint8_t *)d_acts + t0 * blocks * 34u, (uint32_t)t_here, d_out + t0 * out_stride + r0,
                               out_stride, n_rt, (uint32_t)((t_here + G::TOK - 1u) / G::TOK));
        }
    }
}

/* see oxh_internal.h */
extern "C" int oxh_internal_mmq32(int leg, const void *d_w, size_t rows, size_t blocks, const void *d_acts, size_t n_vec,
                                  float *d_out, size_t out_stride, size_t cus, void *stream)
{
    hipStream_t st = (hipStream_t)stream;
    const bool wide = mmq32_wide(rows, n_vec, cus);
#define OXH_M32(LEG) (wide ? mmq32_launch<LEG, true> : mmq32_launch<LEG, false>)(d_w, rows, blocks, d_acts, n_vec, d_out, out_stride, st)
    switch (leg) {
    case 1:  OXH_M32(1); break;
    case 2:  OXH_M32(2); break;
    case 3:  OXH_M32(3); break;
    case 4:  OXH_M32(4); break;
    case 5:  OXH_M32(5); break;
    default: OXH_M32(0); break;
    }
#undef OXH_M32
    return (int)hipGetLastError();
}
