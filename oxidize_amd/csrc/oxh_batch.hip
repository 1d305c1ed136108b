/* oxh_batch.hip — K-quant matrices under a small batch (at most 64 activations),
 * the super-blocks of a 16-row group shared between the waves of one workgroup.
 *
 * Arithmetic and operand layouts are those of mmq_tile() / mmq6_tile()
 * (mmq_tiles.inc; oxidize-c/src/compute/oxk.c:263-294, :870-897, :913-964), and so
 * are the bits: one f32 term per result and super-block, added up in block order.
 *
 * Why.  The tiles of mmq_tile() stage weights and activations through LDS for four
 * waves at a time and a workgroup walks its rows' super-blocks one after the other
 * behind a barrier each, so a matrix of few rows and many columns leaves most of
 * the device waiting (4096 x 14336, Q6_K: 64 tiles of 56 steps), and sharing a
 * tile's columns between workgroups costs a workspace of every term, written and
 * read (15 MB next to 48 MB of weights), and a second launch.  Here a workgroup owns 16
 * rows and all their columns; its waves take super-blocks in turn, each through an
 * LDS part of its own that nobody else waits for (two buffers, the next block's
 * loads under way while one is computed), and the terms meet in LDS, where they are
 * summed in order at the end.
 *
 * Why LDS at all: the memory pipeline charges for every cache line an instruction
 * touches, and loads in the operands' layout (16 rows, 64 bytes of each) touch
 * twice the lines of loads along a row's bytes: straight into registers 4096 x 14336
 * (Q6_K, 16 activations) took 29.6 us, this way 18.1, quantiser included; the split
 * tiles 26.
 * What bounds it: not settled.  48 MB in some 13 us is 3.7 TB/s; the compiled loop
 * has 209 vector instructions per super-block and wave (Q6_K, 16 activations), at 4
 * cycles each 5 us of it; each super-block begins with a wait for loads asked for one
 * super-block earlier. */
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "oxhip.h"
#include "oxh_internal.h"
#include "oxh_device.inc"
#include "mmq_tiles.inc"

enum { BAT_Q4 = 0, BAT_Q5 = 1, BAT_Q6 = 2, BAT_Q2W = 3 };

template <int FMT, int CH> struct BatGeom {
    static constexpr bool DMA = FMT == BAT_Q4 || FMT == BAT_Q5;         /* 16-byte aligned blocks: straight to LDS */
    static constexpr uint32_t WB = FMT == BAT_Q4 ? 144u : FMT == BAT_Q5 ? 176u : 210u;
    static constexpr uint32_t WP = DMA ? WB / 16u : 13u;                /* 16-byte pieces of a block */
    static constexpr uint32_t PIECES = 16u * WP, LOADS = (PIECES + 63u) / 64u;
    /* a wave's LDS: its 16 rows' blocks (two buffers where loads go straight there, one behind registers, 240
     * bytes a row: an odd number of 16-byte slots), then two buffers of the chunks' values, [token][slot] */
    static constexpr uint32_t W_PITCH = DMA ? WB : 240u, W_BYTES = 16u * W_PITCH;
    static constexpr uint32_t A_OFF = (DMA ? 2u : 1u) * W_BYTES, A_BYTES = CH * 4096u;
    static constexpr uint32_t WAVE_BYTES = A_OFF + 2u * A_BYTES;
};

/* the parts of a block that lane (r, kq) builds its operands from, out of row r's LDS image */
template <int FMT> struct BatRaw {
    u32x4 hdr;                  /* Q4/Q5: d, dmin, scales; Q6: the sixteen scales; Q2: minima and dmin */
    u32x4 v[4];                 /* Q4/Q5: two pieces of nibbles, two k steps each (mmq_tile()); Q6/Q2: ql, ql, qh, qh */
    u32x4 plane;                /* Q5: fifth bits */
    uint32_t d;                 /* Q6/Q2: f16 d */
};

template <int FMT>
__device__ __forceinline__ BatRaw<FMT> bat_read(const uint8_t *row, uint32_t kq)
{
    BatRaw<FMT> r;
    auto get = [&](uint32_t at) -> u32x4 { return *reinterpret_cast<const u32x4 *>(row + at); };
    r.plane = (u32x4){ 0u, 0u, 0u, 0u };
    r.d = 0u;
    if (FMT == BAT_Q4 || FMT == BAT_Q5) {
        r.hdr = get(0u);
        if (FMT == BAT_Q5) r.plane = get(16u + 16u * (kq & 1u));
#pragma unroll
        for (uint32_t p = 0; p < 2u; p++) r.v[p] = get((FMT == BAT_Q5 ? 48u : 16u) + 16u * kq + 64u * p);
    } else {
#pragma unroll
        for (uint32_t n = 0; n < 2u; n++) {
            r.v[n] = get(64u * n + 16u * kq);
            r.v[2u + n] = get(128u + 32u * n + 16u * (kq & 1u));
        }
        r.hdr = get(192u);
        r.d = *reinterpret_cast<const uint16_t *>(row + 208u);
    }
    return r;
}

/* the operands of a super-block: two (Q5_K: three) int8 chains, the minima of Q4_K / Q5_K as f16 */
template <int FMT> struct BatOps {
    v4i lo[4], hi[4], x[FMT == BAT_Q5 ? 4 : 1];
    v4h bm;
    float dw, dmin;
};

template <int FMT>
__device__ __forceinline__ BatOps<FMT> bat_build(const BatRaw<FMT> &r, uint32_t kq)
{
    BatOps<FMT> o;
    o.bm = (v4h){ (_Float16)0, (_Float16)0, (_Float16)0, (_Float16)0 };
    o.dmin = 0.0f;
    if (FMT == BAT_Q4 || FMT == BAT_Q5) {
        const uint32_t u0 = r.hdr.y, u1 = r.hdr.z, u2 = r.hdr.w, half = kq >> 1;
        const uint32_t sc_w[2] = { u0 & 0x3F3F3F3Fu, (u2 & 0x0F0F0F0Fu) | ((u0 >> 2) & 0x30303030u) };
        const uint32_t mn_lo = u1 & 0x3F3F3F3Fu, mn_hi = ((u2 >> 4) & 0x0F0F0F0Fu) | ((u1 >> 2) & 0x30303030u);
        const uint32_t mn2 = ((kq & 2u) ? mn_hi : mn_lo) >> (16u * (kq & 1u));
        const _Float16 m_even = (_Float16)(unsigned short)(mn2 & 0xFFu), m_odd = (_Float16)(unsigned short)((mn2 >> 8) & 0xFFu);
        o.bm = (v4h){ m_even, m_even, m_odd, m_odd };
        o.dw = half_to_float_hw(r.hdr.x & 0xFFFFu);
        o.dmin = half_to_float_hw(r.hdr.x >> 16);
#pragma unroll
        for (int gp = 0; gp < 4; gp++) {
            const uint32_t sc = (sc_w[gp >> 1] >> (16u * half + 8u * (uint32_t)(gp & 1))) & 0xFFu;
            const unsigned short sl = (unsigned short)(sc & 7u), sh = (unsigned short)(sc >> 3), sx = (unsigned short)(2u * sc);
            const v2u16 sl2 = { sl, sl }, sh2 = { sh, sh }, sx2 = { sx, sx };
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const v2u16 p = __builtin_bit_cast(v2u16, (gp & 1 ? r.v[gp >> 1][k] >> 4 : r.v[gp >> 1][k]) & 0x0F0F0F0Fu);
                o.lo[gp][k] = __builtin_bit_cast(int, (v2u16)(p * sl2));
                o.hi[gp][k] = __builtin_bit_cast(int, (v2u16)(p * sh2));
                if (FMT == BAT_Q5) {
                    const uint32_t fifth = (r.plane[k] >> (4u * (uint32_t)(gp >> 1) + 2u * half + (uint32_t)(gp & 1))) & 0x01010101u;
                    o.x[gp][k] = __builtin_bit_cast(int, (v2u16)(__builtin_bit_cast(v2u16, fifth) * sx2));
                }
            }
        }
    } else {
        o.dw = half_to_float_hw(r.d);
        if (FMT == BAT_Q2W) o.dmin = half_to_float_hw(r.hdr[2] & 0xFFFFu);
        const uint32_t h2 = 2u * (kq >> 1);
#pragma unroll
        for (int gp = 0; gp < 4; gp++) {
            const u32x4 ql = r.v[gp >> 1], qh = r.v[2 + (gp >> 1)];
            const uint32_t rot = (h2 + 4u * (uint32_t)(gp & 1) - 4u) & 31u;
            const int sc = __builtin_amdgcn_sbfe((int)r.hdr[gp], 8u * kq, 8u);
            const short scs = (short)sc, m32 = (short)(128 - 32 * sc);
            const v2i16 sc2 = { scs, scs }, off2 = { m32, m32 };
            const uint32_t mins = FMT == BAT_Q2W
                ? ((r.hdr[gp >> 1] >> (16u * (uint32_t)(gp & 1) + 4u * kq)) & 15u) * 0x01010101u : 0u;
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const uint32_t c = (((gp & 1) ? ql[k] >> 4 : ql[k]) & 0x0F0F0F0Fu) |
                                   (__builtin_amdgcn_alignbit(qh[k], qh[k], rot) & 0x30303030u);
                if (FMT == BAT_Q2W) {
                    o.lo[gp][k] = (int)c;
                    o.hi[gp][k] = (int)mins;
                    continue;
                }
                const v2i16 ce = __builtin_bit_cast(v2i16, __builtin_amdgcn_perm(c, c, 0x0C020C00u));
                const v2i16 co = __builtin_bit_cast(v2i16, __builtin_amdgcn_perm(c, c, 0x0C030C01u));
                const uint32_t ue = __builtin_bit_cast(uint32_t, (v2i16)(ce * sc2 + off2));
                const uint32_t uo = __builtin_bit_cast(uint32_t, (v2i16)(co * sc2 + off2));
                o.lo[gp][k] = (int)(__builtin_amdgcn_perm(uo, ue, 0x06020400u) ^ 0x80808080u);
                o.hi[gp][k] = (int)__builtin_amdgcn_perm(uo, ue, 0x07030501u);
            }
        }
    }
    return o;
}

/* LDS: every wave's own part, the chunks' token scales [block][token], the terms [block][chunk][token][row] */
template <int FMT, int CH> static inline uint32_t bat_lds_bytes(uint32_t B, uint32_t waves)
{
    return waves * BatGeom<FMT, CH>::WAVE_BYTES + B * CH * (64u + 1024u);
}

/* One workgroup's 16 rows under at most CH * 16 activations, all columns.  w0: the first row's blocks; a0: the first
 * activation; out: &out[first activation][first row].  TM: the tile-major layout, whose 16 blocks of a block index lie
 * next to each other (whole groups only). */
template <int FMT, int CH, bool TM>
__device__ __forceinline__ void
bat_tile(const uint8_t *__restrict__ w0, uint32_t rows_here, uint32_t B, const uint8_t *__restrict__ a0, uint32_t toks,
         float *__restrict__ out, size_t out_stride)
{
    typedef BatGeom<FMT, CH> G;
    extern __shared__ __attribute__((aligned(16))) uint8_t bat_lds[];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, waves = blockDim.x >> 6;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t r16 = lane & 15u, kq = lane >> 4;
    uint8_t *my = bat_lds + wave * G::WAVE_BYTES;
    const uint32_t my_at = (uint32_t)(size_t)(__attribute__((address_space(3))) uint8_t *)bat_lds + wave * G::WAVE_BYTES;
    float *s_dq = reinterpret_cast<float *>(bat_lds + waves * G::WAVE_BYTES), *s_term = s_dq + B * CH * 16u;
    const uint32_t act_stride = B * 292u;
    static_assert(!TM || G::DMA, "Q4_K and Q5_K have a tile-major form");
    constexpr uint32_t W_STEP = TM ? 16u * G::WB : G::WB;                /* from one super-block to the next */

    /* loads run along the contiguous bytes of a row's block and of a token's values; rows and tokens past the
     * last are the last again */
    uint32_t w_off[G::LOADS], w_dst[G::LOADS], q_off[CH * 4];
#pragma unroll
    for (uint32_t i = 0; i < G::LOADS; i++) {
        const uint32_t g = min(64u * i + lane, G::PIECES - 1u), r = g / G::WP, part = g - G::WP * r;
        w_off[i] = TM ? 16u * g : min(r, rows_here - 1u) * (B * G::WB) + 16u * part;
        w_dst[i] = r * G::W_PITCH + 16u * part;
    }
#pragma unroll
    for (uint32_t i = 0; i < CH * 4u; i++) {
        const uint32_t t = 4u * i + kq;
        q_off[i] = min(t, toks - 1u) * act_stride + 4u + 16u * (r16 ^ (t & 15u));
    }
    const uint32_t d_off = min(r16, rows_here - 1u) * (B * G::WB) + 208u;
    uint32_t s_off[CH];
#pragma unroll
    for (uint32_t c = 0; c < CH; c++) s_off[c] = min(16u * c + r16, toks - 1u) * act_stride + 260u + 8u * kq;

    struct { U32x4u2 q[G::DMA ? 1 : G::LOADS]; uint16_t d; } wr;         /* Q6/Q2: the next block on its way */
    uint2 sums[CH];                                                     /* Q4/Q5: its tokens' sums 4 kq .. + 3 */
    auto request = [&](uint32_t b, uint32_t buf) {
        const uint8_t *wb = w0 + (size_t)b * W_STEP, *ab = a0 + (size_t)b * 292u;
        if constexpr (G::DMA) {
#pragma unroll
            for (uint32_t i = 0; i < G::LOADS; i++)
                if (64u * (i + 1u) <= G::PIECES || 64u * i + lane < G::PIECES)
                    mmq_dma16<true>(wb, w_off[i], my_at + buf * G::W_BYTES + 1024u * i);
        } else {
#pragma unroll
            for (uint32_t i = 0; i < G::LOADS; i++) wr.q[i] = *reinterpret_cast<const U32x4u2 *>(wb + w_off[i]);
            wr.d = *reinterpret_cast<const uint16_t *>(wb + d_off);
        }
#pragma unroll
        for (uint32_t i = 0; i < CH * 4u; i++) mmq_dma16<true>(ab, q_off[i], my_at + G::A_OFF + buf * G::A_BYTES + 1024u * i);
        if constexpr (G::DMA) {
#pragma unroll
            for (uint32_t c = 0; c < CH; c++) {
                const uint32_t *s = reinterpret_cast<const uint32_t *>(ab + s_off[c]);
                sums[c] = make_uint2(s[0], s[1]);
            }
        }
    };
    /* the first super-block's loads, then the token scales, which every wave reads */
    request(min(wave, B - 1u), 0u);
    for (uint32_t i = tid; i < B * CH * 16u; i += blockDim.x) {
        const uint32_t b = i / (CH * 16u), t = i % (CH * 16u);
        s_dq[i] = *reinterpret_cast<const float *>(a0 + min(t, toks - 1u) * act_stride + b * 292u);
    }
    __syncthreads();

    /* the slot of this lane's values of step 0, and what the other steps change in it */
    const uint32_t a_rd = G::A_OFF + r16 * 256u + (((G::DMA ? 4u * (kq >> 1) + (kq & 1u) : kq) ^ r16) * 16u);
    auto a_step = [](int gp) -> uint32_t { return G::DMA ? 32u * ((uint32_t)gp & 1u) + 128u * ((uint32_t)gp >> 1) : 64u * (uint32_t)gp; };
    const v4i zero = { 0, 0, 0, 0 };
    const v4f fzero = { 0.0f, 0.0f, 0.0f, 0.0f };
    uint32_t buf = 0;
    for (uint32_t b = wave; b < B; b += waves, buf ^= 1u) {
        /* the block's loads have landed, and the reads of the buffer the next one's will fill are done (the
         * wave's own part of LDS: no barrier) */
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        if constexpr (!G::DMA) {
#pragma unroll
            for (uint32_t i = 0; i < G::LOADS; i++)
                if (64u * (i + 1u) <= G::PIECES || 64u * i + lane < G::PIECES)
                    *reinterpret_cast<u32x4 *>(my + w_dst[i]) = (u32x4){ wr.q[i].x, wr.q[i].y, wr.q[i].z, wr.q[i].w };
            *reinterpret_cast<uint16_t *>(my + r16 * G::W_PITCH + 208u) = wr.d;
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        }
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        uint2 sm[CH];
#pragma unroll
        for (int c = 0; c < CH; c++) sm[c] = sums[c];
        request(min(b + waves, B - 1u), buf ^ 1u);
        const BatOps<FMT> o = bat_build<FMT>(bat_read<FMT>(my + (G::DMA ? buf * G::W_BYTES : 0u) + r16 * G::W_PITCH, kq), kq);
#pragma unroll
        for (int c = 0; c < CH; c++) {
            v4i lo = zero, hi = zero;
#pragma unroll
            for (int gp = 0; gp < 4; gp++) {
                const v4i av = *reinterpret_cast<const v4i *>(my + (a_rd ^ a_step(gp)) + buf * G::A_BYTES + 4096u * (uint32_t)c);
                lo = __builtin_amdgcn_mfma_i32_16x16x64_i8(av, o.lo[gp], lo, 0, 0, 0);
                hi = __builtin_amdgcn_mfma_i32_16x16x64_i8(av, o.hi[gp], hi, 0, 0, 0);
                if (FMT == BAT_Q5) hi = __builtin_amdgcn_mfma_i32_16x16x64_i8(av, o.x[gp], hi, 0, 0, 0);
            }
            const float4 dq4 = *reinterpret_cast<const float4 *>(s_dq + (b * CH + (uint32_t)c) * 16u + 4u * kq);
            const float dqs[4] = { dq4.x, dq4.y, dq4.z, dq4.w };
            v4f mn = fzero;
            if (FMT == BAT_Q4 || FMT == BAT_Q5) {
                const v4h ab = { (_Float16)(short)(sm[c].x & 0xFFFFu), (_Float16)(short)(sm[c].x >> 16),
                                 (_Float16)(short)(sm[c].y & 0xFFFFu), (_Float16)(short)(sm[c].y >> 16) };
                mn = __builtin_amdgcn_mfma_f32_16x16x16f16(ab, o.bm, fzero, 0, 0, 0);
            }
#pragma unroll
            for (int i = 0; i < 4; i++) {
                float term;
                if (FMT == BAT_Q4 || FMT == BAT_Q5) {
                    const int pos = lo[i] + 8 * hi[i];
                    const float t_pos = o.dw * dqs[i], t_min = o.dmin * dqs[i];
                    const float up = t_pos * (float)pos, dn = t_min * mn[i];
                    term = up - dn;
                } else if (FMT == BAT_Q2W) {
                    const float pos = o.dw * (float)lo[i], neg = o.dmin * (float)hi[i];
                    term = dqs[i] * (pos - neg);
                } else {
                    const int isum = lo[i] + 256 * hi[i];
                    const float t = o.dw * dqs[i];
                    term = t * (float)isum;
                }
                /* lane (r, kq): row r, token 4 * kq + i of the chunk */
                s_term[(b * CH + (uint32_t)c) * 256u + (4u * kq + (uint32_t)i) * 16u + r16] = term;
            }
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");        /* the last request's, which nobody reads */
    __syncthreads();
    for (uint32_t i = tid; i < CH * 256u; i += blockDim.x) {
        const uint32_t tok = i >> 4, row = i & 15u;
        float acc = 0.0f;
#pragma unroll 8
        for (uint32_t b = 0; b < B; b++) acc += s_term[b * CH * 256u + i];
        if (tok < toks && row < rows_here) out[(size_t)tok * out_stride + row] = acc;
    }
}

template <int FMT, int CH>
__global__ __launch_bounds__(1024, 4) void
k_mmq_batch(const uint8_t *__restrict__ w, uint32_t rows, uint32_t B, const uint8_t *__restrict__ acts, uint32_t n_vec,
            float *__restrict__ out, size_t out_stride)
{
    const uint32_t row0 = blockIdx.x * 16u, tok0 = blockIdx.y * (CH * 16u);
    bat_tile<FMT, CH, false>(w + (size_t)row0 * B * BatGeom<FMT, CH>::WB, min(rows - row0, 16u), B,
                             acts + (size_t)tok0 * B * 292u, min(n_vec - tok0, CH * 16u),
                             out + (size_t)tok0 * out_stride + row0, out_stride);
}

/* The same over the experts of a mixture-of-experts layer that got tokens, whose numbers are known on the device only:
 * grid.x walks the 16-row groups of the launch's one or two matrices, grid.y the (expert, token tile) pairs, expert by
 * expert.  The grid has as many y as any routing can need; what is beyond the last leaves at once. */
struct BatExperts {
    const uint8_t *w[2];
    float *out[2];
    uint32_t rows, B, groups, n_expert;
    const uint8_t *acts;
    size_t out_stride;
    const uint32_t *counts, *offsets;
};

template <int FMT, int CH, bool TM>
__global__ __launch_bounds__(1024, 4) void
k_mmq_batch_experts(const BatExperts a)
{
    constexpr uint32_t TOK = CH * 16u;
    const uint32_t lane = threadIdx.x & 63u;
    /* a lane per expert: its tiles and, by ballots over the bits of their numbers, how many the experts before it have */
    const uint32_t cnt = lane < a.n_expert ? a.counts[lane] : 0u, off = lane < a.n_expert ? a.offsets[lane] : 0u;
    const uint32_t tiles = (cnt + TOK - 1u) / TOK;
    uint32_t from = 0u;
    for (uint32_t k = 0u; __ballot((tiles >> k) != 0u) != 0ull; k++) {
        const unsigned long long set = __ballot(((tiles >> k) & 1u) != 0u);
        from += __builtin_amdgcn_mbcnt_hi((uint32_t)(set >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)set, 0u)) << k;
    }
    const unsigned long long mine = __ballot(blockIdx.y >= from && blockIdx.y - from < tiles);
    if (mine == 0ull) return;
    const int e = __builtin_ctzll(mine);
    const uint32_t tok0 = (blockIdx.y - (uint32_t)__builtin_amdgcn_readlane((int)from, e)) * TOK;
    const uint32_t toks = min((uint32_t)__builtin_amdgcn_readlane((int)cnt, e) - tok0, TOK);
    const uint32_t first = (uint32_t)__builtin_amdgcn_readlane((int)off, e) + tok0;
    const uint32_t second = blockIdx.x >= a.groups ? 1u : 0u, row0 = (blockIdx.x - second * a.groups) * 16u;
    bat_tile<FMT, CH, TM>((second ? a.w[1] : a.w[0]) + ((size_t)e * a.rows + row0) * a.B * BatGeom<FMT, CH>::WB,
                          min(a.rows - row0, 16u), a.B, a.acts + (size_t)first * a.B * 292u, toks,
                          (second ? a.out[1] : a.out[0]) + (size_t)first * a.out_stride + row0, a.out_stride);
}

template <typename K> static hipError_t bat_whole_lds(K kernel)
{
    return hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                               160 * 1024);
}

extern "C" int oxh_internal_batch_init(void)
{
    hipError_t e;
    if ((e = bat_whole_lds(k_mmq_batch<BAT_Q4, 1>)) != hipSuccess) return (int)e;
    if ((e = bat_whole_lds(k_mmq_batch<BAT_Q4, 2>)) != hipSuccess) return (int)e;
    if ((e = bat_whole_lds(k_mmq_batch<BAT_Q5, 1>)) != hipSuccess) return (int)e;
    if ((e = bat_whole_lds(k_mmq_batch<BAT_Q5, 2>)) != hipSuccess) return (int)e;
    if ((e = bat_whole_lds(k_mmq_batch<BAT_Q6, 1>)) != hipSuccess) return (int)e;
    if ((e = bat_whole_lds(k_mmq_batch<BAT_Q6, 2>)) != hipSuccess) return (int)e;
    if ((e = bat_whole_lds(k_mmq_batch<BAT_Q2W, 1>)) != hipSuccess) return (int)e;
    if ((e = bat_whole_lds(k_mmq_batch_experts<BAT_Q4, 1, false>)) != hipSuccess) return (int)e;
    if ((e = bat_whole_lds(k_mmq_batch_experts<BAT_Q4, 1, true>)) != hipSuccess) return (int)e;
    if ((e = bat_whole_lds(k_mmq_batch_experts<BAT_Q5, 1, false>)) != hipSuccess) return (int)e;
    if ((e = bat_whole_lds(k_mmq_batch_experts<BAT_Q5, 1, true>)) != hipSuccess) return (int)e;
    if ((e = bat_whole_lds(k_mmq_batch_experts<BAT_Q6, 1, false>)) != hipSuccess) return (int)e;
    return (int)bat_whole_lds(k_mmq_batch<BAT_Q2W, 2>);
}

static uint32_t bat_need(int fmt, uint32_t ch, uint32_t B, uint32_t waves)
{
    switch (fmt) {
    case BAT_Q4: return ch == 1 ? bat_lds_bytes<BAT_Q4, 1>(B, waves) : bat_lds_bytes<BAT_Q4, 2>(B, waves);
    case BAT_Q5: return ch == 1 ? bat_lds_bytes<BAT_Q5, 1>(B, waves) : bat_lds_bytes<BAT_Q5, 2>(B, waves);
    default:     return ch == 1 ? bat_lds_bytes<BAT_Q6, 1>(B, waves) : bat_lds_bytes<BAT_Q6, 2>(B, waves);
    }
}

#define BAT_LDS (160u * 1024u)

/* The rule: against the tiles (oxh_mmq; oxh_mmq_split without a workspace), and where a workspace is at hand against
 * the split tiles as well.  Measured on 256 CUs over 29 row counts of 16 to 28672, 28 widths of 1 to 128 super-blocks
 * and 1 to 64 activations, all four formats, matmul launch alone, weights from several copies in turn; us, this
 * kernel / the other.  `grid` counts workgroups: 16-row groups times token tiles.
 *
 * Against the tiles:
 *   One super-block leaves the waves nothing to share: 4.8 / 4.0 at 17-64 activations, whatever the rows.
 *   Up to 16 activations this kernel wins up to two workgroups to a CU (Q4_K, 16 activations: 8192 x 4096 8.4 / 15.1,
 *   4096 x 14336 14.4 / 46.8), to three with five super-blocks or more (12288 x 1024, four: 6.7 / 6.1).  Above, the tiles have enough
 *   workgroups too and stage a token's values for four times the rows: Q4_K and widened Q2_K still win from 12 to
 *   28 super-blocks (14336 x 4096 12.6 / 15.1 at one activation; 14336 x 9216, 16 activations, 37.8 / 34.6) and beyond
 *   with at most eight activations (Q4_K 14336 x 14336 39.5 / 49.3 at five, but 94 / 85 at 95 super-blocks) or, Q2_K,
 *   from 56 on (69 / 72); Q5_K does not (42.9 / 36.0 at 36); Q6_K, whose tiles build operands longest, always does
 *   from eight on (five: 10.4 / 9.5).
 *   Above 16 activations a wave takes twice the LDS and time per weight: past a workgroup per CU not with fewer than
 *   12 super-blocks (Q6_K: eight; 5120 x 1024 7.6 / 6.5), and not beyond some fill of the device (14336 x 4096
 *   23.7 / 21.4).  LDS holds the terms of 36, 34, 38 super-blocks there (Q4_K, Q5_K, the others).
 * Against the split tiles, whose time grows with the terms they move (super-blocks x rows x activations), where this
 * kernel's grows with its rounds (super-blocks over the waves that LDS has room for) and jumps when the grid passes the
 * CUs: up to a number of super-blocks that is linear in the grid and in the part of its 16 (32) tokens a token tile has.
 *   Q4_K, 16 activations: 4096 x 14336 14.4 / 20.5; one: 16 x 9216 7.5 / 6.8, 1024 x 24320 18.9 / 14.2, 5120 x 24320
 *   47 / 29; 24: 512 x 8192 12.6 / 8.5, 5120 x 8704 24.9 / 19.1. */
struct SplitLine { double at0, slope, per_share, most; };

static bool beats_split(int fmt, size_t groups, size_t blocks, size_t n_vec, size_t cus)
{
    /* [up to 16 activations, more][Q4_K, Q5_K, 210-byte blocks][grid up to a workgroup per CU, larger] */
    static const SplitLine lines[2][3][2] = {
        { { { 31, 84, 91, 80 }, { -5, 31, 19, 80 } }, { { 23, 59, 23, 76 }, { -23, 45, 0, 64 } }, { { 20, 116, 11, 80 }, { 12, 17, 0, 80 } } },
        { { { 7, 35, 61, 40 }, { 18, 0, 0, 18 } }, { { -17, 91, 75, 40 }, { -27, 43, 5, 40 } }, { { -1, 107, 24, 40 }, { -20, 36, 9, 40 } } } };
    const int kind = fmt == BAT_Q4 ? 0 : fmt == BAT_Q5 ? 1 : 2;
    const size_t tok = n_vec <= 16 ? 16 : 32, tiles = (n_vec + tok - 1) / tok, grid = groups * tiles;
    if (grid <= cus && blocks <= 15) return true;           /* 200 x 3840, 17-64 activations: 7.2 / 8.3 */
    if (kind == 2 && tok == 16) {
        /* at ten waves at most, 32 super-blocks take four rounds as 40 do: 512 x 8192 11.1 / 10.0 */
        if (16 * grid < 5 * cus && blocks > 28) return false;
        if (grid <= cus ? 8 * grid >= 5 * cus : 16 * grid >= 25 * cus) return true;
    }
    const SplitLine &l = lines[tok == 16 ? 0 : 1][kind][grid > cus ? 1 : 0];
    const double share = (double)n_vec / (double)(tok * tiles);
    const double line = l.at0 + (l.slope + l.per_share * share) * (double)grid / (double)cus;
    return (double)blocks <= (line < l.most ? line : l.most);
}

extern "C" int oxh_internal_mmq_batch_takes(int fmt, size_t rows, size_t blocks, size_t n_vec, size_t cus, int split)
{
    const size_t groups = (rows + 15) / 16;
    if (n_vec > 64 || blocks < 2 || blocks > 128) return 0;
    const uint32_t ch = n_vec <= 16 ? 1 : 2;
    if (bat_need(fmt, ch, (uint32_t)blocks, 4) > BAT_LDS) return 0;
    if (split && !beats_split(fmt, groups, blocks, n_vec, cus)) return 0;
    const bool two_planes = fmt == BAT_Q6;
    if (n_vec <= 16) {
        if (groups <= 2 * cus) return 1;
        if (groups <= 3 * cus) return blocks >= 5;
        if (groups > 4 * cus || fmt == BAT_Q5) return 0;
        if (two_planes) return blocks >= 8;
        return blocks >= 12 && (blocks <= 28 || (fmt == BAT_Q4 ? n_vec <= 8 && blocks <= 80 : n_vec <= 8 || blocks >= 56));
    }
    const size_t grid = groups * ((n_vec + 31) / 32);
    if (grid > cus && blocks < (two_planes ? 8u : 12u)) return 0;
    if (n_vec <= 32) return groups <= (two_planes ? 2 * cus : cus + cus / 4);
    return grid <= (two_planes ? 2 * cus : cus);
}

/* Two workgroups of four waves to a CU where there are that many and LDS holds them: while one sums, the other
 * streams (8192 x 4096, 16 activations: 9.4 us against 11.0 with one of eight).  Otherwise as many waves as LDS
 * holds, as evenly used as the super-blocks allow. */
extern "C" uint32_t oxh_internal_mmq_batch_waves(int fmt, size_t rows, size_t blocks, size_t n_vec, size_t cus)
{
    const uint32_t B = (uint32_t)blocks, ch = n_vec <= 16 ? 1 : 2;
    const size_t groups = (rows + 15) / 16 * ((n_vec + 16 * ch - 1) / (16 * ch));
    uint32_t waves = 4;
    if (groups <= cus || 2u * bat_need(fmt, ch, B, 4) > BAT_LDS)
        while (waves < 16u && bat_need(fmt, ch, B, waves + 1u) <= BAT_LDS) waves++;
    const uint32_t rounds = (B + waves - 1u) / waves;
    return (B + rounds - 1u) / rounds;
}

/* see oxh_internal.h */
extern "C" int oxh_internal_mmq_batch(int fmt, const void *d_w, size_t rows, size_t blocks, const void *d_acts, size_t n_vec,
                                      float *d_out, size_t out_stride, void *stream)
{
    const uint32_t B = (uint32_t)blocks, ch = n_vec <= 16 ? 1 : 2;
    const size_t cus = (size_t)(oxh_internal_n_cu() > 0 ? oxh_internal_n_cu() : 256);
    const dim3 grid((uint32_t)((rows + 15) / 16), (uint32_t)((n_vec + 16 * ch - 1) / (16 * ch)));
    const uint32_t waves = oxh_internal_mmq_batch_waves(fmt, rows, blocks, n_vec, cus);
    const uint32_t lds = bat_need(fmt, ch, B, waves);
#define OXH_BATCH(FMT, CH)                                                                                           \
    hipLaunchKernelGGL((k_mmq_batch<FMT, CH>), grid, dim3(64u * waves), lds, (hipStream_t)stream, (const uint8_t *)d_w, \
                       (uint32_t)rows, B, (const uint8_t *)d_acts, (uint32_t)n_vec, d_out, out_stride)
#define OXH_BATCH_F(CH)                                \
    switch (fmt) {                                     \
    case BAT_Q4: OXH_BATCH(BAT_Q4, CH); break;         \
    case BAT_Q5: OXH_BATCH(BAT_Q5, CH); break;         \
    case BAT_Q6: OXH_BATCH(BAT_Q6, CH); break;         \
    default:     OXH_BATCH(BAT_Q2W, CH); break;        \
    }
    if (ch == 1) {
        OXH_BATCH_F(1)
    } else {
        OXH_BATCH_F(2)
    }
    return (int)hipGetLastError();
}

/* (expert, token tile) pairs any routing can need */
static size_t exp_slots(size_t n_expert, size_t pairs, size_t max_tokens)
{
    const size_t by_pairs = (pairs + n_expert * 15) / 16, each = (max_tokens + 15) / 16;
    const size_t live = pairs < n_expert ? pairs : n_expert;
    return live * each < by_pairs ? live * each : by_pairs;
}

/* Workgroups that find tokens when each token chooses its experts evenly: the experts some token chose, a token tile
 * each, or where they have more tokens than eight half a tile more than those fill. */
static double exp_workgroups(size_t n_mat, size_t n_expert, size_t rows, size_t pairs, size_t n_tok)
{
    const double missed = 1.0 - (double)pairs / (double)n_tok / (double)n_expert;
    const double hit = (double)n_expert * (1.0 - pow(missed > 0.0 ? missed : 0.0, (double)n_tok));
    const double filled = 0.5 * hit + (double)pairs / 16.0;
    return (double)(n_mat * ((rows + 15) / 16)) * (hit > filled ? hit : filled);
}

/* The rule, against the 64-row tiles of the experts (and the long ones, where those are taken).  From 1300 random layers
 * (4, 8 and 16 experts, top 1 to 3, 1024 x 768 to 4096 x 14336, 1 to 100 tokens; the layer's time with this kernel for one
 * of its launches / without): the fewer workgroups a CU gets the more is gained, and more than the tiles' way through
 * all of a row's super-blocks costs is lost once the device is full of tiles as well, since each of these workgroups
 * stages the tokens for 16 rows only.  Where LDS holds two workgroups the lines lie at four to a CU (Q4_K, Q5_K) and six
 * (Q6_K, whose tiles take longest), where it holds one at three and four and a half: one layer in a hundred within them is
 * slower, by 1 to 4 %.  us a layer, without / with: down of 16 experts 2560 x 6144, Q6_K, 3 tokens 69.6 / 44.3; of four
 * 1536 x 5120, Q4_K, 36 tokens 38.8 / 31.3; gate and up of 16 of 4096 x 3072, Q4_K, two tokens 50.2 / 40.3; beyond the
 * lines, down of 8 of 4096 x 14336, Q4_K, 16 tokens 162 / 190. */
extern "C" int oxh_internal_experts_batch_takes(int fmt, size_t n_mat, size_t n_expert, size_t rows, size_t blocks, size_t pairs,
                                                size_t n_tok, size_t cus)
{
    if (blocks < 2 || blocks > 128 || pairs == 0 || n_tok == 0 || n_expert > 64) return 0;
    const uint32_t need = bat_need(fmt, 1, (uint32_t)blocks, 4);
    if (need > BAT_LDS) return 0;
    const double per_cu = 2u * need > BAT_LDS ? 0.75 : 1.0;
    return exp_workgroups(n_mat, n_expert, rows, pairs, n_tok) <= per_cu * (fmt == BAT_Q6 ? 6.0 : 4.0) * (double)cus;
}

/* see oxh_internal.h */
extern "C" int oxh_internal_experts_batch(int fmt, int tile_major, const void *const *d_w, float *const *d_out, size_t n_mat,
                                          size_t n_expert, size_t rows, size_t blocks, const void *d_acts, size_t out_stride,
                                          const uint32_t *d_counts, const uint32_t *d_offsets, size_t pairs,
                                          size_t max_tokens, void *stream)
{
    const size_t cus = (size_t)(oxh_internal_n_cu() > 0 ? oxh_internal_n_cu() : 256);
    BatExperts a;
    for (int i = 0; i < 2; i++) {
        a.w[i] = (const uint8_t *)d_w[(size_t)i < n_mat ? i : 0];
        a.out[i] = d_out[(size_t)i < n_mat ? i : 0];
    }
    a.rows = (uint32_t)rows;
    a.B = (uint32_t)blocks;
    a.groups = (uint32_t)((rows + 15) / 16);
    a.n_expert = (uint32_t)n_expert;
    a.acts = (const uint8_t *)d_acts;
    a.out_stride = out_stride;
    a.counts = d_counts;
    a.offsets = d_offsets;
    const size_t slots = exp_slots(n_expert, pairs, max_tokens);
    const dim3 grid((uint32_t)(n_mat * a.groups), (uint32_t)slots);
    const uint32_t waves = oxh_internal_mmq_batch_waves(fmt, 16 * n_mat * a.groups * slots, blocks, 1, cus);
    const uint32_t lds = bat_need(fmt, 1, a.B, waves);
#define OXH_EXPB(FMT, TM) hipLaunchKernelGGL((k_mmq_batch_experts<FMT, 1, TM>), grid, dim3(64u * waves), lds, (hipStream_t)stream, a)
    if (fmt == BAT_Q6) OXH_EXPB(BAT_Q6, false);
    else if (fmt == BAT_Q5 && tile_major) OXH_EXPB(BAT_Q5, true);
    else if (fmt == BAT_Q5) OXH_EXPB(BAT_Q5, false);
    else if (tile_major) OXH_EXPB(BAT_Q4, true);
    else OXH_EXPB(BAT_Q4, false);
#undef OXH_EXPB
    return (int)hipGetLastError();
}
