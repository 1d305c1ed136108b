/* oxh_mmq6.hip — the prefill matmul of Q6_K (and widened Q2_K) weights in tiles
 * whose weight operands are built once per workgroup.
 *
 * Arithmetic, operand roles and the activations' LDS image are those of
 * mmq6_tile() (mmq_tiles.inc; oxidize-c/src/compute/oxk.c:913-964): a 210-byte
 * block becomes two int8 operand planes, (code - 32) * scale = 256 * hi + lo, and
 * the f32 step is the reference's per super-block.
 *
 * Why another tile.  A wave of mmq6_tile() builds the planes of its own 16 rows,
 * some 200 vector instructions per super-block, against 20 per 16 x 16 chunk of
 * results: with 128 tokens to a tile that is as much as the results themselves,
 * with 32 four times as much, and a matrix of 4096 rows under a few hundred
 * tokens has only enough tiles of the small kinds to fill the device.  Here a
 * workgroup covers 64 rows x 128 tokens with eight waves, four row chunks x two
 * token halves; all 512 threads build the next super-block's planes, each
 * thread an eighth of one row's block straight from its global loads (no trip of
 * the raw block through LDS), and both waves of a row chunk read them back as
 * MFMA operands.  Per wave that is half the build of a 64 x 128 tile on four waves at
 * twice the waves per SIMD.  The build of super-block b + 1 is spread between
 * the chunks of super-block b, where the matrix cores cover it; one barrier per
 * super-block. */
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "oxhip.h"
#include "oxh_internal.h"
#include "oxh_device.inc"
#include "mmq_tiles.inc"

struct Q6sGeom {
    static constexpr uint32_t ROWS = 64u, TOK = 128u;
    /* one stage: token values [token][slot] x 16 B, token scales, the two planes [row][slot] x 16 B with the
     * activations' slot swizzle, d (and dmin) per row */
    static constexpr uint32_t D_OFF = TOK * 256u;
    static constexpr uint32_t LO_OFF = D_OFF + TOK * 4u;
    static constexpr uint32_t HI_OFF = LO_OFF + ROWS * 256u;
    static constexpr uint32_t DW_OFF = HI_OFF + ROWS * 256u;
    static constexpr uint32_t STAGE_BYTES = DW_OFF + ROWS * 8u;
    static constexpr uint32_t LDS_BYTES = 2u * STAGE_BYTES;
};

/* an eighth of a block: 16 bytes of ql (two groups' low bits), the 16 bytes of qh that belong to them, the eight bytes
 * their two scales are in (Q2: all sixteen minima), and the dwords d (upper half) and, Q2, dmin (lower half) are in:
 * dwords and more, because a byte or half word would be widened by an instruction that waits for its load */
typedef uint32_t u32x4_2 __attribute__((ext_vector_type(4), aligned(2)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x2_2 __attribute__((ext_vector_type(2), aligned(2)));
struct Q6sRaw {
    u32x4 ql, qh;
    u32x2 sc;
    uint32_t d, dmin;
};

/* dword k of the planes of the group in the low (HIGH: high) nibbles */
template <bool Q2, bool HIGH>
__device__ __forceinline__ void q6s_dword(uint32_t ql, uint32_t qh, uint32_t sc, uint32_t rot, uint32_t &lo, uint32_t &hi)
{
    const uint32_t c = ((HIGH ? ql >> 4 : ql) & 0x0F0F0F0Fu) | (__builtin_amdgcn_alignbit(qh, qh, rot) & 0x30303030u);
    if (Q2) {
        lo = c;
        hi = sc;                    /* the group's minimum in every byte, set up by the caller */
        return;
    }
    const short scs = (short)sc, m32 = (short)(128 - 32 * (int)(short)sc);
    const v2i16 sc2 = { scs, scs }, off2 = { m32, m32 };
    const v2i16 ce = __builtin_bit_cast(v2i16, __builtin_amdgcn_perm(c, c, 0x0C020C00u));
    const v2i16 co = __builtin_bit_cast(v2i16, __builtin_amdgcn_perm(c, c, 0x0C030C01u));
    const uint32_t ue = __builtin_bit_cast(uint32_t, (v2i16)(ce * sc2 + off2));
    const uint32_t uo = __builtin_bit_cast(uint32_t, (v2i16)(co * sc2 + off2));
    lo = __builtin_amdgcn_perm(uo, ue, 0x06020400u) ^ 0x80808080u;
    hi = __builtin_amdgcn_perm(uo, ue, 0x07030501u);
}

/* The workgroup's barrier where its waves stand in different instantiations of q6s_walk().  __syncthreads() asks
 * every thread to reach the same call; s_barrier, which it becomes, is defined per wave: a wave waits until every
 * wave of its workgroup has executed one, wherever it stands in the program.  So the instruction itself, between
 * the fences __syncthreads() puts around it: LDS written before is seen after. */
__device__ __forceinline__ void q6s_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

/* A wave's N chunks of 16 tokens, the first of them chunk c_first of the tile, over all super-blocks; results
 * of tokens below toks_end are its to store.  The waves of a workgroup may run it for different N: each executes
 * 1 + B barriers, whatever N is. */
template <int N, bool Q2>
__device__ __forceinline__ void
q6s_walk(const uint8_t *__restrict__ w_base, uint32_t rows_here, uint32_t B, const uint8_t *__restrict__ a_base,
         uint32_t toks_here, float *__restrict__ out_base, size_t out_stride, uint32_t c_first, uint32_t toks_end)
{
    typedef Q6sGeom G;
    extern __shared__ __attribute__((aligned(16))) uint8_t mmq_lds[];
    const uint32_t lds_base = (uint32_t)(size_t)(__attribute__((address_space(3))) uint8_t *)mmq_lds;
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t r16 = lane & 15u, kq = lane >> 4;
    const uint32_t act_stride = B * 292u;

    /* activations: 64-lane load wave + 8 * i covers tokens 4 * (wave + 8 * i) .. +3, as in mmq6_tile() */
    uint32_t q_off[4];
#pragma unroll
    for (uint32_t i = 0; i < 4u; i++) {
        const uint32_t t = 4u * (wave + 8u * i) + (lane >> 4);
        q_off[i] = min(t, toks_here - 1u) * act_stride + 4u + 16u * ((lane & 15u) ^ (t & 15u));
    }
    /* this thread's eighth u = 4n + 2h + lh of row tid / 8: ql piece u, qh piece 2n + lh, groups 8n + 2h + lh
     * (low nibbles) and four further on (high nibbles) */
    const uint32_t b_row = tid >> 3, u = tid & 7u;
    const uint32_t grp = 8u * (u >> 2) + (u & 3u);
    const uint32_t w_off = min(b_row, rows_here - 1u) * (B * 210u);
    const uint32_t ql_off = w_off + 16u * u, qh_off = w_off + 128u + 32u * (u >> 2) + 16u * (u & 1u);
    const uint32_t sc_off = w_off + 192u + (Q2 ? 0u : 8u * (u >> 2));
    /* where in those eight bytes: group grp and the one four on (Q2: nibbles) */
    const uint32_t sc_bit = Q2 ? 4u * (grp & 7u) : 8u * (u & 3u);
    const uint32_t rot0 = ((u & 2u) - 4u) & 31u, rot1 = u & 2u;      /* bits 2h, 2h + 1 (2h + 4, 2h + 5) to 4, 5 */
    /* group 8n + 4h + j of a row goes to slot (8h + 4n + j) ^ row: a row's eight threads then write eight different
     * slots of 128 bytes */
    const uint32_t pl_wr = G::LO_OFF + b_row * 256u + (((4u * (u >> 2) + (u & 3u)) ^ (b_row & 15u)) * 16u);  /* ^ 128: four groups on */
    const uint32_t a_d_off = min(tid & (G::TOK - 1u), toks_here - 1u) * act_stride;

    auto request = [&](uint32_t blk, uint32_t buf) {
#pragma unroll
        for (uint32_t i = 0; i < 4u; i++)
            mmq_dma16(a_base + (size_t)blk * 292u, q_off[i], lds_base + buf * G::STAGE_BYTES + (wave + 8u * i) * 1024u);
    };
    auto load_raw = [&](uint32_t blk) -> Q6sRaw {
        const uint8_t *wb = w_base + (size_t)blk * 210u;
        Q6sRaw r;
        r.ql = *reinterpret_cast<const u32x4_2 *>(wb + ql_off);
        r.qh = *reinterpret_cast<const u32x4_2 *>(wb + qh_off);
        r.sc = *reinterpret_cast<const u32x2_2 *>(wb + sc_off);
        r.d = reinterpret_cast<const U32u2 *>(wb + w_off + 206u)->v;
        r.dmin = Q2 ? reinterpret_cast<const U32u2 *>(wb + w_off + 200u)->v : 0u;
        return r;
    };
    auto load_dq = [&](uint32_t blk) -> uint32_t {
        return *reinterpret_cast<const uint32_t *>(a_base + (size_t)blk * 292u + a_d_off);
    };
    /* the two groups' scales (Q2: minima, spread over four bytes) as the dword builder takes them.  Q2: groups 8n + j and
     * 8n + j + 4 are nibbles j and j + 4 of dword n */
    auto scale_of = [&](const Q6sRaw &r, int second) -> uint32_t {
        if (Q2) return (((u & 4u ? r.sc[1] : r.sc[0]) >> ((sc_bit + 16u * (uint32_t)second) & 31u)) & 15u) * 0x01010101u;
        return (uint32_t)__builtin_amdgcn_sbfe((int)r.sc[second], sc_bit, 8u);
    };
    u32x4 p_lo[2], p_hi[2];
    auto build_dword = [&](const Q6sRaw &r, int k) {
        uint32_t lo, hi;
        q6s_dword<Q2, false>(r.ql[k], r.qh[k], scale_of(r, 0), rot0, lo, hi);
        p_lo[0][k] = lo;
        p_hi[0][k] = hi;
        q6s_dword<Q2, true>(r.ql[k], r.qh[k], scale_of(r, 1), rot1, lo, hi);
        p_lo[1][k] = lo;
        p_hi[1][k] = hi;
    };
    auto store_planes = [&](float d, float dmin, uint32_t dq, uint32_t buf) {
        uint8_t *st = mmq_lds + buf * G::STAGE_BYTES;
        *reinterpret_cast<u32x4 *>(st + pl_wr) = p_lo[0];
        *reinterpret_cast<u32x4 *>(st + (pl_wr ^ 128u)) = p_lo[1];
        *reinterpret_cast<u32x4 *>(st + pl_wr + (G::HI_OFF - G::LO_OFF)) = p_hi[0];
        *reinterpret_cast<u32x4 *>(st + (pl_wr ^ 128u) + (G::HI_OFF - G::LO_OFF)) = p_hi[1];
        /* the eight threads of a row, and the four of a token, store the same values: no branch in the loop */
        float *dw = reinterpret_cast<float *>(st + G::DW_OFF) + 2u * b_row;
        dw[0] = d;
        if (Q2) dw[1] = dmin;
        *reinterpret_cast<uint32_t *>(st + G::D_OFF + 4u * (tid & (G::TOK - 1u))) = dq;
    };

    v4f acc[N];
#pragma unroll
    for (int c = 0; c < N; c++) acc[c] = (v4f){ 0.0f, 0.0f, 0.0f, 0.0f };

    const uint32_t a_rd = r16 * 256u + ((kq ^ r16) * 16u);                          /* ^ 64 * gp */
    const uint32_t p_rd = G::LO_OFF + (wave & 3u) * 4096u + a_rd;
    const uint32_t dw_rd = G::DW_OFF + ((wave & 3u) * 16u + r16) * 8u;
    const uint32_t dq_rd = G::D_OFF + 16u * kq + 64u * c_first;

    constexpr int RAW_LOADS = Q2 ? 5 : 4;           /* vector loads of one load_raw() */
    /* Two sets of raw blocks: while super-block b is computed one holds b + 1, complete, and is sent for b + 3 once its
     * planes are built; the other holds b + 2, still on its way. */
    Q6sRaw set0, set1;
    {
        request(0, 0);
        __builtin_amdgcn_sched_barrier(0);
        const Q6sRaw r = load_raw(0);
        const uint32_t dq = load_dq(0);
#pragma unroll
        for (int k = 0; k < 4; k++) build_dword(r, k);
        store_planes(half_to_float_hw(r.d >> 16), half_to_float_hw(r.dmin & 0xFFFFu), dq, 0);
        __builtin_amdgcn_sched_barrier(0);
        /* the LDS-bound loads, which the compiler does not count.  All that is on its way here, and next to nothing to
         * wait for behind the loads above, which are younger; a count that leaves set0 and set1 out would hold only as
         * long as the compiler requests both in front of it (it requests set1 behind the barrier) */
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        set0 = load_raw(min(1u, B - 1u));
        __builtin_amdgcn_sched_barrier(0);
        set1 = load_raw(min(2u, B - 1u));
        __builtin_amdgcn_sched_barrier(0);
        q6s_barrier();
    }

    auto step = [&](uint32_t b, Q6sRaw &next) {
        const uint32_t buf = b & 1u;
        const uint8_t *st = mmq_lds + buf * G::STAGE_BYTES;
        /* `next` is complete since the last barrier's wait; said here, before this step's LDS-bound loads are issued,
         * because the compiler would count those out of its own wait for it and so wait for them too */
        asm volatile("" : "+v"(next.ql), "+v"(next.qh), "+v"(next.sc), "+v"(next.d), "+v"(next.dmin));
        __builtin_amdgcn_sched_barrier(0);
        request(min(b + 1u, B - 1u), buf ^ 1u);
        const uint32_t dq_next = load_dq(min(b + 1u, B - 1u));
        __builtin_amdgcn_sched_barrier(0);
        v4i dl[4], dh[4];
        auto slot_of = [](int gp) -> uint32_t { return 2u * ((uint32_t)gp & 1u) + ((uint32_t)gp >> 1); };
#pragma unroll
        for (int gp = 0; gp < 4; gp++) {
            dl[gp] = *reinterpret_cast<const v4i *>(st + (p_rd ^ (64u * slot_of(gp))));
            dh[gp] = *reinterpret_cast<const v4i *>(st + (p_rd ^ (64u * slot_of(gp))) + (G::HI_OFF - G::LO_OFF));
        }
        const float2 dwm = *reinterpret_cast<const float2 *>(st + dw_rd);
        /* Chunk by chunk: the operands of chunk c + 1 are on their way, and the f32 step of chunk c - 1 and a share
         * of the next super-block's planes go between the MFMAs of chunk c.  The order is pinned. */
        float d_next = 0.0f, dmin_next = 0.0f;
        v4i an[4], lo_p = { 0, 0, 0, 0 }, hi_p = { 0, 0, 0, 0 };
        float4 dq_p = { 0.0f, 0.0f, 0.0f, 0.0f };
        auto read_a = [&](int c) {
#pragma unroll
            for (int gp = 0; gp < 4; gp++)
                an[gp] = *reinterpret_cast<const v4i *>(st + (a_rd ^ (64u * (uint32_t)gp)) + 4096u * (c_first + (uint32_t)c));
        };
        read_a(0);
#pragma unroll
        for (int c = 0; c <= N; c++) {
            v4i lo = { 0, 0, 0, 0 }, hi = { 0, 0, 0, 0 };
            float4 dq4 = { 0.0f, 0.0f, 0.0f, 0.0f };
            if (c < N) {
                const v4i a[4] = { an[0], an[1], an[2], an[3] };
                if (c + 1 < N) read_a(c + 1);
                dq4 = *reinterpret_cast<const float4 *>(st + dq_rd + 64u * (uint32_t)c);
#pragma unroll
                for (int gp = 0; gp < 4; gp++) {
                    lo = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[gp], dl[gp], lo, 0, 0, 0);
                    hi = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[gp], dh[gp], hi, 0, 0, 0);
                }
#pragma unroll
                for (int k = 0; k < 4; k++)
                    if (k * N / 4 == c) build_dword(next, k);
            }
            if (c > 0) {
                const float dqs[4] = { dq_p.x, dq_p.y, dq_p.z, dq_p.w };
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    if (Q2) {
                        const float pos = dwm.x * (float)lo_p[i], neg = dwm.y * (float)hi_p[i];
                        acc[c - 1][i] += dqs[i] * (pos - neg);
                    } else {
                        const int isum = lo_p[i] + 256 * hi_p[i];
                        const float t = dwm.x * dqs[i];
                        acc[c - 1][i] += t * (float)isum;
                    }
                }
            }
            lo_p = lo;
            hi_p = hi;
            dq_p = dq4;
            if (c < N) {
#pragma unroll
                for (int g = 0; g < 8; g++) {
                    __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);        /* an MFMA */
                    __builtin_amdgcn_sched_group_barrier(0x2, 4, 0);        /* vector instructions */
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            if (c == N - 1) {
                d_next = half_to_float_hw(next.d >> 16);
                dmin_next = Q2 ? half_to_float_hw(next.dmin & 0xFFFFu) : 0.0f;
                asm volatile("" : "+v"(d_next), "+v"(dmin_next));      /* out of `next` before it is loaded again */
                __builtin_amdgcn_sched_barrier(0);
                next = load_raw(min(b + 3u, B - 1u));
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        store_planes(d_next, dmin_next, dq_next, buf ^ 1u);
        /* loads return in order: this step's LDS-bound ones and the other set are complete when no more than the
         * raw blocks requested last are missing.  (dq_next, just stored, is younger than the LDS-bound ones: they are
         * complete wherever the compiler puts the raw blocks.) */
        asm volatile("s_waitcnt vmcnt(%0)" :: "n"(RAW_LOADS) : "memory");
        q6s_barrier();
    };
    uint32_t b = 0;
    for (; b + 1u < B; b += 2u) {
        step(b, set0);
        step(b + 1u, set1);
    }
    if (b < B) step(b, set0);
    /* the last requests, which nobody reads: the workgroup's LDS must be its own until they have landed */
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

    const uint32_t row = (wave & 3u) * 16u + r16;
    if (row < rows_here) {
#pragma unroll
        for (int c = 0; c < N; c++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const uint32_t tok = 16u * (c_first + (uint32_t)c) + 4u * kq + (uint32_t)i;
                if (tok < toks_end) out_base[(size_t)tok * out_stride + row] = acc[c][i];
            }
    }
}

/* grid (row tiles, token tiles); the token chunks are dealt evenly to the token tiles, at least one to each, and a
 * tile's to its two halves: both waves of a SIMD belong to one tile, so what counts is the chunks of the two together. */
template <bool Q2>
__global__ __launch_bounds__(512, 2) void
k_mmq_q6_k_shared(const uint8_t *__restrict__ w, uint32_t rows, uint32_t B, const uint8_t *__restrict__ acts,
                  uint32_t n_vec, float *__restrict__ out, size_t out_stride)
{
    const uint32_t row0 = blockIdx.x * Q6sGeom::ROWS;
    const uint32_t chunks = (n_vec + 15u) >> 4;
    /* the first `over` tiles get a chunk more; no product here passes the number of chunks (y * chunks would
     * leave 32 bits at three million activations) */
    const uint32_t each = chunks / gridDim.y, over = chunks - each * gridDim.y;
    const uint32_t c0 = blockIdx.y * each + min(blockIdx.y, over), nc = each + (blockIdx.y < over ? 1u : 0u);
    if (nc == 0u) return;           /* not launched: oxh_internal_mmq6_tok_tiles() is at most the number of chunks */
    const uint32_t tok0 = 16u * c0, here = min(n_vec - tok0, 16u * nc);
    const uint8_t *wb = w + (size_t)row0 * B * 210u, *ab = acts + (size_t)tok0 * B * 292u;
    float *ob = out + (size_t)tok0 * out_stride + row0;
    const uint32_t first_half = (nc + 1u) >> 1;
    const bool upper = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8) != 0u;
    const uint32_t mine = upper ? nc - first_half : first_half, at = upper ? first_half : 0u;
    const uint32_t end = upper ? here : min(here, 16u * first_half);
    if (mine == 4u) q6s_walk<4, Q2>(wb, rows - row0, B, ab, here, ob, out_stride, at, end);
    else if (mine == 3u) q6s_walk<3, Q2>(wb, rows - row0, B, ab, here, ob, out_stride, at, end);
    else if (mine == 2u) q6s_walk<2, Q2>(wb, rows - row0, B, ab, here, ob, out_stride, at, end);
    else q6s_walk<1, Q2>(wb, rows - row0, B, ab, here, ob, out_stride, at, end);
}

extern "C" int oxh_internal_mmq6_init(void)
{
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(k_mmq_q6_k_shared<false>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    if (e == hipSuccess)
        e = hipFuncSetAttribute(reinterpret_cast<const void *>(k_mmq_q6_k_shared<true>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    return (int)e;
}

/* see oxh_internal.h.  At least one tile per eight chunks (what a workgroup has LDS for).  While one round holds the
 * launch, as many more as CUs are left, down to two chunks a tile: a super-block costs a workgroup about a microsecond
 * whatever its tokens, and 0.05 of that per chunk on top (4096 x 14336, us by number of tiles: 128 activations
 * 78 / 62 / 59 on 1 / 2 / 3, 80 66 / 59 / 57, 333 72.2 / 70.7 on 3 / 4).  A second round costs more than it shortens the
 * first (14336 x 4096 under 160: 43 us on 2 tiles, 58 on 3). */
extern "C" size_t oxh_internal_mmq6_tok_tiles(size_t rows, size_t n_vec, size_t cus)
{
    const size_t row_tiles = (rows + Q6sGeom::ROWS - 1) / Q6sGeom::ROWS, chunks = (n_vec + 15) / 16;
    const size_t least = (n_vec + Q6sGeom::TOK - 1) / Q6sGeom::TOK, most = (chunks + 1) / 2, room = cus / row_tiles;
    const size_t more = room < most ? room : most;
    return more > least ? more : least;
}

/* see oxh_internal.h */
extern "C" int oxh_internal_mmq6_shared(int widened_q2, const void *d_w, size_t rows, size_t blocks, const void *d_acts,
                                        size_t n_vec, float *d_out, size_t out_stride, size_t cus, void *stream)
{
    typedef Q6sGeom G;
    const dim3 grid((uint32_t)((rows + G::ROWS - 1) / G::ROWS), (uint32_t)oxh_internal_mmq6_tok_tiles(rows, n_vec, cus));
    auto kernel = widened_q2 ? k_mmq_q6_k_shared<true> : k_mmq_q6_k_shared<false>;
    hipLaunchKernelGGL(kernel, grid, dim3(512), G::LDS_BYTES, (hipStream_t)stream, (const uint8_t *)d_w, (uint32_t)rows,
                       (uint32_t)blocks, (const uint8_t *)d_acts, (uint32_t)n_vec, d_out, out_stride);
    return (int)hipGetLastError();
}
