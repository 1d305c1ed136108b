/* oxh_experts.hip — the expert launches of a mixture-of-experts layer whose
 * experts get more than a handful of tokens each (prompts, large decode batches).
 *
 * What the reference does: per expert, gate / up / down over that expert's
 * tokens only (oxidize-c/src/model/llama.c:6060-6150).  Here one launch covers
 * every expert's tokens; which expert has how many is known on the device only. */
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "oxhip.h"
#include "oxh_internal.h"
#include "oxh_device.inc"
#include "mmq_tiles.inc"

/* The MFMA tiles over (expert, token tile) pairs.  grid.x walks the row tiles of
 * the launch's one or two matrices, grid.y the token tiles of all experts one
 * after the other: tile y belongs to the expert in whose run of ceil(tokens / TOK)
 * tiles it falls.  The grid has as many y as any routing can need (the counts are
 * on the device); what is beyond the last tile leaves at once, and comes last.
 *
 * What bounds these launches is the vector issue port, so what matters is not to
 * compute tokens nobody has: an expert's 16-token chunks are dealt evenly to its
 * tiles, and a tile runs the loop unrolled for the number of chunks it got.  (A
 * loop of fixed-size 64-token tiles per workgroup did a quarter of its work on
 * empty chunks at 128 +- 10 tokens per expert, and a matrix with few rows had no
 * workgroups for the second and third tile of an expert.) */
enum { EXP_Q4 = 0, EXP_Q5 = 1, EXP_Q6 = 2 };

struct ExpertArgs {
    const uint8_t *w[2];
    float *out[2];
    uint32_t rows, B, row_tiles, n_expert, tile_major;
    const uint8_t *acts;
    size_t out_stride;
    const uint32_t *counts, *offsets;
};

template <int FMT, int TCMAX, int RC>
__global__ __launch_bounds__(512, TCMAX <= 4 && FMT == EXP_Q4 ? 4 : 2) void
k_mmq_experts_long(const ExpertArgs a)
{
    constexpr uint32_t WB = FMT == EXP_Q4 ? 144u : FMT == EXP_Q5 ? 176u : 210u;
    constexpr uint32_t ROWS = 8u * RC * 16u, TOK = TCMAX * 16u;
    const uint32_t lane = threadIdx.x & 63u;
    /* a lane per expert: its tiles and where they start, the expert tile y falls in.  Workgroups start in the order of
     * y, so experts whose tiles hold the most chunks come first: with the counts as they fall a launch of little more
     * than one round ended with a whole tile that started late (8 experts, 1024 pairs, 4096 rows, one expert above 144
     * tokens: 265 us, 219 in this order; no difference where all fit one round).  A tile holds at most TCMAX chunks, so
     * the order is a counting sort: size by size, from the largest, the tiles of that size's experts by ballots over the
     * bits of their numbers.  (Every expert compared with every other one, a layer of 64 took 2.5 to 6 % longer.) */
    const uint32_t cnt = lane < a.n_expert ? a.counts[lane] : 0u;
    const uint32_t off = lane < a.n_expert ? a.offsets[lane] : 0u;
    const uint32_t tiles = (cnt + TOK - 1u) / TOK;
    const uint32_t size = tiles ? (((cnt + 15u) >> 4) + tiles - 1u) / tiles : 0u;
    uint32_t bits = 0u, base = 0u, from = 0u;
    while (__ballot((tiles >> bits) != 0u) != 0ull) bits++;
    unsigned long long here_is = 0ull;
    for (uint32_t s = TCMAX; s != 0u; s--) {
        const bool in = size == s;
        uint32_t all = 0u, before = 0u;
        for (uint32_t k = 0; k < bits; k++) {
            const unsigned long long set = __ballot(in && ((tiles >> k) & 1u) != 0u);
            all += (uint32_t)__popcll(set) << k;
            before += __builtin_amdgcn_mbcnt_hi((uint32_t)(set >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)set, 0u)) << k;
        }
        if (blockIdx.y - base < all) {
            from = base + before;
            here_is = __ballot(in && blockIdx.y >= from && blockIdx.y - from < tiles);
            break;
        }
        base += all;
    }
    if (here_is == 0ull) return;
    const int e = __builtin_ctzll(here_is);
    const uint32_t nv = (uint32_t)__builtin_amdgcn_readlane((int)cnt, e);
    const uint32_t n_tiles = (uint32_t)__builtin_amdgcn_readlane((int)tiles, e);
    const uint32_t tile = blockIdx.y - (uint32_t)__builtin_amdgcn_readlane((int)from, e);
    const uint32_t chunks = (nv + 15u) >> 4;
    const uint32_t c0 = tile * chunks / n_tiles, nc = (tile + 1u) * chunks / n_tiles - c0;
    const uint32_t first = (uint32_t)__builtin_amdgcn_readlane((int)off, e) + 16u * c0;
    const uint32_t here = min(nv - 16u * c0, 16u * nc);

    const uint32_t second = blockIdx.x >= a.row_tiles ? 1u : 0u;
    const uint32_t row0 = (blockIdx.x - second * a.row_tiles) * ROWS;
    const uint8_t *w = (second ? a.w[1] : a.w[0]) + ((size_t)e * a.rows + row0) * a.B * WB;
    float *out = (second ? a.out[1] : a.out[0]) + (size_t)first * a.out_stride + row0;
    const uint8_t *acts = a.acts + (size_t)first * a.B * 292u;
#define OXH_CHUNKS(N)                                                                                              \
    do {                                                                                                           \
        if constexpr (FMT == EXP_Q6) mmq6_tile<N, RC, 8>(w, a.rows - row0, a.B, acts, here, out, a.out_stride);    \
        else mmq_tile<N, RC, 8, FMT == EXP_Q5>(w, a.rows - row0, a.B, acts, here, out, a.out_stride, 0u, 0u,       \
                                               a.tile_major);                                                      \
        return;                                                                                                    \
    } while (0)
    if constexpr (TCMAX == 4) {
        if (nc <= 2u) OXH_CHUNKS(2);
        if (nc == 3u) OXH_CHUNKS(3);
        OXH_CHUNKS(4);
    } else {
        if (nc <= 2u) OXH_CHUNKS(2);
        if (nc <= 4u) OXH_CHUNKS(4);
        if (nc == 5u) OXH_CHUNKS(5);
        if (nc == 6u) OXH_CHUNKS(6);
        if (nc == 7u) OXH_CHUNKS(7);
        if (nc == 8u) OXH_CHUNKS(8);
        OXH_CHUNKS(9);
    }
#undef OXH_CHUNKS
}

template <typename K> static hipError_t whole_lds(K kernel)
{
    return hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                               160 * 1024);
}

extern "C" int oxh_internal_experts_init(void)
{
    hipError_t e;
    if ((e = whole_lds(k_mmq_experts_long<EXP_Q4, 9, 2>)) != hipSuccess) return (int)e;
    if ((e = whole_lds(k_mmq_experts_long<EXP_Q4, 9, 1>)) != hipSuccess) return (int)e;
    if ((e = whole_lds(k_mmq_experts_long<EXP_Q4, 4, 1>)) != hipSuccess) return (int)e;
    if ((e = whole_lds(k_mmq_experts_long<EXP_Q5, 9, 1>)) != hipSuccess) return (int)e;
    if ((e = whole_lds(k_mmq_experts_long<EXP_Q5, 4, 1>)) != hipSuccess) return (int)e;
    if ((e = whole_lds(k_mmq_experts_long<EXP_Q6, 9, 1>)) != hipSuccess) return (int)e;
    if ((e = whole_lds(k_mmq_experts_long<EXP_Q6, 4, 1>)) != hipSuccess) return (int)e;
    return 0;
}

/* Which tile.  Up to 64 tokens per expert the 128 x 64 one, two to a CU, holds them all (Mixtral-shaped, Q4_K,
 * 50 tokens per expert: 303 us a layer against 335 on 128 x 144 tiles and 369 on 256 x 144); above, a tile
 * that holds 144 saves building an expert's operands again (8 x 128 tokens: 573 us against 655), of 256 rows
 * (Q4_K; one takes as long as 1.75 of the other kind: the layer of 4 x 250 tokens 518 us against 547) or of 128,
 * whichever takes fewer rounds of the CUs, as long as there is one for nearly every CU. */
static int long_shape(int fmt, size_t n_mat, size_t n_expert, size_t rows, size_t pairs, size_t cus)
{
    const size_t avg = pairs / n_expert, tok_tiles = n_expert * ((avg + 143) / 144);
    const size_t mid = n_mat * ((rows + 127) / 128) * tok_tiles, large = n_mat * ((rows + 255) / 256) * tok_tiles;
    if (avg <= 64 || mid < cus - cus / 8) return 3;
    return fmt == EXP_Q4 && 1.75 * (double)((large + cus - 1) / cus) <= (double)((mid + cus - 1) / cus) ? 1 : 2;
}

static int long_fmt(uint32_t file_type)
{
    return file_type == OXH_Q6_K ? EXP_Q6 : file_type == OXH_Q5_K_M || file_type == OXH_Q5_K_S ? EXP_Q5 : EXP_Q4;
}

/* see oxh_internal.h */
extern "C" void oxh_internal_experts_long_tile(uint32_t file_type, size_t n_mat, size_t n_expert, size_t rows, size_t pairs,
                                               size_t cus, uint32_t tile[2])
{
    const int shape = long_shape(long_fmt(file_type), n_mat, n_expert, rows, pairs, cus);
    tile[0] = shape == 1 ? 256u : 128u;
    tile[1] = shape == 3 ? 64u : 144u;
}

/* see oxh_internal.h */
extern "C" int oxh_internal_experts_long(uint32_t file_type, int tile_major, const void *const *d_w, float *const *d_out,
                                         size_t n_mat, size_t n_expert, size_t rows, size_t cols, const void *d_acts,
                                         size_t out_stride, const uint32_t *d_counts, const uint32_t *d_offsets,
                                         size_t pairs, size_t max_tokens, void *stream)
{
    const int fmt = long_fmt(file_type);
    const size_t cus = (size_t)(oxh_internal_n_cu() > 0 ? oxh_internal_n_cu() : 256);
    ExpertArgs a;
    for (int i = 0; i < 2; i++) {
        a.w[i] = (const uint8_t *)d_w[(size_t)i < n_mat ? i : 0];
        a.out[i] = d_out[(size_t)i < n_mat ? i : 0];
    }
    a.rows = (uint32_t)rows;
    a.B = (uint32_t)(cols / OXH_QK_K);
    a.n_expert = (uint32_t)n_expert;
    a.tile_major = tile_major ? 1u : 0u;
    a.acts = (const uint8_t *)d_acts;
    a.out_stride = out_stride;
    a.counts = d_counts;
    a.offsets = d_offsets;
    /* token tiles any routing can need */
    auto most = [&](size_t tok) {
        const size_t by_pairs = (pairs + n_expert * (tok - 1)) / tok, by_tokens = n_expert * ((max_tokens + tok - 1) / tok);
        return by_pairs < by_tokens ? by_pairs : by_tokens;
    };
    const int shape = long_shape(fmt, n_mat, n_expert, rows, pairs, cus);
#define OXH_LONG(FMT, TC, RC, GEOM)                                                                            \
    do {                                                                                                       \
        a.row_tiles = (uint32_t)((rows + GEOM::ROWS - 1) / GEOM::ROWS);                                        \
        hipLaunchKernelGGL((k_mmq_experts_long<FMT, TC, RC>), dim3((uint32_t)(n_mat * a.row_tiles), (uint32_t)most(TC * 16)), \
                           dim3(512), GEOM::LDS_BYTES, (hipStream_t)stream, a);                                \
    } while (0)
    typedef MmqGeom<9, 2, 8> G4l;
    typedef MmqGeom<9, 1, 8> G4m;
    typedef MmqGeom<4, 1, 8> G4s;
    typedef MmqGeom<9, 1, 8, true> G5m;
    typedef MmqGeom<4, 1, 8, true> G5s;
    typedef Mmq6Geom<9, 1, 8> G6m;
    typedef Mmq6Geom<4, 1, 8> G6s;
    if (fmt == EXP_Q4) {
        if (shape == 1) OXH_LONG(EXP_Q4, 9, 2, G4l);
        else if (shape == 2) OXH_LONG(EXP_Q4, 9, 1, G4m);
        else OXH_LONG(EXP_Q4, 4, 1, G4s);
    } else if (fmt == EXP_Q5) {
        if (shape == 2) OXH_LONG(EXP_Q5, 9, 1, G5m);
        else OXH_LONG(EXP_Q5, 4, 1, G5s);
    } else {
        if (shape == 2) OXH_LONG(EXP_Q6, 9, 1, G6m);
        else OXH_LONG(EXP_Q6, 4, 1, G6s);
    }
#undef OXH_LONG
    return (int)hipGetLastError();
}
