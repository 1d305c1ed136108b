/* oxhip_lab.h — test hooks and measurement aids of liboxhip.
 *
 * None of these has a counterpart in the reference and none belongs to the
 * drop-in surface: the shared library exports exactly the functions that
 * include/oxhip.h declares plus the one accessor below, and everything here is
 * reached through the table it returns.  The parity tests use the hooks to
 * read intermediates (sub-block sums, the expert layer's workspace), the
 * benchmark uses the probes to measure what the device itself can do.
 */
#ifndef OXHIP_LAB_H
#define OXHIP_LAB_H

#include "oxhip.h"

#ifdef __cplusplus
extern "C" {
#endif

typedef struct OxhLab {
    /* With d_stamps set (n_ops * workgroups * 8 uint64 of device memory, or
     * NULL to switch it off) wave 0 of every workgroup of a plan launch stores
     * the shader clock at eight points of every operation: start, dependency
     * met, activation staged, workgroup barrier passed, passes done, rows
     * summed, barrier passed, outputs stored and announced. */
    int (*plan_stamps)(OxhPlan *plan, uint64_t *d_stamps);
    /* With `on` set the waits of a plan also expect a workgroup that does not
     * exist, so every wait runs into the poll limit: the way to test the
     * give-up path from the host without hanging anything. */
    int (*plan_phantom)(OxhPlan *plan, int on);
    /* Byte offsets inside oxh_moe_ffn's workspace of, in this order, ids,
     * weights, slot_pos, perm, counts, offsets, the gathered Q8_K activations,
     * gate, up (f32 [pair][ffn]), the Q8_K form of silu(gate)*up, the down
     * outputs (f32 [pair][hidden]), and the total size.  After a call the
     * parity tests read every intermediate from there. */
    int (*moe_workspace_parts)(const OxhMoe *m, size_t n_tok, size_t parts[12]);
    /* One launch that only reads `bytes` of device memory (a workgroup per CU,
     * 16-byte loads, nothing computed); d_sink may be NULL.  Timed on a buffer
     * the size of a weight matrix it gives the ceiling any kernel streaming
     * that matrix once can reach on the device, launch cost included. */
    int (*read_probe)(const void *d_buf, size_t bytes, uint32_t *d_sink, void *stream);
    /* The int8 matrix-core rate of the whole device (POP/s) when every
     * v_mfma_i32_16x16x64_i8 is followed by `valu_per_mfma` (0, 1, 2 or 4)
     * independent f32 vector instructions, with 1..4 waves per SIMD.
     * Synchronous (two launches, the second timed with events). */
    int (*mfma_probe)(int valu_per_mfma, int waves_per_simd, double *pops);
    /* The integer sub-block sums the GEMV kernel forms, written by the same
     * device code path.  Q4_K and Q5_K: 8 int32 per super-block (S_j), Q6_K: 16
     * per super-block, Q8_0: 1 per block; layout [row][block][j].  The values
     * are the intermediates of oxidize-c/src/compute/oxk.c:263-283, :870-886,
     * :932-954, :234-237, which the reference's API does not expose. */
    int (*subblock_sums)(uint32_t qtype, const void *d_w, size_t rows, size_t cols, const void *d_act,
                         int32_t *d_sums, void *stream);
    /* Which kernel a matrix-core launch of these sizes runs on, on a device of
     * n_cu compute units and with ws_bytes of workspace (oxh_mmq_split; 0 is
     * oxh_mmq): what the launch itself asks, as host arithmetic.  out: the
     * kernel (0 tiles, 1 Q6_K tiles whose operands a workgroup builds once,
     * 2 a workgroup per 16 rows whose waves share the columns, 3 tiles whose
     * columns several workgroups share), rows and tokens of a workgroup (for
     * kernel 1 the tokens it has room for), and for kernel 2 its waves, for
     * kernel 1 the token tiles the launch is cut into.  OXH_DECLINED for a
     * type without such a kernel. */
    int (*mmq_kernel)(uint32_t qtype, size_t rows, size_t cols, size_t n_vec, size_t n_cu, size_t ws_bytes,
                      uint32_t out[4]);
    /* The same for one expert launch of oxh_moe_ffn: n_mat matrices of `rows`
     * rows per expert (gate and up 2, down 1) under `pairs` (token, expert)
     * pairs in all; tile: rows and tokens of a workgroup, where the launch is
     * one of tiles (see experts_batch). */
    int (*experts_tile)(uint32_t qtype, size_t n_mat, size_t n_expert, size_t rows, size_t pairs, size_t n_cu,
                        uint32_t tile[2]);
    /* Chunks that host batches have moved through the library's own
     * page-locked slots so far, both ways together. */
    size_t (*host_ring_chunks)(void);
    /* Whether an expert launch of oxh_moe_ffn over rows x cols matrices gives
     * every workgroup 16 rows and all their columns (1) or runs on the tile
     * that experts_tile names (0); n_mat as there. */
    int (*experts_batch)(uint32_t qtype, size_t n_mat, size_t n_expert, size_t rows, size_t cols, size_t top_k,
                         size_t n_tok, size_t n_cu);
    /* Whether the operations of a chained plan hand their results over by
     * value (1) or wait for whole operations (0). */
    int (*plan_by_value)(const OxhPlan *plan);
    /* Prompts of the 32-value formats: the byte, counted from the start of
     * its wave's first row, at which the thread that stages block `blk` (0..7)
     * of row `row` (0..7) of the wave fetches step `step` of rows of `blocks`
     * blocks, with the kernel's own 32-bit arithmetic.  The thread's block is
     * number 8 * step + blk; past the row's end it is the one eight before,
     * in rows of fewer than eight the last. */
    uint64_t (*mmq32_fetched)(uint32_t block_bytes, uint32_t blocks, uint32_t row, uint32_t blk, uint32_t step);
    /* What oxh_plan_create would make of these operations on a device of n_cu
     * compute units, without one: host arithmetic on the addresses given, which
     * are not read.  out, 3 + 16 * n_ops words: whether results are handed over
     * by value, the workgroups, the bytes of a set of slots; per operation by
     * value: which inputs come out of slots (1 x, 2 the addend, 4 the prologue's
     * other input), the workgroups that have rows, the first one of each of four
     * segments, and, as offsets into a set of slots plus 4, or 0: x, the
     * prologue's other input, the addend, the prologue's output, its sum, the
     * segments' results; bit 0: the other set, bit 1: the sets change places
     * from launch to launch.  (Inputs that come out of no slot: their address.)
     * Else: 0, or 1 + the operation that has to be complete, and the first
     * five of the rest. */
    int (*plan_draft)(const OxhPlanOp *ops, size_t n_ops, uint32_t n_cu, uint64_t *out);
} OxhLab;

const OxhLab *oxh_lab(void);

#ifdef __cplusplus
}
#endif
#endif
