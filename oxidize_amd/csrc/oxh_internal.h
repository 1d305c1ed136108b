/* oxh_internal.h — symbols shared between the HIP translation unit and the C
 * host layer of liboxhip; not part of the public ABI: the library's export list is
 * made from the public headers, so nothing declared here is visible outside it. */
#ifndef OXH_INTERNAL_H
#define OXH_INTERNAL_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* printf-style with exactly two %s slots (either may be NULL). */
void oxh_set_error(const char *fmt, const char *a, const char *b);
/* The stream created by oxh_init(). */
void *oxh_internal_stream(void);
/* Largest n_vec (1..8) one GEMV launch can stage for (qtype, cols); 0 when
 * even a single activation does not fit. */
size_t oxh_gemv_max_nvec(uint32_t qtype, size_t cols);
/* The same for a launch that passes a buffer for the quantised activations
 * (up to 16 for Q8_0 weights, which then run on the matrix cores). */
size_t oxh_gemv_max_nvec_buffered(uint32_t qtype, size_t cols);

/* Sets the thread's error text (printf-style) and returns `status`. */
int oxh_internal_errorf(int status, const char *fmt, ...);
/* Compute units and index of the device oxh_init() chose (0 / -1 before it ran). */
int oxh_internal_n_cu(void);
int oxh_internal_device(void);
/* Host layer: drop the weight registry and the staging buffers (oxh_shutdown). */
void oxh_internal_host_reset(void);

/* Plans over the 32-value formats: a table of plain GEMV launches walked by one grid (oxh_kernels.hip).
 * `ops` is an array of OxhPlanOp; which = -1 for a type without such a launch. */
struct OxhPlanOp;
int oxh_internal_multi_which(uint32_t qtype);
int oxh_internal_multi_create(const struct OxhPlanOp *ops, size_t n_ops, void **handle);
int oxh_internal_multi_launch(void *handle, void *stream);
void oxh_internal_multi_info(const void *handle, size_t *n_items, size_t *workgroups, size_t *lds_bytes);
int oxh_internal_multi_destroy(void *handle);
/* Expert matmuls over many tokens per expert (oxh_experts.hip); both return a hipError_t.  `file_type` is
 * the weights' type without the tile-major mark, `pairs` the (token, expert) pairs in all, `max_tokens` the
 * most one expert can get; counts and offsets are in device memory.  The caller has checked the sizes. */
int oxh_internal_experts_init(void);
int oxh_internal_experts_long(uint32_t file_type, int tile_major, const void *const *d_w, float *const *d_out,
                              size_t n_mat, size_t n_expert, size_t rows, size_t cols, const void *d_acts,
                              size_t out_stride, const uint32_t *d_counts, const uint32_t *d_offsets, size_t pairs,
                              size_t max_tokens, void *stream);
/* the tile (rows, tokens) such a launch runs on; host arithmetic */
void oxh_internal_experts_long_tile(uint32_t file_type, size_t n_mat, size_t n_expert, size_t rows, size_t pairs, size_t cus,
                                    uint32_t tile[2]);
/* Q6_K (or widened Q2_K) prefill in 64 x 128 tiles whose weight operands the workgroup builds once
 * (oxh_mmq6.hip); both return a hipError_t.  Arguments checked by the caller. */
int oxh_internal_mmq6_init(void);
int oxh_internal_mmq6_shared(int widened_q2, const void *d_w, size_t rows, size_t blocks, const void *d_acts, size_t n_vec,
                             float *d_out, size_t out_stride, size_t cus, void *stream);
/* the token tiles such a launch is cut into; host arithmetic */
size_t oxh_internal_mmq6_tok_tiles(size_t rows, size_t n_vec, size_t cus);
/* The 32-value formats under a batch, in tiles of 64 or 128 rows x 64 tokens (oxh_mmq32.hip); init and launch return a
 * hipError_t.  leg: 0 Q8_0, 1 Q4_0, 2 Q4_1, 3 Q5_0, 4 Q5_1, 5 AL5_XS; `fits`: whether the grid holds the launch's tiles,
 * `tile`: their rows and tokens.  Arguments checked by the caller. */
#define OXH_MMQ32_MAX_BLOCKS 0xFFFFFFu       /* blocks of a row: 536 870 880 columns */
int oxh_internal_mmq32_init(void);
int oxh_internal_mmq32_fits(size_t rows, size_t n_vec);
void oxh_internal_mmq32_tile(size_t rows, size_t n_vec, size_t cus, uint32_t tile[2]);
int oxh_internal_mmq32(int leg, const void *d_w, size_t rows, size_t blocks, const void *d_acts, size_t n_vec, float *d_out,
                       size_t out_stride, size_t cus, void *stream);
/* K-quant matrices under at most 64 activations, a 16-row group to a workgroup (oxh_batch.hip); init and launch
 * return a hipError_t, `takes` whether a launch of these sizes belongs there (split: and could run as tiles that share
 * their columns through a workspace instead), `waves` the waves of its workgroups.
 * fmt: 0 Q4_K, 1 Q5_K, 2 Q6_K, 3 widened Q2_K.  Arguments checked by the caller. */
int oxh_internal_batch_init(void);
int oxh_internal_mmq_batch_takes(int fmt, size_t rows, size_t blocks, size_t n_vec, size_t cus, int split);
uint32_t oxh_internal_mmq_batch_waves(int fmt, size_t rows, size_t blocks, size_t n_vec, size_t cus);
int oxh_internal_mmq_batch(int fmt, const void *d_w, size_t rows, size_t blocks, const void *d_acts, size_t n_vec, float *d_out,
                           size_t out_stride, void *stream);
int oxh_internal_experts_batch_takes(int fmt, size_t n_mat, size_t n_expert, size_t rows, size_t blocks, size_t pairs,
                                     size_t n_tok, size_t cus);
int oxh_internal_experts_batch(int fmt, int tile_major, const void *const *d_w, float *const *d_out, size_t n_mat,
                               size_t n_expert, size_t rows, size_t blocks, const void *d_acts, size_t out_stride,
                               const uint32_t *d_counts, const uint32_t *d_offsets, size_t pairs, size_t max_tokens, void *stream);
/* Whether the runtime knows all of this memory (page-locked, managed or on the device) and so copies it without a
 * detour through staging of its own. */
int oxh_internal_runtime_memory(const void *p, size_t bytes);
size_t oxh_debug_host_ring_chunks(void);
/* Bytes of workspace an oxh_mmq_split launch of these sizes makes use of: what oxh_mmq_split_workspace says, or 0
 * where the launch runs on a kernel that needs none. */
size_t oxh_internal_mmq_split_use(uint32_t qtype, size_t rows, size_t cols, size_t n_vec, size_t out_stride);
/* 16-byte-granular copy by a kernel (either side may be page-locked host memory). */
int oxh_internal_copy16(void *dst, const void *src, size_t bytes, void *stream);
/* Wait for a stream by polling it `spins` times before blocking. */
int oxh_internal_stream_sync_spin(void *stream, unsigned spins);


/* The functions behind include/oxhip_lab.h's table (not exported by name). */
struct OxhPlan;
struct OxhMoe;
int oxh_debug_plan_stamps(struct OxhPlan *plan, uint64_t *d_stamps);
int oxh_debug_plan_phantom(struct OxhPlan *plan, int on);
int oxh_debug_plan_by_value(const struct OxhPlan *plan);
int oxh_debug_plan_draft(const struct OxhPlanOp *ops, size_t n_ops, uint32_t n_cu, uint64_t *out);
int oxh_debug_moe_workspace_parts(const struct OxhMoe *m, size_t n_tok, size_t parts[12]);
int oxh_debug_read_probe(const void *d_buf, size_t bytes, uint32_t *d_sink, void *stream);
int oxh_debug_mfma_probe(int valu_per_mfma, int waves_per_simd, double *pops);
int oxh_debug_mmq_kernel(uint32_t qtype, size_t rows, size_t cols, size_t n_vec, size_t n_cu, size_t ws_bytes, uint32_t out[4]);
int oxh_debug_experts_batch(uint32_t qtype, size_t n_mat, size_t n_expert, size_t rows, size_t cols, size_t top_k, size_t n_tok,
                            size_t n_cu);
int oxh_debug_experts_tile(uint32_t qtype, size_t n_mat, size_t n_expert, size_t rows, size_t pairs, size_t n_cu, uint32_t tile[2]);
uint64_t oxh_debug_mmq32_fetched(uint32_t block_bytes, uint32_t blocks, uint32_t row, uint32_t blk, uint32_t step);
int oxh_debug_subblock_sums(uint32_t qtype, const void *d_w, size_t rows, size_t cols, const void *d_act,
                            int32_t *d_sums, void *stream);

#ifdef __cplusplus
}
#endif
#endif
