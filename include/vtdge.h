/*
 * vtdge -- C ABI of the MI355X (gfx950) Dynamic Grained Encoder query path.
 *
 * One entry point per operator of the reference's native module `vtpack._C`
 * (vtpack/layers/csrc/vision.cpp:9-29) that lies on the inference query path,
 * plus the dense pieces of the transformer block that sit between them
 * (LayerNorm, Linear) so a whole block runs without leaving the library.
 *
 * Conventions
 *   - every pointer is a DEVICE pointer unless its name ends in `_host`;
 *   - the library never allocates, frees or synchronises: the caller owns all
 *     buffers, every kernel is enqueued on `stream` (a hipStream_t, passed as
 *     void* so the header needs no HIP include) and the call returns at once;
 *   - tensors are dense row-major unless explicit element strides are given;
 *   - `dtype` selects storage AND arithmetic flavour: VTDGE_F32 = fp32 storage,
 *     fp32 arithmetic; VTDGE_BF16 = bf16 storage, fp32 accumulation, one
 *     round-to-nearest-even on store;
 *   - packed ("sparse") operands are [rows, C] matrices whose row count is only
 *     known on the device after routing.  Such calls take `rows` (a host-side
 *     upper bound: grid size, buffer capacity) and `rows_dev` (nullable device
 *     pointer to the live int64 row count; when NULL, `rows` itself is live);
 *   - return value: VTDGE_OK (0) or a negative VTDGE_ERR_*; vtdge_last_error()
 *     gives a thread-local message.  No exceptions cross the ABI.
 */
#ifndef VTDGE_H
#define VTDGE_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define VTDGE_OK 0
#define VTDGE_ERR_ARG (-1)         /* NULL pointer, non-positive size, bad enum     */
#define VTDGE_ERR_UNSUPPORTED (-2) /* valid request outside the built kernel family */
#define VTDGE_ERR_LAUNCH (-3)      /* hipLaunchKernel / hipGetLastError failed      */

#define VTDGE_F32 0
#define VTDGE_BF16 1

#define VTDGE_ACT_NONE 0
#define VTDGE_ACT_GELU 1 /* exact erf GELU (torch.nn.GELU default) */

#define VTDGE_MAX_SPLITS 8

int vtdge_version(void);
const char *vtdge_last_error(void);
/* The demangled name of the kernel that the calling thread's latest launch was (the last one, for an entry point
 * that launches several), as a profiler lists it; "" before the first launch.  For measurement tools. */
const char *vtdge_last_kernel(void);
/* The same of the launch `back` (0 .. 7) before the latest one; "" where the thread has made fewer. */
const char *vtdge_recent_kernel(int back);

/* Router: region mean of the spatial tokens, Linear(C -> S), argmax.
 * Replaces DynamicRouter.forward + argmax (vtpack/layers/dge.py:145-150, :75).
 *   x       [B, extra + H*W, C]      weight [S, C]      bias [S]
 *   gate    [B, H/R, W/R, S] in `dtype` (nullable)      indices int64 [B, H/R, W/R]
 * The mean is taken over the R x R window in dy-outer / dx-inner order in fp32;
 * with VTDGE_BF16 the pooled value and the logits are rounded to bf16 as the
 * reference's modules would, and the argmax (lowest index wins a tie) is taken
 * on the rounded logits. */
int vtdge_router(const void *x, const void *weight, const void *bias, void *gate, int64_t *indices,
                 int B, int H, int W, int C, int extra, int R, int S, int dtype, void *stream);

/* The router and the block's first LayerNorm in one pass over x: gate / indices as vtdge_router, plus
 *   ln_out [B, extra + H*W, C] = LayerNorm(x) * ln_weight + ln_bias   (every token, the extra ones included).
 * Replaces DynamicRouter.forward + argmax (vtpack/layers/dge.py:145-150, :75) together with norm1 applied to
 * all tokens (vtpack/models/dge/deit_dge.py:127); both results are bit-identical to vtdge_router and
 * vtdge_layernorm.  R must be 4 or 2 and a row must fit one 16-byte vector per lane (C <= 512 in bf16, 256 in
 * fp32); VTDGE_ERR_UNSUPPORTED otherwise. */
int vtdge_router_layernorm(const void *x, const void *weight, const void *bias, void *gate, int64_t *indices,
                           const void *ln_weight, const void *ln_bias, float ln_eps, void *ln_out, int B, int H,
                           int W, int C, int extra, int R, int S, int dtype, void *stream);

/* Gate indices -> packed query descriptors.
 * Replaces grained_sample_index_to_patch
 * (vtpack/layers/csrc/grained_sample/grained_sample.cu:302-345, kernel :146-196).
 *   indices int64 [B, Hr, Wr]   splits int64 [S] (device, as in the reference)
 *   patches int64 [capacity_rows, 4] rows = [sample, y0, x0, size]; extra-token
 *           rows are [sample, -(e+1), 0, 1] (the reference leaves column 2 of
 *           those rows unwritten; 0 is written here).  Nullable: lengths only.
 *   offsets int64 [B+1] exclusive prefix of lengths (offsets[B] = total rows L)
 *   lengths int64 [B]   (the reference returns these on the host; copying them
 *           is the caller's business so that the fused path needs no sync)
 * Rows past `capacity_rows` are never written.  Gate indices outside [0,S) are
 * clamped (the reference reads out of bounds). */
int vtdge_index_to_patch(const int64_t *indices, const int64_t *splits, int B, int Hr, int Wr, int S,
                         int R, int extra, int64_t *patches, int64_t capacity_rows, int64_t *offsets,
                         int64_t *lengths, void *stream);

/* The same with the lengths on the host when the call returns, as the reference's callers take them: the kernel writes them to
 * `pinned` itself (int64 [B] of page-locked, coherent host memory), the call looks for them there for some time, waits for the
 * stream if they have not come by then, and copies them to lengths_host int64 [B] and their sum to total_host int64 [1].  Only
 * the lengths are there on return: patches and offsets are, like any result, ordered on `stream` and may still be being
 * written.  vtdge_index_to_patch_host_fits: 1 for the sizes that it takes (up to 16384 regions); others, and a stream
 * that is being captured: VTDGE_ERR_UNSUPPORTED, nothing launched. */
int vtdge_index_to_patch_host_fits(int B, int Hr, int Wr);
int vtdge_index_to_patch_host(const int64_t *indices, const int64_t *splits, int B, int Hr, int Wr, int S, int R, int extra,
                              int64_t *patches, int64_t capacity_rows, int64_t *offsets, int64_t *pinned,
                              int64_t *lengths_host, int64_t *total_host, void *stream);

/* Every patch of every granularity (exported by the reference, unused by its
 * models).  Replaces grained_sample_index_to_patch_dense (grained_sample.cu:347-433).
 *   patches int64 [B * per_sample, 4], per_sample = extra + Hr*Wr*sum(splits^2)
 *   splits_host: HOST pointer (the reference copies it to the host too, :401). */
int vtdge_index_to_patch_dense(const int64_t *splits_host, int B, int Hr, int Wr, int S, int R, int extra,
                               int64_t *patches, void *stream);

/* Grained sampling ("compress"): one packed query row per patch = mean of its
 * size x size token window (fp32 accumulation, dy outer / dx inner, one divide),
 * or a copy of the extra token.
 * Replaces grained_sample_compress (grained_sample.cu:198-239, kernel :31-69).
 *   x [B, N, C]   patches [rows, 4]   out [rows, C]
 * Optional fused LayerNorm of the (rounded) output row, as the block applies
 * norm1 to the compressed queries (vtpack/models/dge/deit_dge.py:127):
 *   ln_out [rows, C] nullable; ln_weight, ln_bias [C]. */
int vtdge_compress(const void *x, const int64_t *patches, const int64_t *rows_dev, int64_t rows,
                   void *out, void *ln_out, const void *ln_weight, const void *ln_bias, float ln_eps,
                   int B, int N, int C, int W, int extra, int dtype, void *stream);

/* Scatter back ("decompress"): every token covered by a patch receives
 *   out[b,t,:] = (in[row,:] - sub[row,:]) + ref[b,t,:]
 * with `sub` and `ref` each optional (NULL = term absent).
 * Replaces grained_sample_decompress, both overloads (grained_sample.cu:241-300,
 * kernels :71-144; ref == NULL is is_add_ref = false) and, with `sub`, the
 * subtraction in DynamicGrainedEncoder.decompress (vtpack/layers/dge.py:88).
 * In bf16 the difference is rounded to bf16 before the add, as the reference's
 * separate elementwise op would.  Tokens no patch covers are left untouched. */
int vtdge_decompress(const void *in, const void *sub, const int64_t *patches, const int64_t *rows_dev,
                     int64_t rows, const void *ref, void *out, int B, int N, int C, int W, int extra,
                     int dtype, void *stream);

/* The same scatter with `ref` present, plus the LayerNorm of every token written:
 *   out[b,t,:] = (in[row,:] - sub[row,:]) + ref[b,t,:],   ln_out[b,t,:] = LayerNorm(out[b,t,:])
 * i.e. the last step of one block (vtpack/layers/dge.py:87-112) together with the first LayerNorm of the next
 * (norm1 at vtpack/models/dge/deit_dge.py:127), which would read the same tokens back.  The statistics are taken
 * from the values as stored in `out`.  Rows of at most 64 16-byte vectors (C <= 512 in bf16, 256 in fp32). */
int vtdge_decompress_layernorm(const void *in, const void *sub, const int64_t *patches, const int64_t *rows_dev,
                               int64_t rows, const void *ref, void *out, void *ln_out, const void *ln_weight,
                               const void *ln_bias, float ln_eps, int B, int N, int C, int W, int extra, int dtype,
                               void *stream);

/* The adjoints of the two, for their gradients (vtpack/layers/grained_sample.py:26-38, :61-78):
 *   vtdge_compress_sum     out[row] = the SUM of the tokens its patch covers (the gradient of vtdge_decompress's `in`)
 *   vtdge_decompress_mean  out[token] = in[row] / area of the patch that covers it (+ add[token], nullable): the gradient of
 *                          vtdge_compress's `x` */
int vtdge_compress_sum(const void *x, const int64_t *patches, int64_t rows, void *out, int B, int N, int C, int W, int extra,
                       int dtype, void *stream);
int vtdge_decompress_mean(const void *in, const int64_t *patches, int64_t rows, const void *add, void *out, int B, int N,
                          int C, int W, int extra, int dtype, void *stream);

/* Scatter back by region, and the NEXT block's router on the tokens just written:
 *   out[b,t,:] = (in[row,:] - sub[row,:]) + ref[b,t,:]        (as vtdge_decompress with `sub` and `ref`; sub nullable)
 *   next_gate [B, H/R, W/R, S2], next_indices int64 [B, H/R, W/R] = vtdge_router(out, next_weight, next_bias)
 * i.e. the last step of one block (vtpack/layers/dge.py:87-112) together with DynamicRouter.forward + argmax of the
 * block that follows (vtpack/layers/dge.py:145-150, :75), which would read the same tokens back.  The packed rows
 * are found from this block's gate indices `cur_indices` [B, H/R, W/R] (S splits in `splits`, as given to
 * vtdge_index_to_patch) and `offsets` [B+1] instead of the patch list.  Both results are bit-identical to the two
 * separate calls.  next_weight == NULL (with next_bias, next_indices) leaves the router out.  R must be 4 and every
 * split size must divide it; VTDGE_ERR_UNSUPPORTED for another R.
 * out_records (nullable) [B * (extra + H*W), 16] bf16: the statistics record of every row of `out` as stored (mean
 * and sqrt(var + records_eps), see vtdge_layernorm_stats), for the next block's norm1 -> kv through
 * vtdge_linear_layernorm; one-pass fp32 sums about a value of the row itself.  bf16 rows of 264 to 512 channels.
 * next_counts (nullable; needs the next router) uint8 [B * H/R * W/R]: the number of queries the next block takes
 * from every region, next_splits[next_indices]^2 with next_splits int64 [S2] on the device: what
 * vtdge_compress_regions adds up to place a region's queries.
 * region_rows (nullable) int32 [B * H/R * W/R] with cur_counts uint8 of the same length: the first packed row and the
 * query count of every region of THIS block as vtdge_compress_regions left them; the kernel then takes a region's
 * place from them instead of adding it up from cur_indices and offsets. */
int vtdge_decompress_router(const void *in, const void *sub, const int64_t *cur_indices, const int64_t *splits,
                            const int64_t *offsets, const void *ref, void *out, const void *next_weight,
                            const void *next_bias, void *next_gate, int64_t *next_indices, void *out_records,
                            float records_eps, const int64_t *next_splits, uint8_t *next_counts,
                            const int32_t *region_rows, const uint8_t *cur_counts, int B, int H, int W, int C,
                            int extra, int R, int S, int S2, int dtype, void *stream);

/* vtdge_decompress_router that goes on to pack the NEXT block's queries from the tokens it has just written: the
 * scatter-back of one block (vtpack/layers/dge.py:87-112), the next block's router (:145-150, :75) and the next
 * block's index->patch + compress (:76-79) in one launch, i.e. vtdge_decompress_router followed by
 * vtdge_compress_regions without a second pass over the tokens.  All outputs are bit-identical to those two calls.
 *   next_comp [capacity_rows, C], next_comp_records [capacity_rows, 16] bf16 with next_records_eps,
 *   next_patches (nullable) [capacity_rows, 4], next_offsets [B+1], next_region_rows (nullable) int32 [regions]:
 *   as vtdge_compress_regions writes comp, records, patches, offsets and region_rows (lengths are the differences
 *   of the offsets and are not written)
 *   workspace: vtdge_decompress_router_compress_workspace(B, H, W, R) bytes of device memory, 8-byte aligned, all
 *   zero when the kernel starts (clear_workspace != 0: the call clears it first with a small fill kernel; a caller
 *   that keeps one slice per block can clear them all at once instead).  The workgroups hand the running number of
 *   queries along through it (one 64-bit word each); word 0 is raised to 1 if a workgroup gave up waiting for the
 *   ones before it, in which case rows are missing from next_comp and next_offsets[B] exceeds capacity_rows.
 * bf16 rows of 264 to 512 channels, R = 4, splits out of {1, 2, 4}, the regions a multiple of 4 up to 65536, the
 * next router with its splits and count bytes, out_records present; VTDGE_ERR_UNSUPPORTED otherwise. */
int64_t vtdge_decompress_router_compress_workspace(int B, int H, int W, int R);
int vtdge_decompress_router_compress(const void *in, const void *sub, const int64_t *cur_indices,
                                     const int64_t *splits, const int64_t *offsets, const void *ref, void *out,
                                     const void *next_weight, const void *next_bias, void *next_gate,
                                     int64_t *next_indices, void *out_records, float records_eps,
                                     const int64_t *next_splits, uint8_t *next_counts, const int32_t *region_rows,
                                     const uint8_t *cur_counts, void *next_comp, void *next_comp_records,
                                     float next_records_eps, int64_t *next_patches, int64_t capacity_rows,
                                     int64_t *next_offsets, int32_t *next_region_rows, void *workspace,
                                     int64_t workspace_bytes, int clear_workspace, int B, int H, int W, int C,
                                     int extra, int R, int S, int S2, int dtype, void *stream);

/* vtdge_decompress_router_compress for callers that cannot allocate device memory (code under HIP graph capture,
 * serving loops and harnesses that forbid hipMalloc); it has no counterpart in the reference.  The arguments are
 * those of vtdge_decompress_router_compress without the workspace: the status words live in an array inside the
 * library's device image (128 KB on every GPU the library runs on, held until the process ends), cleared by a small
 * fill kernel on `stream` before the kernel runs.  The call allocates and frees nothing.  At most 65536 regions
 * (VTDGE_ERR_UNSUPPORTED beyond).  All calls on one GPU share the array: calls that overlap on one GPU (two streams,
 * two threads) race - run them in turn.  The first call on a GPU looks the array's address up
 * (hipGetSymbolAddress) and should therefore come before any stream capture.  A kernel that gave up shows as
 * next_offsets[B] > capacity_rows, as in vtdge_decompress_router_compress. */
int vtdge_decompress_router_compress_static(const void *in, const void *sub, const int64_t *cur_indices,
                                            const int64_t *splits, const int64_t *offsets, const void *ref,
                                            void *out, const void *next_weight, const void *next_bias,
                                            void *next_gate, int64_t *next_indices, void *out_records,
                                            float records_eps, const int64_t *next_splits, uint8_t *next_counts,
                                            const int32_t *region_rows, const uint8_t *cur_counts, void *next_comp,
                                            void *next_comp_records, float next_records_eps, int64_t *next_patches,
                                            int64_t capacity_rows, int64_t *next_offsets, int32_t *next_region_rows,
                                            int B, int H, int W, int C, int extra, int R, int S, int S2, int dtype,
                                            void *stream);

/* Up to some thousand regions (see vtdge_region_step_fits): from the packed queries of one block to those of the next in one launch, a
 * workgroup per 4 x 4 region - vtdge_decompress_router, vtdge_compress_regions (or vtdge_index_to_patch and vtdge_compress)
 * and, of tokens and packed rows, either the statistics records or the LayerNorm, each bit for bit.
 *   in, sub [.., C]: the packed queries after and before the block   cur_indices, splits, offsets: its gate indices, splits and
 *   first rows   region_rows with cur_counts (nullable) as in vtdge_decompress_router   ref, out [B, extra + H*W, C]
 *   next_*: of the block that follows, as in vtdge_decompress_router_compress; S and S2 split sizes, all of them 1, 2 or 4
 *   out_records, next_comp_records (nullable, bf16 rows of 264 to 512 channels) or out_ln [B * (extra + H*W), C], next_comp_ln
 *   [capacity_rows, C] (nullable) with ln_weight, ln_bias; eps of either
 *   workspace: vtdge_region_step_workspace bytes, zero; its first word stays 0 unless the kernel gave up waiting (rows are missing then
 *   and next_offsets[B] exceeds capacity_rows)
 * vtdge_region_step_fits: 1 for rows of 1 to 192 whole 16-byte vectors, up to 64 extra tokens and as many regions (1280 to 12800, by
 * width and type) as the launch is faster for than the separate ones. */
int vtdge_region_step_fits(int B, int H, int W, int C, int extra, int dtype);
int64_t vtdge_region_step_workspace(int B, int H, int W);
int vtdge_region_step(const void *in, const void *sub, const int64_t *cur_indices, const int64_t *splits,
                      const int64_t *offsets, const int32_t *region_rows, const uint8_t *cur_counts, const void *ref, void *out,
                      const void *next_weight, const void *next_bias, void *next_gate, int64_t *next_indices,
                      const int64_t *next_splits, uint8_t *next_counts, void *out_records, void *out_ln,
                      const void *ln_weight, const void *ln_bias, float eps, void *next_comp, void *next_comp_records,
                      void *next_comp_ln, int64_t *next_patches, int64_t capacity_rows, int64_t *next_offsets,
                      int32_t *next_region_rows, void *workspace, int64_t workspace_bytes, int B, int H, int W, int C, int extra,
                      int S, int S2, int dtype, void *stream);

/* The router of a model's FIRST block together with the statistics records of all its tokens (no scatter-back
 * precedes it that could leave them): vtdge_router and vtdge_layernorm_stats in one pass over x, i.e.
 * DynamicRouter.forward + argmax (vtpack/layers/dge.py:145-150, :75) and the statistics half of norm1
 * (vtpack/models/dge/deit_dge.py:127).  gate / indices are bit-identical to vtdge_router's; the records are one-pass
 * fp32 sums about a value of the row itself, as vtdge_decompress_router writes them.
 *   x [B, extra + H*W, C]   records [B * (extra + H*W), 16] bf16   counts (nullable) as in vtdge_decompress_router,
 *   from `splits` int64 [S] on the device
 *   front_rows (nullable) [extra, C]: rows that are first stored as tokens 0 .. extra-1 of EVERY sample of x - the
 *   class (and distillation) token plus its position embedding, which the reference concatenates in front of the
 *   patch tokens (deit_dge.py:270-277) and which do not depend on the sample.
 *   clear_words (nullable) with n_clear_words: 64-bit words the launch sets to zero on the way - the workspaces of
 *   the vtdge_decompress_router_compress calls that follow it on the stream, so that a forward needs no fill kernel.
 * bf16 rows of 264 to 512 channels, R = 4. */
int vtdge_router_stats(void *x, const void *front_rows, const void *weight, const void *bias, void *gate,
                       int64_t *indices, void *records, float records_eps, const int64_t *splits, uint8_t *counts,
                       void *clear_words, int64_t n_clear_words, int B, int H, int W, int C, int extra, int R, int S,
                       int dtype, void *stream);

/* Gate indices -> packed queries in one step, by region: vtdge_index_to_patch and vtdge_compress together, i.e.
 * grained_sample_index_to_patch followed by grained_sample_compress
 * (vtpack/layers/csrc/grained_sample/grained_sample.cu:302-345 with :146-196, and :198-239 with :31-69) as
 * DynamicGrainedEncoder.compress calls them (vtpack/layers/dge.py:76-79), without the descriptor list in between: a
 * region's packed rows are consecutive, so the kernel places them from the query counts of the regions before it.
 *   x [B, extra + H*W, C]   indices int64 [B, H/R, W/R]   splits int64 [S] (device)
 *   counts  nullable uint8 [B * H/R * W/R, padded to a multiple of 16 bytes]: splits[indices]^2 per region, as
 *           vtdge_decompress_router leaves them; without it the kernel works the counts out from `indices`
 *   comp    [capacity_rows, C]: the packed queries, bit for bit those of vtdge_compress
 *   records nullable [capacity_rows, 16] bf16: the statistics record of every row of comp as stored (mean and
 *           sqrt(var + records_eps), see vtdge_layernorm_stats) for a vtdge_linear_layernorm that takes comp next
 *           (norm1 -> q, vtpack/models/dge/deit_dge.py:127 with :72); bf16 only
 *   patches (nullable), offsets [B+1], lengths [B]: as vtdge_index_to_patch writes them
 *   region_rows (nullable) int32 [B * H/R * W/R]: the first packed row of every region, for vtdge_decompress_router
 * The caller guarantees capacity_rows >= the number of queries (B * (extra + H*W) always is).  R must be 4 with splits
 * out of {1, 2, 4}, a row one 16-byte vector per lane (C <= 512 in bf16, 256 in fp32), at most 65536 regions and
 * 64 extra tokens; VTDGE_ERR_UNSUPPORTED otherwise. */
int vtdge_compress_regions(const void *x, const int64_t *indices, const int64_t *splits, const uint8_t *counts,
                           void *comp, void *records, float records_eps, int64_t *patches, int64_t capacity_rows,
                           int64_t *offsets, int64_t *lengths, int32_t *region_rows, int B, int H, int W, int C,
                           int extra, int R, int S, int dtype, void *stream);

/* The patch embedding of a pyramid model's first stage in one pass over the images: Conv2d(Cin, N, kernel P, stride P)
 * + bias, the embedding's LayerNorm and `+ pos_embed` (vtpack/models/dge/pvt_dge.py:143-176 with :312-314), each
 * rounded to the storage type as the separate modules would round.
 *   images [B, Cin, S, S]   weight [N, Cin*P*P] (the convolution's weight, flattened)   bias, ln_weight, ln_bias [N]
 *   pos (nullable) [(S/P)^2, N]   out [B * (S/P)^2, N]
 * bf16, Cin = 3, P = 4, N = 64, S a multiple of 64; VTDGE_ERR_UNSUPPORTED otherwise (the caller then gathers the patches
 * and uses vtdge_linear, vtdge_layernorm_add). */
int vtdge_patch_embed_norm(const void *images, const void *weight, const void *bias, const void *ln_weight,
                           const void *ln_bias, float ln_eps, const void *pos, void *out, int B, int Cin, int S, int P,
                           int N, int dtype, void *stream);

/* vtdge_layernorm followed by the addition of a periodic set of rows: out[r] = LayerNorm(x[r]) + add[r mod add_rows],
 * the LayerNorm's result rounded to the storage type before the addition as the two modules would.  Stands in for a
 * patch embedding's norm followed by `x + pos_embed` (vtpack/models/dge/pvt_dge.py:176 with :312-314; add =
 * pos_embed [H*W, C], rows = B * H*W). */
int vtdge_layernorm_add(const void *x, const void *weight, const void *bias, const void *add, int64_t add_rows,
                        void *out, int64_t rows, int C, float eps, int dtype, void *stream);

/* Token rows x [B, tokens, C] (rows dense, samples batch_stride elements apart) as feature maps out [B, C, tokens], dense: the
 * permute(0, 3, 1, 2).contiguous() of vtpack/models/dge/pvt_dge.py's stage outputs. */
int vtdge_rows_to_maps(const void *x, int64_t batch_stride, void *out, int B, int tokens, int C, int dtype, void *stream);

/* Row-wise LayerNorm over the last dimension (biased variance, fp32 statistics).
 * Stands in for nn.LayerNorm(eps=1e-6) at vtpack/models/dge/deit_dge.py:127-128. */
int vtdge_layernorm(const void *x, const void *weight, const void *bias, void *out, const int64_t *rows_dev,
                    int64_t rows, int C, float eps, int dtype, void *stream);
/* The same for input rows that lie in groups: row r is x + (r / x_group_rows) * x_group_stride + (r % x_group_rows) * C
 * (elements); out [rows, C] is dense.  The final norm of a model only on the rows the classifier reads - the class
 * (and distillation) tokens, the first rows of every sample (vtpack/models/dge/deit_dge.py:283-285 with :288-299) -
 * without a gathered copy of them: x_group_rows = extra, x_group_stride = N * C. */
int vtdge_layernorm_rows(const void *x, int64_t x_group_stride, int x_group_rows, const void *weight, const void *bias,
                         void *out, int64_t rows, int C, float eps, int dtype, void *stream);

/* Packed-M Linear: out[m, n] = act(sum_k A[m,k] * W[n,k] + bias[n]) + residual[m,n].
 * The M dimension is the packed query set of all samples (weights are shared),
 * which is what the reference's q / proj / fc1 / fc2 nn.Linear calls compute on
 * [L, C] (vtpack/models/dge/deit_dge.py:72,96,38-44) and kv on [B*N, C] (:73).
 *   A [rows, K] leading dim lda      W [N, K] dense      bias [N] nullable
 *   residual [rows, N] leading dim ldr, nullable         out [rows, N] leading dim ldo
 * MFMA kernels; K must be a multiple of 16 bytes worth of elements (4 fp32 / 8 bf16).  Rows of K that are a
 * multiple of 128 bytes (and 16-byte aligned operands) take the direct-to-LDS persistent kernel. */
int vtdge_linear(const void *A, int64_t lda, const void *W, const void *bias, const void *residual,
                 int64_t ldr, void *out, int64_t ldo, const int64_t *rows_dev, int64_t rows, int N, int K,
                 int act, int dtype, void *stream);

/* The same Linear with a packed copy of W beside it.  The weight-stationary kernels keep a strip of W in registers
 * for the life of a workgroup; from a copy laid out in the order of those registers they fill them with contiguous
 * loads (half the start-up time of a launch).  The weights of an nn.Linear (vtpack/models/dge/deit_dge.py:70-74,
 * :38-44) do not change between calls at inference, so a caller packs them once:
 *   vtdge_linear_packed_size  *bytes = size of the packed copy of W [N, K], or 0 when no kernel for this shape uses
 *                             one (pass packed = NULL then)
 *   vtdge_linear_prepack      fills `packed` (16-byte aligned, *bytes long) from W; VTDGE_ERR_UNSUPPORTED when the
 *                             size is 0
 *   vtdge_linear_prepacked    vtdge_linear with `packed` (nullable; must have been made from this W).  W itself is
 *                             still required: the kernels chosen for few rows read it.
 * Results are bit-identical with and without the packed copy. */
int vtdge_linear_packed_size(int N, int K, int dtype, int64_t *bytes);
int vtdge_linear_prepack(const void *W, int N, int K, int dtype, void *packed, void *stream);
int vtdge_linear_prepacked(const void *A, int64_t lda, const void *W, const void *packed, const void *bias,
                           const void *residual, int64_t ldr, void *out, int64_t ldo, const int64_t *rows_dev,
                           int64_t rows, int N, int K, int act, int dtype, void *stream);

/* fp32 Linears on the bf16 matrix instructions: for VTDGE_F32, `packed` of vtdge_linear_prepacked is a copy of W split into
 * three bf16 parts (6 bytes a value).  The sums of the partial products of weight 2^-17 and above, in fp32, are as exact as
 * those of the fp32 instructions (not the same bits; up to 2^-24 of a product is left out) and 1.2 to 1.5 times as fast, the
 * split (3 to 16 us for the weights of a block) aside.
 *   vtdge_linear_split_size    *bytes = size of the split copy of W [N, K], or 0 when there is none (N no multiple of 64, K
 *                              none of 32)
 *   vtdge_linear_split         fills `split` (16-byte aligned, *bytes long) from W; VTDGE_ERR_UNSUPPORTED where the size is 0
 *   vtdge_linear_split_set     the same for `count` weights in one launch: weights_host[i] [N_host[i], K_host[i]] to byte
 *                              at_host[i] of `split` (all four tables on the host)
 *   vtdge_linear_split_wanted  1 where vtdge_linear_prepacked uses the copy for that many rows, 0 where W is multiplied as it
 *                              is, with or without one
 * W itself is always required: blocks of the result with infinities, NaN or values outside the range of the split are
 * worked out from it. */
int vtdge_linear_split_size(int N, int K, int64_t *bytes);
int vtdge_linear_split(const void *W, int N, int K, void *split, void *stream);
int vtdge_linear_split_set(const void *const *weights_host, const int32_t *N_host, const int32_t *K_host, const int64_t *at_host,
                           int count, void *split, void *stream);
int vtdge_linear_split_wanted(int64_t rows, int N, int K);

/* Patch embedding, position embedding included: the stride-P P x P convolution of the reference's PatchEmbed
 * (nn.Conv2d, vtpack/models/dge/deit_dge.py:141-155) as a Linear over the patches, read straight from the images
 * (no unfolded copy), with the addition of the position table (x = x + pos_embed, deit_dge.py:277) in its epilogue:
 *   images [B, Cin, S, S]   weight [C, Cin * P * P] (the convolution's weight, flattened)   bias [C]
 *   pos_embed [extra + G*G, C], G = S / P   tokens [B, extra + G*G, C]
 *   tokens[b, extra + gy*G + gx, :] = conv(images)[b, :, gy, gx] + bias + pos_embed[extra + gy*G + gx, :]
 * in fp32 with one rounding; rows 0 .. extra-1 of every sample (class / distillation tokens) are left untouched.
 * A patch row must be 16, 32, 64 or 128 bytes (P = 16: both types) and all operands 16-byte aligned, else
 * VTDGE_ERR_UNSUPPORTED. */
int vtdge_patch_embed(const void *images, const void *weight, const void *bias, const void *pos_embed, void *tokens,
                      int B, int Cin, int S, int P, int C, int extra, int dtype, void *stream);

/* A stride-P P x P convolution over a channels-last token grid, as a Linear over the P x P blocks of tokens read
 * straight from the grid (no gathered copy): the spatial reduction in front of the key/value projection
 * (nn.Conv2d(dim, dim, sr_ratio, sr_ratio), vtpack/models/dge/pvt_dge.py:62, :81-83) and the patch embedding of the
 * later stages (nn.Conv2d(in_chans, embed_dim, patch_size, patch_size), pvt_dge.py:164, :175), whose input here stays
 * [B, H*W, C] tokens instead of going back to [B, C, H, W]:
 *   tokens [B, H*W, C]   weight [N, P*P*C], the convolution's weight in (kh, kw, c) order   bias [N]
 *   out [B*(H/P)*(W/P), N]:  out[(b, gy, gx), :] = sum over (dy, dx, c) of
 *        tokens[b, (gy*P + dy)*W + gx*P + dx, c] * weight[:, (dy*P + dx)*C + c]  + bias,   fp32 sums, one rounding.
 * C values must fill whole 128-byte pieces (C % 64 == 0 for bf16, % 32 for fp32), H and W be multiples of P and all
 * operands 16-byte aligned, else VTDGE_ERR_UNSUPPORTED. */
int vtdge_patch_linear(const void *tokens, const void *weight, const void *bias, void *out, int B, int H, int W, int C,
                       int P, int N, int dtype, void *stream);

/* vtdge_patch_linear on LayerNorm(tokens), each token normalised on its way (norm1 in front of the spatial reduction,
 * vtpack/models/dge/pvt_dge.py:81-83): the LayerNorm rounded to the storage type, products of C columns with fp32 sums and
 * one rounding, and with out_ln_weight / out_ln_bias (nullable together) the LayerNorm of those rows in their place, as the
 * separate calls would.  Taken where vtdge_layernorm_patch_linear_fits says 1 (bf16, 64 or 128 channels, P a multiple of
 * 256 / C); VTDGE_ERR_UNSUPPORTED otherwise.  vtdge_layernorm_patch_linear_wanted: whether it is also the faster way.
 *   packed   the weight [C, P*P*C] as vtdge_layernorm_patch_pack leaves it: `count` weights one behind the other, of
 *            C * P*P*C values each */
int vtdge_layernorm_patch_linear_fits(int B, int H, int W, int C, int P, int dtype);
int vtdge_layernorm_patch_linear_wanted(int B, int H, int W, int C, int P, int dtype);
int vtdge_layernorm_patch_pack(const void *const *weights_host, int count, void *packed, int C, int P, void *stream);
int vtdge_layernorm_patch_linear(const void *tokens, const void *ln_weight, const void *ln_bias, float eps,
                                 const void *packed, const void *bias, const void *out_ln_weight, const void *out_ln_bias,
                                 float out_eps, void *out, int B, int H, int W, int C, int P, int dtype, void *stream);

/* LayerNorm folded into the Linear that consumes it: out = act(LayerNorm(A) W^T + bias) computed from the raw rows
 * of A, so that nn.LayerNorm followed by nn.Linear (norm1 -> kv and norm2 -> fc1,
 * vtpack/models/dge/deit_dge.py:127-128 with :73 and :38-44) costs no pass over the rows of its own:
 *     LayerNorm(a) W^T + bias = rstd * (a W'^T - mean * colsum(W') + sigma * b'),
 *     W' = W * ln_weight (rounded to the storage type),  b' = bias + W ln_bias,  sigma = 1 / rstd = sqrt(var + eps).
 *   vtdge_layernorm_stats   records [rows, 16] bf16 (32 bytes a row): mean and sigma of every row of x [rows, C],
 *                           each split into bf16 parts in the operand order of the matrix instruction (two-pass
 *                           fp32 statistics, as vtdge_layernorm).  Other kernels that produce the rows can write
 *                           the same records (see vtdge_decompress_router, vtdge_linear_stats).
 *   vtdge_layernorm_fold    once per weight: W_folded [N, K] = W', col_records [N, 16] bf16 = -colsum(W') and b'
 *                           in the matching order.  bias is nullable.
 *   vtdge_linear_layernorm  the Linear: A [rows, K] raw rows with their row_records, W_folded (and optionally its
 *                           packed copy from vtdge_linear_prepack), col_records.  Weight-stationary kernel only:
 *                           bf16, K = 384, N a multiple of 384 up to 3072, rows >= 2048 (capacity; the live count
 *                           may be anything), else VTDGE_ERR_UNSUPPORTED.
 * Against vtdge_layernorm followed by vtdge_linear the result differs by the rounding of W' instead of that of
 * LayerNorm(a) to bf16: the same order of magnitude, not the same bits. */
/* vtdge_linear (no activation) that also writes the statistics records of its output rows, for a
 * vtdge_linear_layernorm that takes `out` next: proj + residual followed by norm2 -> fc1
 * (vtpack/models/dge/deit_dge.py:96, :128, :38-44).  The records are computed from the fp32 sums before their rounding
 * to bf16.  Weight-stationary kernel with one column group only: bf16, K = 384, N = 384, rows >= 2048. */
int vtdge_linear_stats(const void *A, int64_t lda, const void *W, const void *packed, const void *bias,
                       const void *residual, int64_t ldr, void *out, int64_t ldo, void *out_records,
                       float records_eps, const int64_t *rows_dev, int64_t rows, int N, int K, int dtype,
                       void *stream);
int vtdge_layernorm_stats(const void *x, void *records, const int64_t *rows_dev, int64_t rows, int C, float eps,
                          int dtype, void *stream);
int vtdge_layernorm_fold(const void *W, const void *bias, const void *ln_weight, const void *ln_bias, int N, int K,
                         int dtype, void *W_folded, void *col_records, void *stream);
int vtdge_linear_layernorm(const void *A, int64_t lda, const void *row_records, const void *W_folded,
                           const void *packed, const void *col_records, void *out, int64_t ldo,
                           const int64_t *rows_dev, int64_t rows, int N, int K, int act, int dtype, void *stream);

/* Two vtdge_linear_layernorm calls without activation as ONE launch: norm1 -> kv on all tokens and norm1 -> q on the
 * packed queries (vtpack/models/dge/deit_dge.py:127 with :73 and :72), which the reference issues one after the
 * other.  The workgroups are dealt out between the two in proportion to their live rows (read on the device), so
 * the smaller one no longer runs a few tiles per workgroup behind the fixed cost of a launch of its own.  Operands
 * with suffix 0 and 1 as in vtdge_linear_layernorm, same K; results are bit-identical to the two separate calls. */
int vtdge_linear_layernorm_pair(const void *A0, int64_t lda0, const void *row_records0, const void *W_folded0,
                                const void *packed0, const void *col_records0, void *out0, int64_t ldo0,
                                const int64_t *rows_dev0, int64_t rows0, int N0, const void *A1, int64_t lda1,
                                const void *row_records1, const void *W_folded1, const void *packed1,
                                const void *col_records1, void *out1, int64_t ldo1, const int64_t *rows_dev1,
                                int64_t rows1, int N1, int K, int dtype, void *stream);

/* Sparse attention of packed queries against each sample's full K/V:
 *   out[rows of sample i, head a] = softmax(scale * Q_i,a K_i,a^T) V_i,a
 * Replaces batched_sparse_attention_forward
 * (vtpack/layers/csrc/batched_sparse_gemm/batched_sparse_gemm.cu:219-305).
 * All operands are addressed through element strides so that both the
 * reference's contiguous [h, L, d] / [h, B, n, d] tensors and the un-permuted
 * outputs of the q / kv Linears ([L, h*d] and [B, n, 2, h, d]) can be passed:
 *   q(row, a, c)   = q[row*q_row_stride + a*q_head_stride + c]
 *   k(i, t, a, c)  = k[i*kv_batch_stride + t*kv_tok_stride + a*kv_head_stride + c]  (same for v)
 *   out(row, a, c) = out[row*o_row_stride + a*o_head_stride + c]
 *   offsets int64 [B+1] (device) exclusive prefix of the per-sample query counts
 *   max_rows_per_sample: host upper bound of any sample's query count (grid size)
 * head_dim d must be 64 or 32. */
int vtdge_sparse_attention(const void *q, int64_t q_row_stride, int64_t q_head_stride, const void *k,
                           const void *v, int64_t kv_batch_stride, int64_t kv_tok_stride,
                           int64_t kv_head_stride, const int64_t *offsets, void *out, int64_t o_row_stride,
                           int64_t o_head_stride, int B, int h, int d, int n, int max_rows_per_sample,
                           float scale, int dtype, void *stream);

/* Per-sample variable-length batched matmul over heads.
 * Replaces batched_sparse_gemm_forward and batched_sparse_gemm_v2_forward
 * (batched_sparse_gemm.cu:150-195, :83-148):
 *   a [h, La, ka], b [h, Lb, kb]; sample i uses rows a_offsets[i]..a_offsets[i+1]
 *   of a and b_offsets[i]..b_offsets[i+1] of b, each optionally transposed in its
 *   last two dims; out [h, out_rows, out_cols] is the concatenation along dim 1.
 *   a_offsets, b_offsets int64 [B+1] on the device.
 *   max_m: host upper bound of any sample's output row count (grid size). */
int vtdge_batched_sparse_gemm(const void *a, const void *b, const int64_t *a_offsets, const int64_t *b_offsets,
                              void *out, int B, int h, int64_t La, int ka, int64_t Lb, int kb, int trans_a,
                              int trans_b, int64_t out_rows, int64_t out_cols, int64_t max_m, int dtype,
                              void *stream);

/* vtdge_sparse_attention for training: bf16, head dim 64, scores of the queries as given (not rounded once more, times the
 * scale) and of any value, -infinity among the first ones included; the probabilities are those that
 * vtdge_sparse_attention_backward works out again. */
int vtdge_sparse_attention_train(const void *q, int64_t q_row_stride, int64_t q_head_stride, const void *k, const void *v,
                                 int64_t kv_batch_stride, int64_t kv_tok_stride, int64_t kv_head_stride,
                                 const int64_t *offsets, void *out, int64_t o_row_stride, int64_t o_head_stride, int B, int h,
                                 int d, int n, int max_rows_per_sample, float scale, int dtype, void *stream);

/* Gradients of vtdge_sparse_attention: dq, dk, dv from its operands and the output's gradient, as autograd
 * through the reference's training composition would give them (two batched products around a softmax,
 * vtpack/models/dge/deit_dge.py:86-95), without score-sized tensors.  Strides as in vtdge_sparse_attention, those of
 * `dout` under o_*.  `out` is not read and may be NULL.  workspace: 2 * h * L floats, L = offsets[B] = rows of q.  Gradients of keys and values of a sample
 * without queries are zero.  Head dim 64. */
int vtdge_sparse_attention_backward(const void *q, int64_t q_row_stride, int64_t q_head_stride, const void *k, const void *v,
                                    int64_t kv_batch_stride, int64_t kv_tok_stride, int64_t kv_head_stride, const void *out,
                                    const void *dout, int64_t o_row_stride, int64_t o_head_stride, const int64_t *offsets,
                                    void *dq, int64_t dq_row_stride, int64_t dq_head_stride, void *dk, void *dv,
                                    int64_t dkv_batch_stride, int64_t dkv_tok_stride, int64_t dkv_head_stride,
                                    float *workspace, int64_t L, int B, int h, int d, int n, int max_rows_per_sample,
                                    float scale, int dtype, void *stream);

/* The same from a workspace of 3 * h * L floats, which keeps a row's maximum and its sum apart: the gradients of fp32 operands
 * are as exact as the composition's then (2 * h * L floats: about 1.4 times its error). */
int vtdge_sparse_attention_train_backward(const void *q, int64_t q_row_stride, int64_t q_head_stride, const void *k,
                                          const void *v, int64_t kv_batch_stride, int64_t kv_tok_stride,
                                          int64_t kv_head_stride, const void *dout, int64_t o_row_stride,
                                          int64_t o_head_stride, const int64_t *offsets, void *dq, int64_t dq_row_stride,
                                          int64_t dq_head_stride, void *dk, void *dv, int64_t dkv_batch_stride,
                                          int64_t dkv_tok_stride, int64_t dkv_head_stride, float *workspace, int64_t L, int B,
                                          int h, int d, int n, int max_rows_per_sample, float scale, int dtype,
                                          void *stream);

/* offsets int64 [B+1] (device) = 0 and the running sums of the B lengths at lengths_host (HOST memory, read before the call
 * returns): the query counts of a batch as the reference's callers hold them, without a copy of host memory. */
int vtdge_lengths_to_offsets(const int64_t *lengths_host, int B, int64_t *offsets, void *stream);

/* out = act(LayerNorm(A) W^T + bias) for few rows, the LayerNorm done inside the Linear: norm1 -> kv and norm1 -> q
 * (vtpack/models/dge/deit_dge.py:127 with :72-73; the two products share the launch) or norm2 -> fc1 -> GELU (:128 with
 * :38-44) of a small batch.  LayerNorm(A) is rounded to the storage type before it is multiplied, as the two modules
 * would.
 *   A0 [rows0, K] leading dim lda0, W0 [N0, K], bias0 [N0] nullable, out0 [rows0, N0] dense, rows_dev0 nullable; the same
 *   for the second product with the same K and LayerNorm, absent with rows1 = 0
 * Taken where vtdge_layernorm_linear_fits says 1 (rows of whole 128-byte pieces and at most 1024 values, few tiles);
 * VTDGE_ERR_UNSUPPORTED otherwise.  vtdge_layernorm_linear_wanted: whether it is also the faster way. */
int vtdge_layernorm_linear_fits(int64_t rows0, int N0, int64_t rows1, int N1, int K, int dtype);
int vtdge_layernorm_linear_wanted(int64_t rows0, int N0, int64_t rows1, int N1, int K, int dtype);
int vtdge_layernorm_linear(const void *A0, int64_t lda0, const void *W0, const void *bias0, void *out0,
                           const int64_t *rows_dev0, int64_t rows0, int N0, const void *A1, int64_t lda1, const void *W1,
                           const void *bias1, void *out1, const int64_t *rows_dev1, int64_t rows1, int N1,
                           const void *ln_weight, const void *ln_bias, float ln_eps, int K, int act, int dtype,
                           void *stream);

/* out0 = A0 W0^T + bias0 and out1 = A1 W1^T + bias1 over the same K in one launch, for few rows: the key/value and the query
 * projection where the launch before them has written the LayerNorm of tokens and queries (vtdge_region_step).  Operands and
 * sizes as in vtdge_layernorm_linear; the bits of two vtdge_linear calls. */
int vtdge_linear_pair(const void *A0, int64_t lda0, const void *W0, const void *bias0, void *out0, const int64_t *rows_dev0,
                      int64_t rows0, int N0, const void *A1, int64_t lda1, const void *W1, const void *bias1, void *out1,
                      const int64_t *rows_dev1, int64_t rows1, int N1, int K, int dtype, void *stream);

/* What a block does with its packed queries behind attention (vtpack/models/dge/deit_dge.py:127-128 with :74-75 and
 * :38-44), as one kernel without the hidden rows in memory:
 *   q1 = o proj_weight^T + proj_bias + comp,   out = q1 + fc2(gelu(fc1(LayerNorm(q1))))
 * q1, LayerNorm(q1) and the hidden rows are rounded to the storage type as the modules would round them.
 *   o, comp, out  [rows, C] dense, out a buffer of its own; biases nullable, rows_dev nullable (device int64: the live rows)
 * Taken where vtdge_block_tail_fits says 1 (bf16, 64, 128 or 192 channels, hidden a multiple of 64 and at most 4096);
 * VTDGE_ERR_UNSUPPORTED otherwise.  vtdge_block_tail_wanted: whether it is also the faster way for that many rows. */
int vtdge_block_tail_fits(int64_t rows, int C, int hidden, int dtype);
int vtdge_block_tail_wanted(int64_t rows, int C, int hidden, int dtype);
int vtdge_block_tail(const void *o, const void *comp, const void *proj_weight, const void *proj_bias,
                     const void *ln_weight, const void *ln_bias, float ln_eps, const void *fc1_weight, const void *fc1_bias,
                     const void *fc2_weight, const void *fc2_bias, void *out, const int64_t *rows_dev, int64_t rows, int C,
                     int hidden, int dtype, void *stream);

/* A chain of DGE transformer blocks on one token grid (vtpack/models/dge/deit_dge.py:101-131 or pvt_dge.py:111-140,
 * `depth` of them in a row), issued by one host call: the launches are those of the entry points above
 * (vtdge_region_step and vtdge_linear_split_set among them), with nothing of the host between them.
 *   chain        what the blocks have in common.  H, W multiples of 4 and split sizes that divide 4 (`splits_124`: all
 *                of them out of {1, 2, 4}); head dim 32 or 64; sr > 1 only without extra tokens
 *   params_host  HOST table of device pointers, VTDGE_CHAIN_PARAMS per block, in this order (NULL where absent):
 *                norm1 weight, bias, norm2 weight, bias, router weight, bias, splits (int64); q weight, bias, kv weight,
 *                bias, proj weight, bias, fc1 weight, bias, fc2 weight, bias; packed copies (vtdge_linear_prepack, bf16;
 *                split copies of fp32 weights are made in `scratch`) of the q, kv, proj, fc1, fc2 weights; folded weight, column records (vtdge_layernorm_fold) and packed
 *                copy of the folded weight for norm1 -> q, norm1 -> kv, norm2 -> fc1; with sr > 1 the reduction's
 *                weight in [C, sr, sr, C] order, bias, and its norm's weight, bias.  The folded entries are needed
 *                where vtdge_chain_layout says so
 *   front_rows   nullable [extra, C]: stored as the extra tokens of every sample of x before anything reads them
 *   x            [B, extra + H*W, C], the first block's input; out: the last block's output, same shape
 *   ints, big, scratch   device buffers of the sizes vtdge_chain_layout returns, 256-byte aligned, nothing else using
 *                them until the call's work is done.  `scratch` may be reused as soon as later work on `stream` runs
 *   side_stream  nullable: a second stream for the routing half of every block where it helps; the call orders it
 *                against `stream` on both ends
 * vtdge_chain_layout fills layout_host[VTDGE_CHAIN_LAYOUT_HEAD + depth * VTDGE_CHAIN_LAYOUT_BLOCK]:
 *   [0..2] bytes of ints, big, scratch; [3] bytes of status words per block or 0; [4] 1 if folded weights are needed;
 *   then per block: offsets in `ints` of the gate logits, of offsets int64 [B+1], of lengths int64 [B] (-1: the
 *   differences of the offsets), of the status words of the scatter-back that packed the block (-1: none; word 0 stays
 *   0 unless it failed); offsets in `big` of its input tokens (-1: x itself), of its packed queries before and after
 *   the block [B * (extra + H*W), C], of its patch descriptors int64 [B * (extra + H*W), 4]. */
typedef struct {
    int32_t B, H, W, C, heads, hidden, extra, S, depth, dtype, sr, splits_124;
    float eps1, eps2, sr_eps, scale;
} vtdge_chain;
#define VTDGE_CHAIN_PARAMS 35
#define VTDGE_CHAIN_LAYOUT_HEAD 8
#define VTDGE_CHAIN_LAYOUT_BLOCK 8
int vtdge_chain_layout(const vtdge_chain *chain, int64_t *layout_host);
int vtdge_chain_forward(const vtdge_chain *chain, const void *const *params_host, const void *front_rows, void *x,
                        void *ints, void *big, void *scratch, void *out, void *stream, void *side_stream);

#ifdef __cplusplus
}
#endif
#endif /* VTDGE_H */
