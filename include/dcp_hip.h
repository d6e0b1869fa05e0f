/*
 * C ABI of libdcp_hip.so: the gfx950 kernels behind DCP's per-device blockwise
 * attention executor.
 *
 * Conventions
 *  - every pointer marked "device" is a HIP device address on the current
 *    device; "host" pointers are ordinary host memory read before return;
 *  - `stream` is a hipStream_t passed as void* (NULL = the null stream); all
 *    work is enqueued on it and nothing synchronises with the host;
 *  - the library borrows memory for the duration of a launch: it allocates
 *    nothing and keeps no pointer (a caller's own list of recorded calls
 *    aside, see dcp_record_begin);
 *  - return value 0 = launched, nonzero = rejected before any launch (argument
 *    error); dcp_last_error() then returns a message for the calling thread;
 *  - dtype codes follow the reference's wire integers
 *    (dcp/core/serialization.py:410-437): 0 bf16, 1 fp16, 2 fp32.
 *
 * Each entry point names the reference interface it replaces.
 */
#ifndef DCP_HIP_H_
#define DCP_HIP_H_

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define DCP_DTYPE_BF16 0
#define DCP_DTYPE_FP16 1
#define DCP_DTYPE_FP32 2

#define DCP_OK 0
#define DCP_ERR_ARG 1
#define DCP_ERR_UNSUPPORTED 2
#define DCP_ERR_LAUNCH 3

/* Library / ABI version (major*100 + minor). */
int dcp_version(void);

/* Message of the last nonzero return on this thread ("" if none). */
const char* dcp_last_error(void);

/*
 * Per-kernel timing for benchmarks (no counterpart in the reference, which
 * relies on external profilers).  While enabled, each kernel launch of this
 * library is bracketed by two events recorded on its launch stream.
 * dcp_profile_report waits for the recorded events, writes one line per kernel
 * name, "<name> <launches> <total_ms>\n", into `buffer` (NUL-terminated) and
 * forgets them; it returns nonzero if `capacity` was too small.  Disabled (the
 * default), launches record nothing.
 */
void dcp_profile_enable(int on);
int dcp_profile_report(char* buffer, size_t capacity);

/*
 * Recorded calls, for callers that repeat a fixed sequence (a prepared plan).
 * Between dcp_record_begin and dcp_record_end every call of an entry point
 * below that takes a stream, made on this thread, is launched as usual and also
 * added with its arguments to the list dcp_record_begin returned (NULL if the
 * thread is recording already, or host memory has run out; where it runs out
 * later, dcp_record_end says so and the list cannot be run).  dcp_record_run makes calls [begin, end) of a
 * list again, in order, on `stream`, and returns the first nonzero status.  The
 * arguments are kept as they were given: the caller keeps the memory they point
 * to alive and in place for as long as it runs the list.  A list may be run
 * from several threads; nothing in it changes.  No counterpart in the reference
 * (its executor walks the instructions in Python at every call).
 */
void* dcp_record_begin(void);
int dcp_record_end(void);
int dcp_record_size(const void* list);
int dcp_record_run(const void* list, int begin, int end, void* stream);
void dcp_record_free(void* list);

/*
 * Recorded calls of several lists on several streams, with the events between
 * them, in one call: what the plans of several devices that share a GPU come to.
 * Operation i launches calls [begin, end) of `list`, records `event` or makes
 * `stream` wait for it (hipEvent_t, hipStream_t); with on_caller nonzero the
 * operation's stream is the `stream` argument.  Stops at the first error.
 */
#define DCP_SEQUENCE_RUN 0
#define DCP_SEQUENCE_RECORD 1
#define DCP_SEQUENCE_WAIT 2
typedef struct {
  int32_t kind, begin, end, on_caller;
  const void* list;
  void* event;
  void* stream;
} dcp_sequence_op;
int dcp_sequence_run(const dcp_sequence_op* ops, int n_ops, void* stream);

/*
 * Block gather / scatter through pointer tables.
 * Replaces dcp.ops.fused_ops.fused_copy_{bf16,fp16,fp32}_varlen
 * (dcp/ops/fused_ops.py:842-864, 916-938, 1013-1035; kernels :290-335,
 * :472-517, :654-699), called from _handle_memcpy
 * (dcp/runtime/flash_attention/executor.py:793-805).
 *
 * For p in [0, n_ptrs), i in [0, n_elements[p]):
 *   ((T*)dst_ptrs[p])[dst_offsets[p]*dst_strides[p] + i] =
 *   ((T*)src_ptrs[p])[src_offsets[p]*src_strides[p] + i]
 * T has `elem_size` bytes (2 or 4); offsets/strides are in elements.
 * All seven tables are device int64/int32 arrays of length n_ptrs.
 * `block_numel` is the padded block size in elements (upper bound of
 * n_elements[p]); it only sizes the grid.
 */
int dcp_fused_copy_varlen(const int64_t* src_ptrs, const int32_t* src_offsets,
                          const int32_t* src_strides, const int64_t* dst_ptrs,
                          const int32_t* dst_offsets,
                          const int32_t* dst_strides,
                          const int32_t* n_elements, int n_ptrs,
                          int64_t block_numel, int elem_size, void* stream);

/*
 * Copy the first n_tokens[p] tokens (per_token_size elements each) of block p.
 * Replaces fused_copy_{bf16,fp16,fp32}_varlen_dkv (fused_ops.py:867-885,
 * 941-959, 1038-1056; kernel :338-367), used after the GQA backward
 * (executor.py:1102-1114).  src_ptrs/dst_ptrs address the blocks themselves.
 */
int dcp_fused_copy_varlen_dkv(const int64_t* src_ptrs, const int64_t* dst_ptrs,
                              const int32_t* n_tokens, int n_ptrs,
                              int max_n_tokens, int per_token_size,
                              int elem_size, void* stream);

/*
 * Head-strided copy of log-sum-exp blocks.
 * Replaces fused_copy_{bf16,fp16,fp32}_varlen_lse (fused_ops.py:888-913,
 * 962-987, 1059-1084; kernel :370-429), called from _handle_memcpy
 * (executor.py:806-810).
 * For h < head_block_size, t < n_tokens[p]:
 *   dst[p][h*dst_head_strides[p] + dst_token_offsets[p] + t] =
 *   src[p][h*src_head_strides[p] + src_token_offsets[p] + t]
 * Unlike the reference kernel, head_block_size need not be a power of two.
 */
int dcp_fused_copy_varlen_lse(const int64_t* src_ptrs,
                              const int32_t* src_token_offsets,
                              const int32_t* src_head_strides,
                              const int64_t* dst_ptrs,
                              const int32_t* dst_token_offsets,
                              const int32_t* dst_head_strides,
                              const int32_t* n_tokens, int n_ptrs,
                              int head_block_size, int max_n_tokens,
                              int elem_size, void* stream);

/*
 * N-way online-softmax merge of partial (out, lse) blocks, fused with the
 * scatter into the destination.
 * Replaces flash_attn_update_out_lse (fused_ops.py:149-247, kernel :15-146),
 * called from _handle_reduction (executor.py:1299-1329).
 *
 * For op o, head h < n_head, token t < n_tokens_per_block[o], over the
 * sources j < block_lengths[o] with block b_j = src_block_table[o*max_n+j]:
 *   l_j   = src_lse[h*src_lse_head_stride + b_j*lse_block_stride + t*lse_token_stride]
 *   sources with l_j = +-inf are ignored;
 *   lse*  = m + log(sum_j exp(l_j - m)),  m = max_j l_j
 *   out*  = sum_j exp(l_j - lse*) * src_out[b_j*out_block_stride + t*out_token_stride + h*head_dim + :]
 *   no finite source: lse* = -1, out* = 0.
 * dst_out[(dst_token_offsets[o]+t)*out_token_stride + h*head_dim + :] = out*
 * dst_lse[h*dst_lse_head_stride + (dst_token_offsets[o]+t)*lse_token_stride] = lse*
 * Math in fp32; out is stored in `dtype`, lse is fp32.  dst may alias one of
 * the sources of the same op (in-place fold).  max_n_blocks_per_op <= 64.
 */
int dcp_update_out_lse(const void* src_out, void* dst_out,
                       const float* src_lse, float* dst_lse, int n_head,
                       const int32_t* src_block_table,
                       const int32_t* dst_token_offsets,
                       const int32_t* n_tokens_per_block,
                       const int32_t* block_lengths, int n_red_ops,
                       int block_size, int64_t out_block_stride,
                       int64_t out_token_stride, int64_t lse_block_stride,
                       int64_t lse_token_stride, int64_t src_lse_head_stride,
                       int64_t dst_lse_head_stride, int head_dim,
                       int max_n_blocks_per_op, int dtype, void* stream);

/*
 * N-way block sum (dQ / dK / dV accumulation) fused with the scatter.
 * Replaces fused_blockwise_sum (fused_ops.py:1288-1360, kernels :1087-1285),
 * called from _handle_sum (executor.py:1530-1545).
 *   dst[s][dst_offsets[s]*dst_strides[s] + i] =
 *       sum_{j < n_ops_per_block[s]} src[s][src_offsets[s*max_n+j]*src_strides[s] + i]
 * for i < n_elements[s].  Accumulates in fp32 and rounds once (the reference
 * kernel accumulates in the storage type; see its test tolerance 1e-2).
 * dst may alias one of the sources of the same sum.
 */
int dcp_blockwise_sum(const int64_t* src_ptrs, const int32_t* src_offsets,
                      const int32_t* src_strides,
                      const int32_t* n_ops_per_block, const int64_t* dst_ptrs,
                      const int32_t* dst_offsets, const int32_t* dst_strides,
                      const int32_t* n_elements, int n_sums,
                      int max_n_ops_per_block, int64_t block_numel, int dtype,
                      void* stream);
/*
 * The same with fp32 sources whatever the destination's type `dtype`
 * (src_strides in fp32 elements): partial sums that have not been rounded yet,
 * as dcp_attn_bwd_grouped leaves them.  A single source is rounded.
 */
int dcp_blockwise_sum_fp32_sources(
    const int64_t* src_ptrs, const int32_t* src_offsets,
    const int32_t* src_strides, const int32_t* n_ops_per_block,
    const int64_t* dst_ptrs, const int32_t* dst_offsets,
    const int32_t* dst_strides, const int32_t* n_elements, int n_sums,
    int max_n_ops_per_block, int64_t block_numel, int dtype, void* stream);


/*
 * Range-masked, paged, variable-length attention forward.
 * Replaces dcp_flash_attn._flash_attn_varlen_forward as called by
 * _wrapped_flash_attn_varlen_forward (executor.py:117-187) from _handle_attn
 * (:884-913): no causal flag, no window, no dropout, no softcap.
 *
 * Batch row b = one q block.  Its seqlen_q = cu_seqlens_q[b+1]-cu_seqlens_q[b]
 * (<= block_size) queries live in slot q_block_table[b] of `q`
 * ([n_q_slots, block_size, n_heads_q, head_dim]); keys/values are the
 * concatenation of slots kv_block_table[b*max_kv_blocks + j] of `k`/`v`
 * (slot stride kv_slot_stride, token stride kv_token_stride, head stride
 * head_dim, in elements) for kv positions [0, cu_seqlens_kv[b+1]-cu_seqlens_kv[b]).
 * attn_range is int32 [n_ranges, 2, total_q]: query token t (global index
 * cu_seqlens_q[b]+i) attends kv positions in the union of
 * [attn_range[r][0][t], attn_range[r][1][t]).
 * (A range may begin before key 0 or end past the row's last key, at any value of
 * its type: the keys that there are count.  One that does not end past its start is empty.)
 * Writes out ([n_out_slots, block_size, n_heads_q, head_dim]) at slot
 * out_block_table[b] and lse (fp32 [n_heads_q, n_out_slots, block_size]) at the
 * same slot.  Rows with no visible key: out = 0, lse = +inf.
 * q head h reads kv head h / (n_heads_q / n_heads_kv).
 * row_order: optional device int32[batch], a permutation of the rows giving
 * the order in which they are scheduled (put the rows with most keys first);
 * NULL = as numbered.  It changes no result.
 * Supported: dtype bf16/fp16, head_dim 64 or 128, block_size % 64 == 0,
 * softmax_scale > 0.  (A caller with another head size up to 128 zero-pads its
 * buffers to the next of the two and keeps its own softmax_scale, as the
 * reference pads head sizes its kernels do not take; the Python operator layer
 * does so.)
 * Key/value tiles are loaded whole: what a slot holds past the row's keys (and,
 * for keys a range excludes, inside it) reaches the matrix instructions and is
 * masked there.  It must be finite, and small enough that its dot products with
 * q stay finite; the reference's kernels zero-fill such loads instead.  Query
 * rows past seqlen_q are not read.
 * `workspace`: caller-provided device scratch of
 * dcp_attn_fwd_workspace_bytes() bytes, 4-byte aligned, for the kernel's work
 * counters (the launch is persistent: its workgroups take (row, head, query
 * tile) items from per-XCD counters).  DCP_ATTN_FWD_MIN_WORKSPACE_BYTES are
 * enough; the counters then share a cache line, half a percent of a long
 * launch.  Its contents are overwritten (a small
 * kernel zeroes it on `stream` before the attention kernel); one workspace
 * serves any number of launches that follow each other on a stream or in a
 * captured graph, launches that may run at the same time need one each.
 */
#define DCP_ATTN_FWD_MIN_WORKSPACE_BYTES 64
size_t dcp_attn_fwd_workspace_bytes(void);
int dcp_attn_fwd(const void* q, const void* k, const void* v, void* out,
                 float* lse, const int32_t* cu_seqlens_q,
                 const int32_t* cu_seqlens_kv, const int32_t* attn_range,
                 int n_ranges, const int32_t* q_block_table,
                 const int32_t* kv_block_table,
                 const int32_t* out_block_table, const int32_t* row_order,
                 int batch, int max_kv_blocks, int total_q, int block_size,
                 int n_heads_q, int n_heads_kv, int head_dim,
                 int64_t kv_slot_stride, int64_t kv_token_stride,
                 int n_out_slots, float softmax_scale, int dtype,
                 void* workspace, size_t workspace_bytes, void* stream);

/*
 * dcp_attn_fwd with the stride of a table entry spelled out per tensor, so that
 * the tables can address the caller's UNPADDED tensors directly instead of
 * padded slots: entry e of q_block_table places the row's first query at
 * q + e*q_slot_stride (elements), entry e of out_block_table its first output
 * at out + e*out_slot_stride and its first LSE at
 * lse + head*lse_head_stride + e*lse_slot_stride; queries of a row are
 * n_heads_q*head_dim elements apart, their LSEs 1.  With
 *   q_slot_stride = out_slot_stride = block_size*n_heads_q*head_dim,
 *   lse_head_stride = n_out_slots*block_size, lse_slot_stride = block_size
 * this is dcp_attn_fwd.  With q_slot_stride = out_slot_stride =
 * n_heads_q*head_dim, lse_head_stride = tokens of the LSE tensor,
 * lse_slot_stride = 1 and kv_slot_stride = kv_token_stride, every table entry
 * is a TOKEN offset into [tokens, heads, head_dim] tensors (LSE:
 * [n_heads_q, tokens]): what the reference's plans spell out as a gather into
 * slots before the kernel (MemcpyInstr, executor.py:793-811) and a
 * single-source scatter after it (executor.py:1269-1329) then needs no copy.
 * Only the row's seqlen_q queries are read and written; key/value tiles are
 * still loaded whole, block_size keys from every table entry on, so the k/v
 * tensors must be readable (and finite) for block_size tokens past their last
 * block's first token.  merged_form != 0: a query without a visible key gets
 * lse = -1 instead of +inf (out = 0 either way), which is what the reference's
 * merge kernel leaves for a row none of whose sources is finite
 * (fused_ops.py:118-143) -- for outputs written where that merge would have
 * put them.  No counterpart in the reference.
 */
int dcp_attn_fwd_strided(const void* q, const void* k, const void* v, void* out,
                         float* lse, const int32_t* cu_seqlens_q,
                         const int32_t* cu_seqlens_kv,
                         const int32_t* attn_range, int n_ranges,
                         const int32_t* q_block_table,
                         const int32_t* kv_block_table,
                         const int32_t* out_block_table,
                         const int32_t* row_order, int batch,
                         int max_kv_blocks, int total_q, int block_size,
                         int n_heads_q, int n_heads_kv, int head_dim,
                         int64_t kv_slot_stride, int64_t kv_token_stride,
                         int64_t q_slot_stride, int64_t out_slot_stride,
                         int64_t lse_head_stride, int64_t lse_slot_stride,
                         int merged_form, float softmax_scale, int dtype,
                         void* workspace, size_t workspace_bytes, void* stream);

/*
 * dcp_attn_fwd_strided for launches of few, uneven rows: rows may be split along
 * their keys, so that the launch does not last as long as its longest row.
 * `parts` ([n_entries][4] int32: row, part, number of parts n, first partial)
 * takes the place of row_order: an entry computes an equal share of the key tiles
 * of every (head, query tile) of its row; every row appears with parts 0..n-1.
 * Entries with n = 1 write out and lse.  The others leave fp32 sums in partial
 * `first partial` + part of `partials` (16-byte aligned, n_partials *
 * ceil(block_size / 128) * 128 * n_heads_q * (head_dim + 2) floats, contents
 * overwritten; partials of a launch are not shared), and a second kernel adds
 * the parts of the rows that `splits` lists ([n_splits][4]: row, n, first
 * partial, 0) and rounds once.  No counterpart in the reference.
 */
int dcp_attn_fwd_parts(const void* q, const void* k, const void* v, void* out,
                       float* lse, const int32_t* cu_seqlens_q,
                       const int32_t* cu_seqlens_kv, const int32_t* attn_range,
                       int n_ranges, const int32_t* q_block_table,
                       const int32_t* kv_block_table,
                       const int32_t* out_block_table,
                       const int32_t* row_order, int batch, int max_kv_blocks,
                       int total_q, int block_size, int n_heads_q,
                       int n_heads_kv, int head_dim, int64_t kv_slot_stride,
                       int64_t kv_token_stride, int64_t q_slot_stride,
                       int64_t out_slot_stride, int64_t lse_head_stride,
                       int64_t lse_slot_stride, int merged_form,
                       float softmax_scale, int dtype, void* workspace,
                       size_t workspace_bytes, const int32_t* parts,
                       int n_entries, const int32_t* splits, int n_splits,
                       int n_partials, void* partials, size_t partials_bytes,
                       void* stream);

/*
 * The same from a table of the work items there are, one per 128 queries of a row
 * (or of a row's part):
 *   items int32 [n_items][4], 16-byte aligned: a row; which 128 of its queries; part +
 *     65536 * number of parts (65536 where the row is not split); first partial
 * Every (row with queries, 128 of its queries, part) once, taken in this order and
 * dealt to the XCDs in turn.  row_order is not read.  Tiles of a block for which a row
 * has no queries are not listed, and cost nothing.  items null (and n_items and
 * n_splits 0): all tiles of the rows, as dcp_attn_fwd_strided.
 *   one_each: nonzero = a workgroup for every item from the start (the workspace is then
 *     not written, but must be there all the same); 0 = as many as the device holds at
 *     once, which take item after item.
 */
int dcp_attn_fwd_items(const void* q, const void* k, const void* v, void* out,
                       float* lse, const int32_t* cu_seqlens_q,
                       const int32_t* cu_seqlens_kv, const int32_t* attn_range,
                       int n_ranges, const int32_t* q_block_table,
                       const int32_t* kv_block_table,
                       const int32_t* out_block_table,
                       const int32_t* row_order, int batch, int max_kv_blocks,
                       int total_q, int block_size, int n_heads_q,
                       int n_heads_kv, int head_dim, int64_t kv_slot_stride,
                       int64_t kv_token_stride, int64_t q_slot_stride,
                       int64_t out_slot_stride, int64_t lse_head_stride,
                       int64_t lse_slot_stride, int merged_form,
                       float softmax_scale, int dtype, void* workspace,
                       size_t workspace_bytes, const int32_t* items, int n_items, int one_each, const int32_t* splits, int n_splits,
                       int n_partials, void* partials, size_t partials_bytes,
                       void* stream);

/*
 * Range-masked, paged, variable-length attention backward.
 * Replaces dcp_flash_attn._flash_attn_varlen_backward as called by
 * _wrapped_flash_attn_varlen_backward (executor.py:256-337) from
 * _handle_attn_bw (:1058-1115).
 *
 * Inputs as dcp_attn_fwd plus dout/out (slots out_block_table[b]) and lse.
 * dq ([n_dq_slots, block_size, n_heads_q, head_dim]) slot dq_block_table[b]
 * receives the row's dQ.  dk/dv: slot dkv_block_table[b*max_kv_blocks + j]
 * receives the dK/dV of the row's j-th kv block, summed over the q heads of
 * each kv head's group.  The kv positions of the row below its key count
 * (cu_seqlens_kv[b+1]-cu_seqlens_kv[b]) rounded up to 32 are written, all heads
 * and dims, with 0 where no query of the row attends; positions past that keep
 * what the slot held.  A key count that is a multiple of block_size, as every
 * plan has it, therefore needs no pre-zeroing.  No atomics are used: results
 * are bit-reproducible from run to run.
 * `workspace` is caller-provided device scratch of at least
 * dcp_attn_bwd_workspace_bytes(...) bytes, 16-byte aligned; its contents are
 * overwritten.  Slot padding (q/dout/out rows past seqlen_q inside a 64-row
 * tile, k/v rows past the row's keys) is loaded and masked, not skipped: it
 * must be finite and small enough that its dot products with the data stay
 * finite.
 */
int dcp_attn_bwd(const void* dout, const void* q, const void* k, const void* v,
                 const void* out, const float* lse, void* dq, void* dk,
                 void* dv, void* workspace, size_t workspace_bytes,
                 const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_kv,
                 const int32_t* attn_range, int n_ranges,
                 const int32_t* q_block_table, const int32_t* kv_block_table,
                 const int32_t* out_block_table,
                 const int32_t* dq_block_table,
                 const int32_t* dkv_block_table, const int32_t* row_order,
                 int batch, int max_kv_blocks, int total_q, int block_size,
                 int n_heads_q, int n_heads_kv, int head_dim,
                 int64_t kv_slot_stride, int64_t kv_token_stride,
                 int64_t dkv_slot_stride, int64_t dkv_token_stride,
                 int n_out_slots, float softmax_scale, int dtype,
                 void* stream);

/*
 * dcp_attn_bwd with the stride of a table entry spelled out per tensor (see
 * dcp_attn_fwd_strided) and with total_kv, the sum of the rows' key counts
 * (cu_seqlens_kv[batch], which the host side of the call cannot read; 0 = not
 * known, which rules DCP_BWD_THROUGH_DS out): q_slot_stride for q, out_slot_stride for out AND dout
 * (they share out_block_table), dq_slot_stride for dq, lse_head_stride /
 * lse_slot_stride for lse.  With token strides the tables address the caller's
 * unpadded q, out, dout, lse, k and v directly and dQ is written straight into
 * the unpadded dq.  The dK/dV kernel loads whole 64-query tiles of q and dout:
 * those tensors must be readable (and finite) for 64 tokens past the last
 * row's queries.  dk/dv stay padded slots (a row writes whole 32-key groups).
 * No counterpart in the reference.
 */
int dcp_attn_bwd_strided(const void* dout, const void* q, const void* k,
                         const void* v, const void* out, const float* lse,
                         void* dq, void* dk, void* dv, void* workspace,
                         size_t workspace_bytes, const int32_t* cu_seqlens_q,
                         const int32_t* cu_seqlens_kv,
                         const int32_t* attn_range, int n_ranges,
                         const int32_t* q_block_table,
                         const int32_t* kv_block_table,
                         const int32_t* out_block_table,
                         const int32_t* dq_block_table,
                         const int32_t* dkv_block_table,
                         const int32_t* row_order, int batch, int max_kv_blocks,
                         int total_q, int block_size, int n_heads_q,
                         int n_heads_kv, int head_dim, int64_t kv_slot_stride,
                         int64_t kv_token_stride, int64_t dkv_slot_stride,
                         int64_t dkv_token_stride, int64_t q_slot_stride,
                         int64_t out_slot_stride, int64_t dq_slot_stride,
                         int64_t lse_head_stride, int64_t lse_slot_stride,
                         int64_t total_kv, float softmax_scale, int dtype,
                         void* stream);

/*
 * dcp_attn_bwd_strided that adds dK/dV of a kv block over several rows in the
 * kernel, in fp32, instead of leaving one private dK/dV block per (row, kv
 * block), or splits the work of one over several workgroups.  A group is a kv
 * block with up to DCP_ATTN_BWD_MAX_VISITS of the rows that list it, or a part
 * of the queries of these rows:
 *   dkv_groups int32 [n_groups][8]: the block's k/v table entry; where its dK/dV
 *     goes (an entry); tokens to store; which memory that is: 0 = dk/dv (a
 *     slot), 1 = dk_unpadded/dv_unpadded (entry and token strides in elements),
 *     2 = partials, fp32 [..][block_size][dK, dV][n_heads_kv][head_dim]; the
 *     first of its visits; their number; the part's q heads of each kv head's
 *     (begin + 65536 * end, 0 = all of them); the part's 64-query tiles (number
 *     of parts + 65536 * part: every so many tiles, 0 = all of them)
 *   dkv_visits int32 [..][2]: a row, and the position of the group's block in
 *     the row's kv_block_table
 * Every (query, row, position) with keys belongs to exactly one group (a plan's
 * replicas that are not added up form groups of one); dkv_block_table is
 * not read.  block_size must be a multiple of 128; a row's last block may be
 * partly filled (its key count need not be a multiple).  A group's tokens are
 * written whole (zeros where no query attends).  Launch order of the groups:
 * as listed, so the ones with the most visits should come first.  The one-pass
 * backward has no such form (the two-kernel one runs where it is selected).
 * No counterpart in the reference, which sums replicas with a SumInstr
 * (dcp/core/scheduler.py:1764-1940).
 */
#define DCP_ATTN_BWD_MAX_VISITS 32
int dcp_attn_bwd_grouped(const void* dout, const void* q, const void* k,
                         const void* v, const void* out, const float* lse,
                         void* dq, void* dk, void* dv, void* workspace,
                         size_t workspace_bytes, const int32_t* cu_seqlens_q,
                         const int32_t* cu_seqlens_kv,
                         const int32_t* attn_range, int n_ranges,
                         const int32_t* q_block_table,
                         const int32_t* kv_block_table,
                         const int32_t* out_block_table,
                         const int32_t* dq_block_table,
                         const int32_t* dkv_block_table,
                         const int32_t* row_order, int batch, int max_kv_blocks,
                         int total_q, int block_size, int n_heads_q,
                         int n_heads_kv, int head_dim, int64_t kv_slot_stride,
                         int64_t kv_token_stride, int64_t dkv_slot_stride,
                         int64_t dkv_token_stride, int64_t q_slot_stride,
                         int64_t out_slot_stride, int64_t dq_slot_stride,
                         int64_t lse_head_stride, int64_t lse_slot_stride,
                         int64_t total_kv, const int32_t* dkv_groups,
                         int n_groups, const int32_t* dkv_visits,
                         void* dk_unpadded, void* dv_unpadded,
                         int64_t unpadded_entry_stride,
                         int64_t unpadded_token_stride, float* partials,
                         float softmax_scale, int dtype, void* stream);

/*
 * Bytes of scratch dcp_attn_bwd needs for these sizes: rowsum(dO*O) and the
 * base-2 log-sum-exp (total_q*n_heads_q floats each), the per-(row, 64-query
 * tile) range hulls and the dQ kernel's work counters.  No counterpart in the reference (its
 * flash-attention fork allocates these inside the call).
 */
size_t dcp_attn_bwd_workspace_bytes(int batch, int total_q, int block_size,
                                    int n_heads_q, int head_dim);

/*
 * Which of its implementations the backward takes from now on (a setting of the
 * process; DCP_BWD_MODE=0/1/2 in the environment presets it).  All three are
 * free of atomics and bit-reproducible.
 *  DCP_BWD_TWO_KERNELS  a query-outer kernel for dQ and a key-outer one for
 *      dK/dV, each recomputing S and dP: seven matrix products for the
 *      backward's five, nothing but the small workspace.
 *  DCP_BWD_ONE_PASS  one key-outer pass (head size 128 only) in which the key
 *      tiles of a row add their shares of dQ one after the other through an
 *      fp32 partial sum in the workspace: five products.  Measured SLOWER on
 *      MI355X (18 ms against 12.5 ms on 65536 causal tokens) and kept as the
 *      measured alternative; only taken on a device on which the workgroups of
 *      a row share an L2 (the library checks).
 *  DCP_BWD_THROUGH_DS  (the default) the key-outer kernel also stores dS, 2 bytes
 *      per (query, key) pair and head of every tile pair it visits, and the dQ
 *      kernel reads it back instead of recomputing it: five products, paid for
 *      with HBM traffic and workspace (4 KiB per 64 keys x 32 queries x head:
 *      21 GB on 65536 causal tokens with 32 heads).  Only
 *      dcp_attn_bwd_strided, which is told total_kv, can take it.
 * A mode whose workspace the caller did not provide (see
 * dcp_attn_bwd_workspace_bytes_kv) or whose conditions do not hold falls back
 * to DCP_BWD_TWO_KERNELS.  Returns the previous setting; any other argument
 * only asks.  No counterpart in the reference, whose backward is one
 * non-deterministic pass with atomic adds
 * (dcp/runtime/flash_attention/executor.py:292-334).
 */
#define DCP_BWD_TWO_KERNELS 0
#define DCP_BWD_ONE_PASS 1
#define DCP_BWD_THROUGH_DS 2
int dcp_attn_bwd_select(int mode);

/*
 * Bytes of workspace the SELECTED backward needs for these sizes, total_kv =
 * the sum of the rows' key counts (cu_seqlens_kv[batch]); what
 * dcp_attn_bwd_workspace_bytes reports plus, for DCP_BWD_THROUGH_DS, the dS
 * pieces, and for DCP_BWD_ONE_PASS the partial sums and chain counters.
 */
size_t dcp_attn_bwd_workspace_bytes_kv(int batch, int total_q, int64_t total_kv,
                                       int block_size, int n_heads_q,
                                       int head_dim);

/*
 * dcp_attn_bwd for callers that cannot allocate device memory or carry a
 * workspace (code under HIP graph capture, tight serving loops, harnesses that
 * forbid hipMalloc).  No counterpart in the reference.  Same arguments, results
 * and errors as dcp_attn_bwd without `workspace`/`workspace_bytes`: the scratch
 * is a static device array inside the library, DCP_ATTN_BWD_STATIC_SCRATCH_BYTES
 * long, which every GPU the library runs on holds until the process ends.  Its
 * address on a device is looked up once, by the first of
 * dcp_attn_bwd_static_scratch_bytes() or dcp_attn_bwd_static() called with that
 * device current: a caller that records dcp_attn_bwd_static into a HIP graph
 * calls dcp_attn_bwd_static_scratch_bytes() once per device beforehand, outside
 * the capture, and the recorded call then makes no runtime query.  The call
 * allocates and frees nothing.  Sizes for which dcp_attn_bwd_workspace_bytes(...) exceeds the
 * scratch are rejected with DCP_ERR_ARG.  All calls on one GPU share the one
 * array: calls that may overlap on that GPU (different streams, or graphs
 * replayed side by side) race; calls that follow each other on a stream do not.
 */
#define DCP_ATTN_BWD_STATIC_SCRATCH_BYTES (32u << 20)
size_t dcp_attn_bwd_static_scratch_bytes(void);
int dcp_attn_bwd_static(const void* dout, const void* q, const void* k,
                        const void* v, const void* out, const float* lse,
                        void* dq, void* dk, void* dv,
                        const int32_t* cu_seqlens_q,
                        const int32_t* cu_seqlens_kv,
                        const int32_t* attn_range, int n_ranges,
                        const int32_t* q_block_table,
                        const int32_t* kv_block_table,
                        const int32_t* out_block_table,
                        const int32_t* dq_block_table,
                        const int32_t* dkv_block_table,
                        const int32_t* row_order, int batch, int max_kv_blocks,
                        int total_q, int block_size, int n_heads_q,
                        int n_heads_kv, int head_dim, int64_t kv_slot_stride,
                        int64_t kv_token_stride, int64_t dkv_slot_stride,
                        int64_t dkv_token_stride, int n_out_slots,
                        float softmax_scale, int dtype, void* stream);

/*
 * Stage packer of the planner (host code, no GPU work, `stream`-less): decides
 * which attention blocks ("workloads") every device may run in pipeline stage
 * `stage_id` and which data blocks must be sent to it first, under a cap on the
 * bytes each device sends to other nodes in the stage.
 * Replaces dcp_cpp.greedy_selection_per_device
 * (csrc/pipeline_generator/pipeline_generator.cpp:19-323, bound in
 * csrc/interface.cpp:9-11, called from dcp/core/pipeline.py:651-666,703-716).
 * The reference's sets and dicts of (node, rank) tuples become dense tables;
 * all pointers are HOST memory:
 *   device_node[d]               node of device d (devices are 0..n_devices-1)
 *   workload_costs[w], workload_scheduled[w] (nonzero: already placed in an
 *                                earlier stage, i.e. the reference's
 *                                `scheduled_workloads` set)
 *   input_sizes[i], input_kind[i]  size and DCP_BLOCK_* kind of data block i
 *                                (the reference's input_block_type_map strings
 *                                "OUT" / "LSE" / "dOUT", anything else OTHER)
 *   workload_input_offsets/workload_inputs   CSR of workload_input_map
 *   device_workload_offsets/device_workloads CSR of device_workload_map
 *   held_since[d * n_inputs + i] in/out: the stage since which device d holds
 *                                block i (-1 = from the start), DCP_NOT_HELD if
 *                                it does not (device_local_inputs_map; updated
 *                                in place = the third element of the result)
 *   target_cross_node_load[d]    target_comm_load_per_node
 * Results: unlocked_by[w] = device that may now run workload w, or -1 (first
 * element of the reference's result); the transfers (comm_dst[k], comm_input[k],
 * comm_src[k]) for k < *n_comm in the order they were decided (second element;
 * n_devices * n_inputs entries always suffice -- on a nonzero return because
 * `comm_capacity` was too small, *n_comm holds the needed count and held_since
 * has been modified: call again from the original table); optionally each
 * device's outgoing cross-node and same-node bytes (what the reference logs).
 * Where the reference's choice depends on the iteration order of a hash table
 * (equal compute times, equal sender loads, equal costs) the lowest device
 * index / workload id wins.
 */
#define DCP_BLOCK_OTHER 0
#define DCP_BLOCK_OUT 1
#define DCP_BLOCK_LSE 2
#define DCP_BLOCK_DOUT 3
#define DCP_NOT_HELD INT32_MIN
int dcp_greedy_stage_selection(
    int n_devices, const int32_t* device_node, int n_workloads,
    const float* workload_costs, const uint8_t* workload_scheduled,
    int n_inputs, const float* input_sizes, const uint8_t* input_kind,
    const int32_t* workload_input_offsets, const int32_t* workload_inputs,
    const int32_t* device_workload_offsets, const int32_t* device_workloads,
    int32_t* held_since, const float* target_cross_node_load, int is_bw,
    int stage_id, int32_t* unlocked_by, int32_t* comm_dst, int32_t* comm_input,
    int32_t* comm_src, int64_t comm_capacity, int64_t* n_comm,
    float* cross_node_load_out, float* intra_node_load_out);

#ifdef __cplusplus
}
#endif
#endif /* DCP_HIP_H_ */
