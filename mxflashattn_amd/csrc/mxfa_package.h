// Entry points of the library for this package's own bindings (native.py and
// the torch operator). They are not part of the C ABI (include/mxfa_mi355x.h):
// names, arguments and limits may change with the package, which always loads
// the library it was built with.
#pragma once

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

// Columns (query tokens x query heads per kv head) that one launch of
// mxfa_package_decode_tokens_launch takes. extras: the call has a window, soft
// cap, sinks or ALiBi.
int mxfa_package_launch_columns(int head_dim, int page_size, int fp8, int extras);

// Query tokens of each launch of a call of q_len tokens when a launch takes
// `columns`: as many as fit, or, of launches of several column groups, about
// equal shares (64 columns at head dim 128 are two launches of two groups rather
// than one of three and one of one).
int mxfa_package_tokens_per_launch(int q_len, int gq, int columns);

// num_splits for a call of q_len tokens whose launches take `columns`: the
// heuristic's choice for the columns of one launch of one group, or, where that
// is the split kernel and launches are of several groups, for one of those.
int mxfa_package_num_splits(int batch, int q_len, int q_heads, int kv_heads, int head_dim,
                            int page_size, int block_table_width, int fp8, int columns,
                            int num_cus, int *num_splits);

// mxfa_split_decode_multi_launch (same arguments, checks and results) for up
// to mxfa_package_launch_columns columns: every 16 columns past the first are
// another column group of the same wave, so the keys are read once for all.
// With num_splits = MXFA_SPLITS_PER_SEQUENCE at most 16 columns. advance (int32
// [batch], or null) is moved on by advance_by once the call has read the
// lengths; it may be seqlens itself.
int mxfa_package_decode_tokens_launch(
    const void *q, int64_t q_stride_b, int64_t q_stride_t, int64_t q_stride_h, int q_len,
    int causal, int window_left, const float *sinks, float softcap, const float *alibi_slopes,
    const void *k_cache, const void *v_cache, int64_t cache_stride_page,
    int64_t cache_stride_token, int64_t cache_stride_head, const int32_t *block_table,
    int64_t bt_stride, const int32_t *seqlens, int seqlen_add, void *out, int64_t out_stride_b,
    int64_t out_stride_t, int64_t out_stride_h, void *workspace, size_t workspace_bytes,
    float scale, int batch, int q_heads, int kv_heads, int head_dim, int page_size,
    int block_table_width, int num_pages, int dtype, int kv_dtype, const float *k_scale,
    const float *v_scale, int num_splits, int32_t *advance, int advance_by, void *stream);

// Decode over keys that lie in consecutive rows, read in place (16-bit caches):
// k and v rows of kv head h at first_stride * first(b) + token_stride * i +
// head_stride * h elements for token i of sequence b.
//   dense (cu_seqlens_k null): first(b) = b (first_stride: the batch stride;
//     num_firsts: the batch dimension of k), max_len keys each, or
//     seqlens[b] + seqlen_add (at most max_len);
//   packed (cu_seqlens_q, cu_seqlens_k of num_seqs + 1 offsets, int32 or
//     int64): the query rows are the sequences with cu_q[i + 1] > cu_q[i], in
//     order; first_stride = token_stride, num_firsts the total of key rows.
//     host_offsets (2 * (num_seqs + 1) int64 in host memory that the device can
//     write, or null) receives cu_q then cu_k; offsets_event (a hipEvent_t, or
//     null) is recorded once they are there, ahead of the decode.
// rows (2 * batch int32 in device memory): one small launch writes first rows
// and lengths there (unless rows_written: an earlier launch of the same call
// did), and the decode reads them. First rows and lengths are held to the rows
// that exist where they are written, so nothing else (a replay of a graph that
// holds this memory) may write them before the decode has read them.
// page_size: of the pages that hold the same bytes (1 for packed keys). With
// ranges (num_splits > 0) that their heuristic chooses, one launch gives the bits
// of those pages; the per-sequence kernel, which pages of less than a tile do not
// take, gives their error against 64 bits or less.
// q_len query tokens of at most mxfa_package_launch_columns(head_dim, 16, 0, 0)
// columns; mxfa_package_contiguous_workspace_size is the workspace of the widest
// launch of a call of q_len tokens (0 for MXFA_SPLITS_PER_SEQUENCE).
int mxfa_package_contiguous_workspace_size(int batch, int q_heads, int kv_heads, int q_len,
                                           int head_dim, int num_splits, size_t *bytes);
int mxfa_package_contiguous_decode_launch(
    const void *q, int64_t q_stride_b, int64_t q_stride_t, int64_t q_stride_h, int q_len,
    int causal, const void *k, const void *v, int64_t first_stride, int64_t token_stride,
    int64_t head_stride, int64_t num_firsts, int max_len, const void *cu_seqlens_q,
    int cu_q_is_int64, const void *cu_seqlens_k, int cu_k_is_int64, int num_seqs,
    int32_t *rows, int rows_written, int64_t *host_offsets, void *offsets_event,
    const int32_t *seqlens, int seqlen_add, void *out, int64_t out_stride_b, int64_t out_stride_t,
    int64_t out_stride_h, void *workspace, size_t workspace_bytes, float scale, int batch,
    int q_heads, int kv_heads, int head_dim, int page_size, int dtype, int num_splits,
    void *stream);

#ifdef __cplusplus
}
#endif
