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

// mxfa_split_decode_multi_launch (same arguments, checks and results) for up
// to mxfa_package_launch_columns columns: every 16 columns past the first are
// another column group of the same wave, so the keys are read once for all.
// With num_splits = MXFA_SPLITS_PER_SEQUENCE at most 16 columns.
int mxfa_package_decode_tokens_launch(
    const void *q, int64_t q_stride_b, int64_t q_stride_t, int64_t q_stride_h, int q_len,
    int causal, int window_left, const float *sinks, float softcap, const float *alibi_slopes,
    const void *k_cache, const void *v_cache, int64_t cache_stride_page,
    int64_t cache_stride_token, int64_t cache_stride_head, const int32_t *block_table,
    int64_t bt_stride, const int32_t *seqlens, int seqlen_add, void *out, int64_t out_stride_b,
    int64_t out_stride_t, int64_t out_stride_h, void *workspace, size_t workspace_bytes,
    float scale, int batch, int q_heads, int kv_heads, int head_dim, int page_size,
    int block_table_width, int num_pages, int dtype, int kv_dtype, const float *k_scale,
    const float *v_scale, int num_splits, void *stream);

#ifdef __cplusplus
}
#endif
