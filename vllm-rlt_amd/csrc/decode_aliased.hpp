// Decode of rows that read each other's pages (paged_decode.hip): a prefill's
// rows on the per-token path.
#pragma once

#include <cstdint>

namespace rlt {

// rlt_paged_decode with its contract and bits; workgroups are dealt out for
// rows whose neighbours read the same pages.
int paged_decode_aliased(const void* q, const int64_t* q_strides, const void* key_cache, const void* value_cache,
                         const int64_t* kv_strides, const int32_t* block_tables, int64_t table_stride,
                         int64_t max_table_width, const int32_t* context_lengths, void* out,
                         const int64_t* out_strides, int64_t n_rows, int64_t num_q_heads, int64_t num_kv_heads,
                         int64_t head_dim, int64_t page_size, int64_t num_blocks, float scale, int dtype,
                         void* workspace, int64_t workspace_bytes, void* stream);

}  // namespace rlt
