// The fp32 prefill launch (paged_prefill_f32.hip), chosen by rlt_paged_prefill.
#pragma once

#include "common.hpp"

namespace rlt {

struct PrefillF32Args {
  const float* q;
  int64_t q_row, q_head;  // elements, all strides
  const float* k;
  const float* v;
  int64_t kv_block, kv_token, kv_head;
  const int32_t* tables;
  int64_t table_stride, width;
  const int32_t* lens;
  const int32_t* cu;
  float* out;
  int64_t o_row, o_head;
  int num_seqs, hq, hkv;
  int64_t num_blocks;
  int total_q;
  float qscale;  // |scale| * log2(e)
  int negate;    // a negative scale: q's sign flips
};

// head_dim 128, page 16, unit dim strides and 16-byte rows; total_q and
// num_seqs positive and below 2^31.
int launch_prefill_f32(const PrefillF32Args& a, hipStream_t stream);

}  // namespace rlt
