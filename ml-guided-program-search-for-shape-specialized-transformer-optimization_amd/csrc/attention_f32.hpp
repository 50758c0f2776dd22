// The fp32 causal attention's parameters and launch (attention_f32.hip).
#pragma once

#include "sah_common.hpp"

namespace sah {

// head_dim 64; Q, K, V [B, H, S, 64] with 16-byte aligned rows (element
// strides, multiples of 4), O [B, S, H * 64].
struct AttnF32Params {
  const float* q;
  const float* k;
  const float* v;
  float* o;
  int64_t q_sb, q_sh, q_ss;
  int64_t k_sb, k_sh, k_ss;
  int64_t v_sb, v_sh, v_ss;
  int64_t o_sb, o_ss;
  int seq_len;
  int heads;
  float c;      // |scale| log2(e), > 0
  float floor;  // set by the launch: the lowest shift, whose product with c is finite
  uint32_t q_and, q_xor;  // the sign of the scale (or a zero scale), on Q
};

int launch_attention_f32(AttnF32Params p, int batch, hipStream_t stream);

}  // namespace sah
