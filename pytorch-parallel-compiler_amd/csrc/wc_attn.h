// Internal interface of the attention kernels.
#pragma once

#include "wc_common.h"

namespace wc {

struct AttnParams {
  int nb, heads, sq, skv, causal, q_tiles;
  float scale_log2;
  const void* q;
  int64_t q_sb, q_ss;
  const void* k;
  int64_t k_sb, k_ss;
  const void* v;
  int64_t v_sb, v_ss;
  void* o;
  int64_t o_sb, o_ss;
  // additive fp32 mask, element (nb, head, query, key) at nb*m_sb + head*m_sh + query*m_sq + key
  // (general kernel only; NULL = none)
  const float* mask;
  int64_t m_sb, m_sh, m_sq;
  // head dims other than the kernel's own (attn_kernel with GEN): the true head dim, and the
  // first head-dim column of the output chunk this launch computes
  int dh, oc0;
};

// The streaming 16-bit kernel (attention_stream.hip): head dims that are a multiple of 8 up to
// 128, 16-byte aligned rows, no mask, positive scale; 1 when it does not take the problem
// (nothing launched).
template <typename T>
int32_t attn_stream(const AttnParams& p, hipStream_t st);

}  // namespace wc
