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

// ---- shared by the streaming kernels ----
constexpr int kStBK = 64;              // keys per tile

// DHP: the head dim rounded up to a multiple of 32 (columns past p.dh are zero in LDS).
// Bank conflicts: K's 16-byte chunks are permuted within a row so that 16 rows' reads of one
// chunk index cover the 64 banks; V's 64-byte blocks so that 4 consecutive rows' do.
template <int DHP>
__device__ __forceinline__ int k_at(int row, int c) {          // element offset of chunk c
  if constexpr (DHP == 32) c ^= (row >> 1) & 3;
  else if constexpr (DHP == 64) c ^= (row >> 1) & 7;
  else if constexpr (DHP == 96) c ^= (row >> 2) & 3;
  else c ^= row & 15;
  return row * DHP + c * 8;
}
template <int DHP>
__device__ __forceinline__ int v_at(int row, int col) {
  if constexpr (DHP == 64) col ^= ((row >> 1) & 1) << 5;
  else if constexpr (DHP == 128) col ^= (row & 3) << 5;
  return row * DHP + col;
}

// workgroup -> (head, query tile).  XCD x takes every head in [x, x + 1) * heads / 8, whose K
// and V then stay in its L2.  Causal tiles differ in length: the longest of all its heads come
// first, and every second round of one workgroup per CU runs backwards, so that a CU that
// started with a long tile goes on with a short one.
template <bool CAUSAL>
__device__ __forceinline__ void stream_tile(const AttnParams& p, int& bh, int& qt) {
  const int bhs = p.nb * p.heads;
  int heads = bhs, i = blockIdx.x, h0 = 0, cus = 256;
  if ((bhs & 7) == 0) {
    heads = bhs >> 3;
    h0 = (blockIdx.x & 7) * heads;
    i = blockIdx.x >> 3;
    cus = 32;
  }
  if (CAUSAL) {
    const int round = i / cus;
    if ((round & 1) && (round + 1) * cus <= heads * p.q_tiles) i = round * cus + cus - 1 - (i - round * cus);
    const int t = i / heads;
    qt = p.q_tiles - 1 - t;
    bh = h0 + i - t * heads;
  } else {
    bh = h0 + i / p.q_tiles;
    qt = i % p.q_tiles;
  }
}

// The streaming 16-bit kernel (attention_stream.hip): head dims that are a multiple of 8 up to
// 128, 16-byte aligned rows, no mask, positive scale; 1 when it does not take the problem
// (nothing launched).
template <typename T>
int32_t attn_stream(const AttnParams& p, hipStream_t st);
// The same in fp32 (attention_stream32.hip): head dims that are a multiple of 4, same conditions.
int32_t attn_stream32(const AttnParams& p, hipStream_t st);

}  // namespace wc
