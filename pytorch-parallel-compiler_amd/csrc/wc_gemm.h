// Internal interface of the grouped MFMA GEMM, shared by the kernel
// families that call it (recurrent input projection, attention projections).
#pragma once

#include "wc_common.h"

namespace wc {

// C[i][m][o] = act( sum_k A[i][m][k] W[i][o][k] + bias[i][o] + R[i][m][o] ),
// rows m of A / C / R addressed as (m / rows_inner) * s_outer + (m % rows_inner) * s_inner.
struct GemmParams {
  int n, m, o, k;
  int act;
  int tiles_m, tiles_o;
  int remap;
  const void* a;
  int64_t a_sn, a_so, a_si;
  FastDiv a_ri;
  const void* w;
  int64_t w_sn;
  const void* bias;
  int64_t b_sn;
  const void* r;
  int64_t r_sn, r_so, r_si;
  void* c;
  int64_t c_sn, c_so, c_si;
  FastDiv c_ri;
  // persistent XL kernel only: dividers of the stage -> tile -> (model, column tile) map,
  // and the byte extents of one model's C and R regions (their buffer descriptors' range,
  // so a stray offset is dropped by the hardware instead of reaching other memory)
  FastDiv fd_ks, fd_tpm, fd_tm;
  int32_t c_bytes, r_bytes;
  int vec_c;                   // tile kernel only: C and R rows take 16-byte accesses
  // a second weight and bias for the columns from o1 on (0: none); o1 is a multiple of the
  // launched tile, so a workgroup reads one of the two (tile and small-tile kernels)
  int o1 = 0;
  const void* w2 = nullptr;
  int64_t w2_sn = 0;
  const void* bias2 = nullptr;
  int64_t b2_sn = 0;
};

// Row 0 and bias element 0 of the weight that output columns o0 .. belong to, such that both are
// indexed by the output column.
template <typename TA>
__device__ __forceinline__ const TA* gemm_w(const GemmParams& p, int mdl, int o0) {
  if (p.o1 > 0 && o0 >= p.o1)
    return static_cast<const TA*>(p.w2) + static_cast<int64_t>(mdl) * p.w2_sn - static_cast<int64_t>(p.o1) * p.k;
  return static_cast<const TA*>(p.w) + static_cast<int64_t>(mdl) * p.w_sn;
}
template <typename TB>
__device__ __forceinline__ const TB* gemm_bias(const GemmParams& p, int mdl, int o0) {
  if (p.o1 > 0 && o0 >= p.o1)
    return p.bias2 ? static_cast<const TB*>(p.bias2) + static_cast<int64_t>(mdl) * p.b2_sn - p.o1 : nullptr;
  return p.bias ? static_cast<const TB*>(p.bias) + static_cast<int64_t>(mdl) * p.b_sn : nullptr;
}

// The tile kernel (gemm_tile.hip), with 128 x 128 or 64 x 64 tiles (bm); any sizes, strides and
// alignments.
template <typename TA, typename TC, typename TB>
int32_t gemm_tile(const GemmParams& p, int bm, hipStream_t st);

// dtype: A/W element type; out_dtype: WC_F32 or dtype; bias_dtype: WC_F32 or dtype.
int32_t grouped_gemm(const GemmParams& p, int32_t dtype, int32_t out_dtype, int32_t bias_dtype,
                     hipStream_t st);

}  // namespace wc
