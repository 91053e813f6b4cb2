// Internal interface of the convolution kernels.
#pragma once

#include "wc_common.h"

namespace wc {

struct ConvParams {
  int n, batch, ci, co, h, w, kh, kw, sh, sw, ph, pw, dh, dw, ho, wo;
  // depth of a 3-D convolution (2-D: kd = d = dout = 1, sd = dd = 1, pd = 0); only the
  // general kernel reads them.  x_cs / y_cs: channel-plane strides (d*h*w, dout*ho*wo).
  int kd, sd, pd, dd, d, dout;
  int64_t x_cs, y_cs;
  int ci32;                 // input channels padded to a multiple of 32
  int cc;                   // input channels staged per LDS chunk (multiple of 32)
  int tr, tc;               // output tile rows / cols
  int ir, ic;               // input tile rows / cols
  int tiles_r, tiles_c, tiles_co;
  int remap, act, vec_out;
  FastDiv fd_plane, fd_ic;  // ir*ic and ic
  const void* x;
  int64_t x_sn, x_sb;
  const void* wp;           // packed weights [n][co][kh][kw][ci32]
  const void* wn;           // or (resident-weight kernel, tile kernel) the filter bank [n*co][ci][kh][kw]
  const void* bias;         // [n*co] or null
  const void* bn_w;         // eval BN params [n*co] (bn_mean null: no BN)
  const void* bn_b;
  const void* bn_mean;
  const void* bn_var;
  float bn_eps;
  int pdt;                  // element type of bias / BN params
  const void* res;
  int64_t r_sn, r_sb;
  void* y;
  int64_t y_sn, y_sb;
};


constexpr int kConvThreads = 256;

__device__ __forceinline__ float ldp(const void* p, int dt, int64_t i) {
  if (dt == WC_F32) return static_cast<const float*>(p)[i];
  if (dt == WC_F16) return static_cast<float>(static_cast<const f16*>(p)[i]);
  return static_cast<float>(static_cast<const bf16*>(p)[i]);
}


// Second half of a conv kernel's epilogue: the tile cs [64 channels][TPIX + 8] (bias and BN
// applied, output type, in LDS) with residual add and ReLU to coalesced NCHW stores.
template <typename T, int TPIX>
__device__ __forceinline__ void conv_store(const ConvParams& p, const T* cs, int mdl, int bb, int ho0, int wo0,
                                           int co0, int od) {
  constexpr int CPITCH = TPIX + 8;
  const int tid = threadIdx.x;
  const int64_t dpl = static_cast<int64_t>(od) * p.ho * p.wo;   // output depth slice
  T* yb = static_cast<T*>(p.y) + mdl * p.y_sn + bb * p.y_sb + dpl;
  const T* rb = p.res ? static_cast<const T*>(p.res) + mdl * p.r_sn + bb * p.r_sb + dpl : nullptr;
  const int64_t how = p.y_cs;                                    // channel-plane stride
  constexpr int VE = 16 / sizeof(T);
  if (p.vec_out) {
    // tc % VE == 0, wo0 % VE == 0, rows of y / res 16-byte aligned; EB chunks per
    // thread are handled together so their residual loads are in flight at once
    constexpr int EB = 4;
    const int chunks = 64 * (TPIX / VE);
    for (int e0 = tid; e0 < chunks; e0 += EB * kConvThreads) {
      int64_t off[EB];
      int lds_at[EB];
      uint4 rv[EB];
#pragma unroll
      for (int u = 0; u < EB; ++u) {
        const int e = e0 + u * kConvThreads;
        off[u] = -1;
        if (e >= chunks) continue;
        const int col = e / (TPIX / VE);
        const int px = (e - col * (TPIX / VE)) * VE;
        const int pr = px / p.tc, pc = px - (px / p.tc) * p.tc;
        const int co = co0 + col, oh = ho0 + pr, ow = wo0 + pc;
        if (co >= p.co || pr >= p.tr || oh >= p.ho || ow >= p.wo) continue;
        off[u] = static_cast<int64_t>(co) * how + oh * p.wo + ow;
        lds_at[u] = col * CPITCH + px;
        if (rb) rv[u] = *reinterpret_cast<const uint4*>(rb + off[u]);
      }
#pragma unroll
      for (int u = 0; u < EB; ++u) {
        if (off[u] < 0) continue;
        float v[VE];
        const T* src = &cs[lds_at[u]];
#pragma unroll
        for (int q = 0; q < VE; ++q) v[q] = to_f32(src[q]);
        if (rb) {
          const T* rr = reinterpret_cast<const T*>(&rv[u]);
#pragma unroll
          for (int q = 0; q < VE; ++q) v[q] = to_f32(from_f32<T>(v[q] + to_f32(rr[q])));
        }
        uint4 ov;
        T* oo = reinterpret_cast<T*>(&ov);
#pragma unroll
        for (int q = 0; q < VE; ++q) oo[q] = from_f32<T>(p.act == WC_ACT_RELU ? fmaxf(v[q], 0.f) : v[q]);
        *reinterpret_cast<uint4*>(yb + off[u]) = ov;
      }
    }
  } else {
    for (int e = tid; e < 64 * TPIX; e += kConvThreads) {
      const int col = e / TPIX;
      const int px = e - col * TPIX;
      const int pr = px / p.tc, pc = px - (px / p.tc) * p.tc;
      const int co = co0 + col, oh = ho0 + pr, ow = wo0 + pc;
      if (co >= p.co || pr >= p.tr || oh >= p.ho || ow >= p.wo) continue;
      const int64_t off = static_cast<int64_t>(co) * how + oh * p.wo + ow;
      float v = to_f32(cs[col * CPITCH + px]);
      if (rb) v = to_f32(from_f32<T>(v + to_f32(rb[off])));
      if (p.act == WC_ACT_RELU) v = fmaxf(v, 0.f);
      yb[off] = from_f32<T>(v);
    }
  }
}

// The tile kernel (conv_tile.hip); 1 when its tiles do not fit LDS (nothing launched).  p holds the
// sizes, strides and packed weights; tiles are planned inside.
int32_t conv_tile(const ConvParams& p, int32_t dtype, const char* what, hipStream_t st);
// true where the tile kernel reads the filter bank itself (p.wp null)
bool conv_tile_raw(const ConvParams& p, int32_t dtype);

}  // namespace wc
