// General implicit-GEMM convolution (N independent Conv1d / 2d / 3d layers; any stride, dilation,
// kernel and channel count) on 32x32x16 MFMAs, with the epilogue of conv.hip.
//
// Workgroup = (model, image, output depth, tile of up to 128 output pixels, 64 output channels),
// four waves of 64 pixels x 32 channels.  Input channels advance 32 at a time: the input tile
// with its halo is staged in LDS as [pixel][32 channels] (80-byte rows: 32 consecutive pixels'
// fragment reads hit all banks) and serves every tap; per tap the 64 x 32 weights are loaded one
// tap ahead into registers and double-buffered in LDS, one barrier per tap.  Two workgroups
// share a CU, so one's staging runs beside the other's MFMAs.
//
// fp32 values are split into three bf16 planes on their way into LDS and multiplied as the six
// plane products of at most second order (every bit of an fp32 value from 2^-110 on; dropped terms
// below 2^-26 of a product), which six bf16 MFMAs do in 3/8 of the fp32 MFMA's time.  A wave that ends
// with an infinity or NaN recomputes its outputs on the fp32 MFMA from memory, so such inputs give what
// fp32 arithmetic gives.  So does one of a workgroup that holds operands under 2^-110, which are looked
// for where they can show: by a result under kPlaneSmall, or an operand of kPlaneBig or more.  (16 models x 8,
// 64 -> 64, 3x3, 32 x 32: 76 us; a zero filter in every 64: 145 for the look; an infinite or small one: 360.)
//
// What bounds it, in fp32: the MFMAs (34 % of the cycles at 64 -> 64, 3x3) and the VALU work of splitting (30 %);
// for few taps or channels, staging the input tile (its loads are exposed at every 32-channel chunk but
// for the other workgroup).  Measured (us; before: the
// 16x16x4 fp32 MFMA / 16x16x32 with weight fragments read from L2 by every wave; 2-norm error of
// fp32 against fp64 in brackets):
//   fp32  16 models x 8, 64 -> 64, 3x3, 32 x 32    123 -> 72    [4.3e-7 -> 1.3e-7]  (134 TFLOP/s)
//   fp32   2 x 2, 128 -> 128, 7x7, 40 x 50         320 -> 170   [1.4e-6 -> 4.7e-7]
//   fp32  32 x 16, 1 -> 16, 3x3, 28 x 28           182 -> 80    [5.7e-8 -> 3.7e-8]
//   bf16   8 x 4, 64 -> 128, 3x3 stride 2, 33 x 33  41.6 -> 25.7
//   bf16  20 x 8, 96 -> 64, 3x3, 56 x 56           131 -> 116   (before: a 256-pixel tile kernel)
//   fp16  16 x 4, 128 -> 128, 3x3, 32 x 32          83 -> 43
#include <type_traits>

#include "wc_conv.h"

namespace wc {
namespace {

constexpr int kTPix = 128;             // output pixels per tile
constexpr int kXPitch = 40;            // 16-bit elements per staged pixel (32 channels + 8)

// elements per raw weight row: up to 32 channels of all taps, and 16 bytes against bank conflicts
template <typename T>
__host__ __device__ inline int raw_pitch(const ConvParams& p) {
  constexpr int CE = 16 / sizeof(T);
  return ((p.ci < 32 ? p.ci : 32) * p.kh * p.kw + CE - 1) / CE * CE + CE;
}

template <typename T>
__device__ __forceinline__ f32x16 ct_mma(bf16x8 a, bf16x8 b, f32x16 c) {
  if constexpr (std::is_same<T, f16>::value)
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0,
                                                  0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// 8 values as PLANES 16-byte rows; top: the largest fp32 one so far
template <typename T, int PLANES>
__device__ __forceinline__ void ct_planes(const T (&v)[8], uint4 (&pl)[PLANES], float& top) {
  if constexpr (PLANES == 1) {
    __builtin_memcpy(&pl[0], v, 16);
  } else {
    top = abs_max8(v, top);
    split_planes(v, pl);
  }
}

// RAW: the weights come from the module's filter bank [co][ci][taps] instead of the packed layout.  A
// 32-channel chunk's rows of all taps, contiguous per output channel, are staged in LDS as they are,
// and each tap's 8 channels are gathered from there.
template <typename T, bool RAW>
__global__ __launch_bounds__(kConvThreads) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 4 && !RAW ? 3 : 2)))
void conv_tile_kernel(ConvParams p) {
  constexpr int PLANES = sizeof(T) == 4 ? 3 : 1;
  constexpr int WPLANE = 64 * 32;                    // elements of one plane of a tap's weights
  extern __shared__ float4 smem4[];
  uint16_t* const xs = reinterpret_cast<uint16_t*>(smem4);         // [PLANES][pixels][kXPitch]
  const int npix = p.ir * p.ic;
  const int xplane = npix * kXPitch;
  uint16_t* const ws = xs + PLANES * xplane;                       // [2][PLANES][64][32]
  T* const raw = reinterpret_cast<T*>(ws + 2 * PLANES * WPLANE);   // RAW: [64][rp]
  __shared__ int flags[2];                                         // fp32: look at the operands again; compute again
  const int rp = raw_pitch<T>(p);

  // ---- tile coordinates ----
  const int per_img = p.tiles_r * p.tiles_c * p.tiles_co;
  const int nblk = p.n * p.batch * p.dout * per_img;
  int bid = blockIdx.x;
  if (p.remap) bid = (blockIdx.x & 7) * (nblk >> 3) + (blockIdx.x >> 3);
  const int img = bid / per_img;
  int rem = bid - img * per_img;
  const int tco = rem / (p.tiles_r * p.tiles_c);
  rem -= tco * (p.tiles_r * p.tiles_c);
  const int trr = rem / p.tiles_c;
  const int tcc = rem - trr * p.tiles_c;
  const int mdl = img / (p.batch * p.dout);
  const int bd = img - mdl * (p.batch * p.dout);
  const int bb = bd / p.dout;
  const int od = bd - bb * p.dout;
  const int ho0 = trr * p.tr, wo0 = tcc * p.tc, co0 = tco * 64;
  const int hi0 = ho0 * p.sh - p.ph, wi0 = wo0 * p.sw - p.pw;

  const int tid = threadIdx.x;
  const int wave = tid >> 6, lane = tid & 63;
  const int l32 = lane & 31, hf = lane >> 5;
  const int px0 = (wave >> 1) * 64, cw = (wave & 1) * 32;          // the wave's pixels and channels

  const T* const xb = static_cast<const T*>(p.x) + mdl * p.x_sn + bb * p.x_sb;
  const int taps = p.kh * p.kw, taps_all = p.kd * taps;
  const T* const wb = static_cast<const T*>(p.wp) + static_cast<int64_t>(mdl) * p.co * taps_all * p.ci32;

  // LDS offset (tap (0, 0)) of the lane's pixel in each A fragment; pixels past the tile read pixel 0
  int aoff[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int px = px0 + i * 32 + l32;
    const int pr = px / p.tc, pc = px - (px / p.tc) * p.tc;
    aoff[i] = (pr < p.tr ? (pr * p.sh) * p.ic + pc * p.sw : 0) * kXPitch + hf * 8;
  }
  // weights: thread t moves channels-in 8 (t % 4) .. + 8 of output channel t / 4 (past the last: repeated)
  const int wco = tid >> 2, wu = tid & 3;
  const T* const wsrc = wb + static_cast<int64_t>(co0 + wco < p.co ? co0 + wco : p.co - 1) * taps_all * p.ci32 + wu * 8;
  uint16_t* const wdst = ws + wco * 32 + ((wu ^ ((wco >> 1) & 3)) * 8);
  int boff[2];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
    const int row = cw + l32;
    boff[ks] = row * 32 + (((2 * ks + hf) ^ ((row >> 1) & 3)) * 8);
  }
  const T* const wnb = static_cast<const T*>(p.wn) + (static_cast<int64_t>(mdl) * p.co + co0) * p.ci * taps;
  const bool wlive = co0 + wco < p.co;
  T wreg[8];
  auto wload = [&](int tap, int t, int c0) {
    if constexpr (RAW) {
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const int ch = wu * 8 + q;
        wreg[q] = wlive && c0 + ch < p.ci ? raw[wco * rp + ch * taps + tap] : from_f32<T>(0.f);
      }
    } else {
      const int64_t koff = static_cast<int64_t>(t * taps + tap) * p.ci32 + c0;
      __builtin_memcpy(wreg, __builtin_assume_aligned(wsrc + koff, 16), sizeof(wreg));
    }
  };
  // RAW: rows of min(32, ci - c0) channels x taps in 16-byte pieces at element alignment (output
  // channels past the last are not loaded and count as zero)
  auto stage_raw = [&](int c0) {
    constexpr int CE = 16 / sizeof(T), U = 8;
    const int len = (p.ci - c0 < 32 ? p.ci - c0 : 32) * taps, upr = (len + CE - 1) / CE;
    const int rows = p.co - co0 < 64 ? p.co - co0 : 64;
    const int units = rows * upr;
    for (int e0 = tid; e0 < units; e0 += U * kConvThreads) {
      uint4 v[U];
      int dst[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int e = e0 + u * kConvThreads;
        dst[u] = -1;
        if (e < units) {
          const int r = e / upr, off = (e - r * upr) * CE;
          const T* src = wnb + (static_cast<int64_t>(r) * p.ci + c0) * taps + off;
          if (off + CE <= len) {
            __builtin_memcpy(&v[u], src, 16);
          } else {
            T tail[CE];
#pragma unroll
            for (int z = 0; z < CE; ++z) tail[z] = off + z < len ? src[z] : from_f32<T>(0.f);
            __builtin_memcpy(&v[u], tail, 16);
          }
          dst[u] = r * rp + off;
        }
      }
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (dst[u] >= 0) *reinterpret_cast<uint4*>(raw + dst[u]) = v[u];
    }
  };
  float top = 0.f;
  auto wstash = [&](int buf) {
    uint4 pl[PLANES];
    ct_planes<T, PLANES>(wreg, pl, top);
#pragma unroll
    for (int q = 0; q < PLANES; ++q)
      *reinterpret_cast<uint4*>(wdst + (buf * PLANES + q) * WPLANE) = pl[q];
  };

  // fp32: the largest plane product in one accumulator and the five small ones in another, whose
  // roundings are 2^-8 of the first's, so a k-step rounds the sum about once, like an fp32 MFMA
  constexpr int NACC = PLANES == 3 ? 2 : 1;
  f32x16 accs[NACC][2];
#pragma unroll
  for (int a = 0; a < NACC; ++a)
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e) accs[a][i][e] = 0.f;

  if (PLANES == 3 && tid < 2) flags[tid] = 0;
  bool staged = false;
  for (int t = 0; t < p.kd; ++t) {
    const int di = od * p.sd - p.pd + t * p.dd;
    if (di < 0 || di >= p.d) continue;               // uniform over the workgroup
    for (int c0 = 0; c0 < p.ci; c0 += 32) {
      const int nks = p.ci - c0 > 16 ? 2 : 1;        // 16-channel steps that hold a channel
      if (staged) __syncthreads();                   // everyone is done with the last chunk
      staged = true;
      if constexpr (RAW) stage_raw(c0);
      else wload(0, t, c0);
      // input tile: unit = 8 channels of one pixel, consecutive lanes on consecutive pixels
      {
        const int units = nks * 2 * npix;
        constexpr int U = 4;
        for (int e0 = tid; e0 < units; e0 += U * kConvThreads) {
          T v[U][8];
          int dst[U];
#pragma unroll
          for (int u = 0; u < U; ++u) {
            const int e = e0 + u * kConvThreads;
            dst[u] = -1;
            if (e < units) {
              const int cg = static_cast<int>(fdiv(static_cast<uint32_t>(e), p.fd_plane));
              const int rc = e - cg * npix;
              const int r = static_cast<int>(fdiv(static_cast<uint32_t>(rc), p.fd_ic));
              const int col = rc - r * p.ic;
              const int hi = hi0 + r, wi = wi0 + col, ch0 = c0 + cg * 8;
              const bool in = hi >= 0 && hi < p.h && wi >= 0 && wi < p.w;
              const T* src = xb + static_cast<int64_t>(ch0) * p.x_cs + (static_cast<int64_t>(di) * p.h + hi) * p.w + wi;
#pragma unroll
              for (int q = 0; q < 8; ++q)
                v[u][q] = (in && ch0 + q < p.ci) ? src[q * p.x_cs] : from_f32<T>(0.f);
              dst[u] = rc * kXPitch + cg * 8;
            }
          }
#pragma unroll
          for (int u = 0; u < U; ++u) {
            if (dst[u] < 0) continue;
            uint4 pl[PLANES];
            ct_planes<T, PLANES>(v[u], pl, top);
#pragma unroll
            for (int q = 0; q < PLANES; ++q) *reinterpret_cast<uint4*>(xs + q * xplane + dst[u]) = pl[q];
          }
        }
      }
      if constexpr (RAW) {
        __syncthreads();
        wload(0, t, c0);
      }
      wstash(0);
      __syncthreads();

      int r = 0, s = 0;                              // tap = r * kw + s
      for (int tap = 0; tap < taps; ++tap) {
        if (tap + 1 < taps) wload(tap + 1, t, c0);
        const int toff = ((r * p.dh) * p.ic + s * p.dw) * kXPitch;
        const uint16_t* const wt = ws + (tap & 1) * PLANES * WPLANE;
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
          if (ks < nks) {
            bf16x8 a[2][PLANES], b[PLANES];
#pragma unroll
            for (int q = 0; q < PLANES; ++q) {
#pragma unroll
              for (int i = 0; i < 2; ++i)
                a[i][q] = *reinterpret_cast<const bf16x8*>(xs + q * xplane + aoff[i] + toff + ks * 16);
              b[q] = *reinterpret_cast<const bf16x8*>(wt + q * WPLANE + boff[ks]);
            }
#pragma unroll
            for (int order = 0; order < PLANES; ++order)
#pragma unroll
              for (int q = 0; q <= order; ++q)
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                  f32x16& acc = accs[order == 0 ? 0 : NACC - 1][i];
                  acc = ct_mma<T>(a[i][q], b[order - q], acc);
                }
          }
        }
        if (++s == p.kw) {
          s = 0;
          ++r;
        }
        if (tap + 1 < taps) {
          wstash((tap + 1) & 1);                     // last read before the previous barrier
          __syncthreads();
        }
      }
    }
  }

  f32x16 acc[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    acc[i] = accs[0][i];
    if constexpr (NACC == 2) acc[i] += accs[1][i];
  }
  bool bad = false;                                  // fp32: the planes did not carry something
  if constexpr (PLANES == 3) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e) bad |= !(__builtin_fabsf(acc[i][e]) <= 3.402823466e38f);
    bool small = co0 + cw + l32 < p.co && abs_min16(acc[1], abs_min16(acc[0], INFINITY)) < kPlaneSmall;
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(small) != 0, 0)) {
      // of outputs that exist?  The wave's pixels, one a lane; then the lane's own: bit 32 i + 8 q + e
      const int px = px0 + lane, pr = px / p.tc;
      const uint64_t mine = __builtin_amdgcn_ballot_w64(pr < p.tr && ho0 + pr < p.ho && wo0 + px - pr * p.tc < p.wo) >>
                            (4 * hf);
      bool real = false;
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e)
          real |= __builtin_fabsf(acc[i][e]) < kPlaneSmall && (mine >> (32 * i + 8 * (e >> 2) + (e & 3)) & 1) != 0;
      small &= real;
    }
    // could an operand under kPlaneMin show?
    if (top >= kPlaneBig || small) flags[0] = 1;
  }
  // ---- bias and folded BN of the lane's channel, into LDS as [channel][pixel] ----
  const int co = co0 + cw + l32;
  float alpha = 1.f, beta = 0.f;
  if (co < p.co) {
    const int64_t pi = static_cast<int64_t>(mdl) * p.co + co;
    const float bv = p.bias ? ldp(p.bias, p.pdt, pi) : 0.f;
    beta = bv;
    if (p.bn_mean) {
      const float inv = 1.0f / sqrtf(ldp(p.bn_var, p.pdt, pi) + p.bn_eps);
      alpha = p.bn_w ? inv * ldp(p.bn_w, p.pdt, pi) : inv;
      beta = (p.bn_b ? ldp(p.bn_b, p.pdt, pi) : 0.f) - ldp(p.bn_mean, p.pdt, pi) * alpha;
      beta += bv * alpha;                            // (acc + bias) * alpha + beta
    }
  }
  __syncthreads();
  if constexpr (PLANES == 3) {
    if (__builtin_expect(flags[0] != 0 || __builtin_amdgcn_ballot_w64(bad) != 0, 0)) {
      // filters: wrow elements per output channel, tap (t, r, s) of channel c at ((t kh + r) kw + s) wts + c wcs
      const int wrow = RAW ? p.ci * taps : taps_all * p.ci32, wts = RAW ? 1 : p.ci32, wcs = RAW ? taps : 1;
      const T* const wall = RAW ? wnb : wb + static_cast<int64_t>(co0) * wrow;
      if (flags[0] != 0) {                             // the same for the whole workgroup
        bool below = false;
        const int64_t welems = static_cast<int64_t>(p.co - co0 < 64 ? p.co - co0 : 64) * wrow;
        for (int64_t e = tid * 8; e < welems; e += kConvThreads * 8) {
          T v[8];
#pragma unroll
          for (int q = 0; q < 8; ++q) v[q] = e + q < welems ? wall[e + q] : from_f32<T>(0.f);
          below |= below_planes(v);
        }
        for (int t = 0; t < p.kd; ++t) {
          const int di = od * p.sd - p.pd + t * p.dd;
          if (di < 0 || di >= p.d) continue;
          for (int e = tid; e < npix * ((p.ci + 7) / 8); e += kConvThreads) {
            const int cg = e / npix, rc = e - cg * npix, r = rc / p.ic;
            const int hi = hi0 + r, wi = wi0 + rc - r * p.ic;
            const bool in = hi >= 0 && hi < p.h && wi >= 0 && wi < p.w;
            const T* const xp = xb + static_cast<int64_t>(cg * 8) * p.x_cs +
                                (static_cast<int64_t>(di) * p.h + hi) * p.w + wi;
            T v[8];
#pragma unroll
            for (int q = 0; q < 8; ++q) v[q] = in && cg * 8 + q < p.ci ? xp[q * p.x_cs] : from_f32<T>(0.f);
            below |= below_planes(v);
          }
        }
        if (below) flags[1] = 1;
        __syncthreads();
        bad |= flags[1] != 0;
      }
      if (__builtin_amdgcn_ballot_w64(bad) != 0) {
        // 8 channels of a tap at a time, 4 of each lane half: a step pairs channels c and c + 4.  A padding pixel is
        // a zero that meets the weight: an infinite weight gives NaN there.
        const T* const wl = wall + static_cast<int64_t>(co0 + cw + l32 < p.co ? cw + l32 : p.co - 1 - co0) * wrow;
        int prow[2], pcol[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const int px = px0 + i * 32 + l32, pr = px / p.tc;
          prow[i] = pr < p.tr ? hi0 + pr * p.sh : hi0; // pixels past the tile repeat its first
          pcol[i] = pr < p.tr ? wi0 + (px - pr * p.tc) * p.sw : wi0;
#pragma unroll
          for (int e = 0; e < 16; ++e) acc[i][e] = 0.f;
        }
        for (int t = 0; t < p.kd; ++t) {
          const int di = od * p.sd - p.pd + t * p.dd;
          if (di < 0 || di >= p.d) continue;
          for (int r = 0; r < p.kh; ++r)
            for (int s = 0; s < p.kw; ++s) {
              const T* xp[2];
              bool in[2];
#pragma unroll
              for (int i = 0; i < 2; ++i) {
                const int hi = prow[i] + r * p.dh, wi = pcol[i] + s * p.dw;
                in[i] = hi >= 0 && hi < p.h && wi >= 0 && wi < p.w;
                xp[i] = xb + (static_cast<int64_t>(di) * p.h + hi) * p.w + wi;
              }
              const T* const wp = wl + static_cast<int64_t>((t * p.kh + r) * p.kw + s) * wts;
              for (int c0 = 4 * hf; c0 - 4 * hf < p.ci; c0 += 8)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                  const int c = c0 + e;
                  const float wv = c < p.ci ? to_f32(wp[c * wcs]) : 0.f;
#pragma unroll
                  for (int i = 0; i < 2; ++i) {
                    const float xv = c < p.ci && in[i] ? to_f32(xp[i][c * p.x_cs]) : 0.f;
                    acc[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(xv, wv, acc[i], 0, 0, 0);
                  }
                }
            }
        }
      }
    }
  }
  constexpr int CPITCH = kTPix + 8;
  T* const cs = reinterpret_cast<T*>(smem4);
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      T o[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = from_f32<T>(acc[i][4 * q + e] * alpha + beta);
      // lane: channel l32, pixels 8 q + 4 hf + (0 .. 3) of the fragment
      __builtin_memcpy(__builtin_assume_aligned(cs + (cw + l32) * CPITCH + px0 + i * 32 + 8 * q + 4 * hf, 4 * sizeof(T)),
                       o, sizeof(o));
    }
  __syncthreads();
  conv_store<T, kTPix>(p, cs, mdl, bb, ho0, wo0, co0, od);
}

// Tile shape: the one whose tiles (128 pixels of MFMA work each, plus their halo's staging) cover the
// output at the least cost, counting a tile that leaves only one workgroup per CU half again.
template <typename T>
bool tile_plan(ConvParams& p, size_t& lds) {
  constexpr int PLANES = sizeof(T) == 4 ? 3 : 1;
  auto bytes = [&](int64_t ir, int64_t ic) {
    const int64_t in = ir * ic * kXPitch * 2 * PLANES + 2 * PLANES * 64 * 64;
    const int64_t epi = static_cast<int64_t>(64) * (kTPix + 8) * sizeof(T);
    return in > epi ? in : epi;
  };
  double best = -1.0;
  for (int cand = kTPix; cand >= 4; cand >>= 1) {
    const int tc = p.wo < cand ? p.wo : cand;
    for (int tr = kTPix / tc < p.ho ? kTPix / tc : p.ho; tr >= 1; tr = tr / 2) {
      const int64_t ir = static_cast<int64_t>(tr - 1) * p.sh + static_cast<int64_t>(p.kh - 1) * p.dh + 1;
      const int64_t ic = static_cast<int64_t>(tc - 1) * p.sw + static_cast<int64_t>(p.kw - 1) * p.dw + 1;
      if (ir > 4096 || ic > 4096 || bytes(ir, ic) > 152 * 1024) continue;
      const double tiles = static_cast<double>(cdiv(p.ho, tr)) * static_cast<double>(cdiv(p.wo, tc));
      // staging a pixel costs about as much as the MFMAs of 4 / taps output pixels
      double cost = tiles * (kTPix + 4.0 * static_cast<double>(ir * ic) / (p.kh * p.kw));
      if (bytes(ir, ic) > 80 * 1024 - 16) cost *= 1.5;     // 16: the kernel's flags
      if (best < 0.0 || cost < best) {
        best = cost;
        p.tr = tr;
        p.tc = tc;
        p.ir = static_cast<int>(ir);
        p.ic = static_cast<int>(ic);
        lds = static_cast<size_t>(bytes(ir, ic));
      }
    }
  }
  return best >= 0.0;
}

// Where the filter bank is read as it is: few tiles (one round of workgroups), at most 9 taps and 160
// values per output channel.  It saves the packing launch, about 6 us of host time; beyond that staging and
// gathering the raw rows take longer than packing.  Measured (us for a whole forward, host included,
// filter bank / packed; models x images, channels, kernel, image):
//   fp32  30 x 8,   16 ->  64, 1x1, 10 x 10   15.7 / 21.2      bf16  2 x 3, 32 -> 32, 1x3, 389   17.8 / 23.5
//   bf16  16 x 8,  128 -> 128, 1x1, 8 x 8     14.7 / 20.4      fp32  1 x 3,  1 -> 32, 3x3, 31 x 15  15.5 / 20.9
//   fp32  16 x 2,   64 ->  64, 3x3, 14 x 14   34.9 / 28.5      fp16  6 x 15, 3 -> 128, 5x5, 8 x 26  22.4 / 21.8
template <typename T>
bool raw_fits(const ConvParams& q, size_t* total) {
  if (q.kd != 1 || q.kh * q.kw > 9 || q.ci * q.kh * q.kw > 160) return false;
  ConvParams p = q;
  size_t lds = 0;
  if (!tile_plan<T>(p, lds)) return false;
  const size_t in = static_cast<size_t>(p.ir) * p.ic * kXPitch * 2 * (sizeof(T) == 4 ? 3 : 1) +
                    2 * (sizeof(T) == 4 ? 3 : 1) * 64 * 64;
  const size_t all = in + static_cast<size_t>(64) * raw_pitch<T>(p) * sizeof(T);
  *total = all > lds ? all : lds;
  const int64_t blocks = mul_sat({p.n, p.batch, cdiv(p.ho, p.tr), cdiv(p.wo, p.tc), cdiv(p.co, 64)});
  int cus = device_cu_count();
  if (cus <= 0) cus = 256;
  return *total <= 152 * 1024 && blocks <= cus;
}

template <typename T>
int32_t launch_conv_tile(ConvParams p, const char* what, hipStream_t st) {
  size_t lds = 0, raw_lds = 0;
  if (!p.wp && !raw_fits<T>(p, &raw_lds)) return 1;
  if (!tile_plan<T>(p, lds)) return 1;
  if (!p.wp) lds = raw_lds;
  p.fd_plane = make_fastdiv(static_cast<uint32_t>(p.ir * p.ic));
  p.fd_ic = make_fastdiv(static_cast<uint32_t>(p.ic));
  p.tiles_r = static_cast<int>(cdiv(p.ho, p.tr));
  p.tiles_c = static_cast<int>(cdiv(p.wo, p.tc));
  p.tiles_co = static_cast<int>(cdiv(p.co, 64));
  constexpr int es = sizeof(T), ve = 16 / es;
  auto rows16 = [&](const void* q, int64_t sn, int64_t sb) {
    return aligned(q, 16) && ubytes(sn, es) % 16 == 0 && ubytes(sb, es) % 16 == 0;
  };
  p.vec_out = rows16(p.y, p.y_sn, p.y_sb) && (!p.res || rows16(p.res, p.r_sn, p.r_sb)) && p.tc % ve == 0 &&
              p.wo % ve == 0;
  const int64_t nblk = mul_sat({p.n, p.batch, p.dout, p.tiles_r, p.tiles_c, p.tiles_co});
  if (nblk >= 0x7fffffffll) return 1;                // conv_kernel's own limit decides
  p.remap = (nblk % 8 == 0) ? 1 : 0;
  auto kern = p.wp ? conv_tile_kernel<T, false> : conv_tile_kernel<T, true>;
  if (lds > 64 * 1024) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
    if (e != hipSuccess)
      return set_error(static_cast<int32_t>(e), "%s: LDS of %zu bytes refused: %s", what, lds, hipGetErrorString(e));
  }
  kern<<<dim3(static_cast<uint32_t>(nblk)), dim3(kConvThreads), lds, st>>>(p);
  return check_launch(what);
}

}  // namespace

bool conv_tile_raw(const ConvParams& p, int32_t dtype) {
  size_t lds = 0;
  if (dtype == WC_F32) return raw_fits<float>(p, &lds);
  return raw_fits<bf16>(p, &lds);                    // fp16 likewise: sizes only
}

int32_t conv_tile(const ConvParams& p, int32_t dtype, const char* what, hipStream_t st) {
  if (dtype == WC_F32) return launch_conv_tile<float>(p, what, st);
  if (dtype == WC_F16) return launch_conv_tile<f16>(p, what, st);
  return launch_conv_tile<bf16>(p, what, st);
}

}  // namespace wc
