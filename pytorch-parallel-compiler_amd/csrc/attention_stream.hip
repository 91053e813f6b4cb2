// Streaming attention for 16-bit types (softmax(Q K^T * scale) V per (model, batch, head), causal
// or full), for keys that do not stay resident in LDS and for fp16.
//
// A workgroup of W waves owns W * 32 queries of one head, 32 per wave, and walks the keys in
// tiles of 64, K and V both row-major in LDS, double-buffered by LDS-DMA loads issued one tile
// ahead.  Per tile and wave, with v_mfma_f32_32x32x16:
//   S^T = K Q^T      lane l holds query l % 32 and the keys 8 (r / 4) + 4 (l / 32) + r % 4 of each
//                    32-key block in register r
//   softmax          in the lane: exp2(s * c - max), one FMA and one exponential per score; the row sum
//                    takes P in fp32, before it is rounded for P V.  The
//                    lane halves that share a query exchange their maxima, and O is rescaled,
//                    only in tiles where a lane of the wave finds a new running maximum.  (Letting
//                    the base lag behind the maximum by up to 2^8 is 12% faster, but rounds the
//                    largest P, which is exactly 1 otherwise: 2.08e-3 against 2.01e-3 from fp64.)
//   O^T += V^T P^T   P^T is the S^T register block itself: k-step j takes registers 8j .. 8j+7.
//                    V^T fragments come from the row-major tile through ds_read_b64_tr_b16, which
//                    hands lane i of 16 the i-th column of a 4-key x 16-column block, so V needs
//                    no transposed copy.
// Blocks past the diagonal are skipped per wave, and only tiles on the diagonal or past the
// last key evaluate a mask.
//
// Bound by the VALU: about 51 full-rate instructions and 16 exponentials per 32 x 32 scores
// against 256 cycles of MFMA at head dim 64; four waves per SIMD (two from head dim 96 on)
// overlap the two (causal, 2048 x 64: MFMAs 25 % of the cycles, other VALU instructions 48 %).  Registers: at
// head dim 64 the full forms spill 4 (eight waves) and 10 (four waves) to stay at four waves per SIMD.  Measured (us, heads x tokens x head dim; before: 16x16x32 MFMAs, V transposed
// on its way into LDS, a mask and a rescale on every tile):
//   bf16  64 x 2048 x 64 causal   159  -> 57.2  (601 TFLOP/s of the lower triangle)
//   bf16  64 x 2048 x 64          212  -> 100   (687 TFLOP/s)
//   bf16  32 x 2048 x 128 causal  244  -> 66.8
//   bf16  64 x 1024 x 80           93  -> 39.4
//   fp16  64 x 2048 x 64 causal   159  -> 55.0
#include "wc_attn.h"

#include <type_traits>

namespace wc {
namespace {


template <typename T>
__device__ __forceinline__ f32x16 st_mma(bf16x8 a, bf16x8 b, f32x16 c) {
  if constexpr (std::is_same<T, f16>::value)
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0,
                                                  0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef f16 f16x2 __attribute__((ext_vector_type(2)));

// two floats rounded to T in one dword
template <typename T>
__device__ __forceinline__ uint32_t st_pack(float lo, float hi) {
  if constexpr (std::is_same<T, f16>::value) {
    const f32x2 v = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, f16x2));
  } else {
    return pack_bf16x2(lo, hi);
  }
}

template <typename T, int DHP, int W, bool CAUSAL>
__global__ __launch_bounds__(W * 64) __attribute__((amdgpu_waves_per_eu(DHP <= 64 ? 4 : 2)))
void attn_stream_kernel(AttnParams p) {
  constexpr int NT = W * 64;
  constexpr int NKS = DHP / 16, DT = DHP / 32;
  constexpr int CPR = DHP / 8;                       // 16-byte chunks per row
  constexpr int CH = kStBK * CPR;                    // chunks of a K (or V) tile
  constexpr int PT = 2 * CH / NT;                    // chunks per thread
  constexpr int TILE = kStBK * DHP;                  // elements of a K (or V) tile
  static_assert(2 * CH % NT == 0, "chunks divide evenly");
  __shared__ __attribute__((aligned(16))) uint16_t lds[2][2 * TILE];   // [buffer][K tile, V tile]

  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int l32 = lane & 31, hf = lane >> 5;

  int bh, qt;
  stream_tile<CAUSAL>(p, bh, qt);
  const int nb = bh / p.heads, h = bh - (bh / p.heads) * p.heads;
  const int dh = p.dh;
  const T* qb = static_cast<const T*>(p.q) + nb * p.q_sb + static_cast<int64_t>(h) * dh;
  const T* kb = static_cast<const T*>(p.k) + nb * p.k_sb + static_cast<int64_t>(h) * dh;
  const T* vb = static_cast<const T*>(p.v) + nb * p.v_sb + static_cast<int64_t>(h) * dh;
  T* ob = static_cast<T*>(p.o) + nb * p.o_sb + static_cast<int64_t>(h) * dh;
  const int q0 = qt * W * 32 + wave * 32;            // the wave's first query
  const int q = q0 + l32;                            // the lane's query

  // ---- Q^T fragments (B operand of S^T): query l32, dims 16 k + 8 hf .. + 8 ----
  bf16x8 qf[NKS];
  {
    const T* qr = qb + static_cast<int64_t>(q < p.sq ? q : p.sq - 1) * p.q_ss;
#pragma unroll
    for (int k = 0; k < NKS; ++k) {
      const int c = 16 * k + 8 * hf;
      uint4 v = make_uint4(0, 0, 0, 0);
      if (c < dh) v = *reinterpret_cast<const uint4*>(qr + c);
      qf[k] = __builtin_bit_cast(bf16x8, v);
    }
  }

  // ---- staging: LDS-DMA loads, 16 bytes per lane.  Position tid + u * NT of a buffer (K's
  // chunks, then V's) belongs to this thread; the permutations of k_at / v_at are applied to the
  // chunk it fetches.  Keys past the last are written as zero (their scores are masked, but a P of
  // zero times what is left of an earlier tile could be NaN), columns past the head dim are not
  // loaded and stay zero. ----
  const int wbase = __builtin_amdgcn_readfirstlane(wave) * 64;
  const char* src[PT];
  int row[PT];
  bool in[PT];
#pragma unroll
  for (int u = 0; u < PT; ++u) {
    const bool isv = wbase + u * NT >= CH;            // the same for all lanes of a wave
    const int e = tid + u * NT - (isv ? CH : 0);
    row[u] = e / CPR;
    const int ch = e % CPR;
    const int col = isv ? v_at<DHP>(row[u], ch * 8) - row[u] * DHP : k_at<DHP>(row[u], ch) - row[u] * DHP;
    in[u] = col < dh;
    src[u] = reinterpret_cast<const char*>((isv ? vb : kb) + col);
  }
  auto fetch = [&](int buf, int k0) {
#pragma unroll
    for (int u = 0; u < PT; ++u) {
      const bool isv = wbase + u * NT >= CH;
      const int key = k0 + row[u];
      const char* from = src[u] + static_cast<int64_t>(key) * (isv ? p.v_ss : p.k_ss) * 2;
      if (in[u] && key < p.skv)
        __builtin_amdgcn_global_load_lds(reinterpret_cast<const void*>(from),
                                         (__attribute__((address_space(3))) void*)(&lds[buf][(wbase + u * NT) * 8]),
                                         16, 0, 0);
      else if (key >= p.skv)
        *reinterpret_cast<uint4*>(&lds[buf][(tid + u * NT) * 8]) = make_uint4(0, 0, 0, 0);
    }
  };

  f32x16 oacc[DT];
#pragma unroll
  for (int d = 0; d < DT; ++d)
#pragma unroll
    for (int e = 0; e < 16; ++e) oacc[d][e] = 0.f;
  const float c = p.scale_log2;
  // base: subtracted from the scaled scores, 0 until the query has met a score above -infinity (fresh;
  // its sums are zero until then); lrun: this lane half's part of the row sum
  float base = 0.f, lrun = 0.f;
  bool fresh = true;

  int kend = p.skv;
  if (CAUSAL) {
    int qlast = qt * W * 32 + W * 32 - 1;
    qlast = qlast < p.sq ? qlast : p.sq - 1;
    kend = qlast + 1 < kend ? qlast + 1 : kend;
  }
  const int ntiles = (kend + kStBK - 1) / kStBK;
  if (dh != DHP) {
    for (int e = tid; e < 2 * 2 * TILE / 8; e += NT) reinterpret_cast<uint4*>(&lds[0][0])[e] = make_uint4(0, 0, 0, 0);
    __syncthreads();
  }
  fetch(0, 0);
  __builtin_amdgcn_s_waitcnt(0x0f70);                // vmcnt(0): the LDS-DMA loads have landed
  __syncthreads();

  // one tile: the scores of its NB 32-key blocks (the second may lie past the diagonal or the last
  // key), the running maximum, then per block the exponentials and P V
  auto tile = [&](const uint16_t* ks, const uint16_t* vs, int k0, auto nblk_tag) {
    constexpr int NB = decltype(nblk_tag)::value;
    f32x16 s[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
#pragma unroll
      for (int e = 0; e < 16; ++e) s[b][e] = 0.f;
#pragma unroll
      for (int k = 0; k < NKS; ++k) {
        const bf16x8 kf = *reinterpret_cast<const bf16x8*>(ks + k_at<DHP>(32 * b + l32, 2 * k + hf));
        s[b] = st_mma<T>(kf, qf[k], s[b]);
      }
    }
    if (k0 + 32 * NB > p.skv || (CAUSAL && k0 + 32 * NB - 1 > q0)) {
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int key = k0 + 32 * b + (r >> 2) * 8 + 4 * hf + (r & 3);
          if (key >= p.skv || (CAUSAL && key > q)) s[b][r] = -INFINITY;
        }
    }
    float mx[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const float m0 = __builtin_fmaxf(__builtin_fmaxf(s[b][0], s[b][1]), s[b][2]);
      const float m1 = __builtin_fmaxf(__builtin_fmaxf(s[b][3], s[b][4]), s[b][5]);
      const float m2 = __builtin_fmaxf(__builtin_fmaxf(s[b][6], s[b][7]), s[b][8]);
      const float m3 = __builtin_fmaxf(__builtin_fmaxf(s[b][9], s[b][10]), s[b][11]);
      const float m4 = __builtin_fmaxf(__builtin_fmaxf(s[b][12], s[b][13]), s[b][14]);
      mx[b] = __builtin_fmaxf(__builtin_fmaxf(__builtin_fmaxf(m0, m1), m2),
                              __builtin_fmaxf(__builtin_fmaxf(m3, m4), s[b][15]));
    }
    float bm = (NB == 2 ? __builtin_fmaxf(mx[0], mx[NB - 1]) : mx[0]) * c;
    if (__builtin_amdgcn_ballot_w64(fresh || bm > base) != 0) {
      bm = __builtin_fmaxf(bm, __shfl_xor(bm, 32, 64));
      const bool up = (fresh || bm > base) && bm > -INFINITY;
      const float nbase = up ? bm : base;
      if (k0 != 0) {
        const float alpha = fresh ? 1.0f : __builtin_amdgcn_exp2f(base - nbase);
#pragma unroll
        for (int d = 0; d < DT; ++d) oacc[d] *= alpha;
        lrun *= alpha;
      }
      base = nbase;
      fresh = fresh && !up;
    }
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      // the row sum takes P before it is rounded for P V, on two independent chains
      uint32_t pk[8];
      float l0 = 0.f, l1 = 0.f;
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[b][2 * r], c, -base));
        const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[b][2 * r + 1], c, -base));
        l0 += p0;
        l1 += p1;
        pk[r] = st_pack<T>(p0, p1);
      }
      lrun += l0 + l1;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const uint4 pu = make_uint4(pk[4 * j], pk[4 * j + 1], pk[4 * j + 2], pk[4 * j + 3]);
        const bf16x8 pf = __builtin_bit_cast(bf16x8, pu);
#pragma unroll
        for (int d = 0; d < DT; ++d) {
          // keys 32 b + 16 j + 8 piece + 4 hf + (0 .. 3), columns 32 d + 16 (lane / 16 % 2) + (0 .. 15)
          const int row = 32 * b + 16 * j + 4 * hf + ((lane & 15) >> 2);
          const int col = 32 * d + (lane & 16) + 4 * (lane & 3);
          typedef __attribute__((address_space(3))) i16x4 lds_i16x4;
          const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(vs + v_at<DHP>(row, col)));
          const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(vs + v_at<DHP>(row + 8, col)));
          typedef short i16x8 __attribute__((ext_vector_type(8)));
          const i16x8 vf = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
          oacc[d] = st_mma<T>(__builtin_bit_cast(bf16x8, vf), pf, oacc[d]);
        }
      }
    }
  };

  for (int kt = 0; kt < ntiles; ++kt) {
    const int k0 = kt * kStBK;
    const uint16_t* ks = lds[kt & 1];
    // the other buffer was last read before the previous barrier
    if (kt + 1 < ntiles) fetch((kt + 1) & 1, k0 + kStBK);
    if (q0 < p.sq && !(CAUSAL && k0 > q0 + 31)) {
      if (k0 + 32 < p.skv && !(CAUSAL && k0 + 32 > q0 + 31))
        tile(ks, ks + TILE, k0, std::integral_constant<int, 2>{});
      else
        tile(ks, ks + TILE, k0, std::integral_constant<int, 1>{});
    }
    if (kt + 1 < ntiles) {
      __builtin_amdgcn_s_waitcnt(0x0f70);
      __syncthreads();
    }
  }

  // ---- O = (O^T / l)^T: lane holds query l32, dims 32 d + 8 (r / 4) + 4 hf + r % 4 ----
  const float lt = lrun + __shfl_xor(lrun, 32, 64);
  if (q < p.sq) {
    const float inv = lt > 0.f ? 1.0f / lt : (lt == 0.f ? 0.f : lt);      // NaN stays NaN
    T* orow = ob + static_cast<int64_t>(q) * p.o_ss;
#pragma unroll
    for (int d = 0; d < DT; ++d)
#pragma unroll
      for (int g4 = 0; g4 < 4; ++g4) {
        const int col = 32 * d + 8 * g4 + 4 * hf;
        if (col < dh) {                              // dh % 8 == 0: whole groups of 4
          const uint2 v = make_uint2(st_pack<T>(oacc[d][4 * g4] * inv, oacc[d][4 * g4 + 1] * inv),
                                     st_pack<T>(oacc[d][4 * g4 + 2] * inv, oacc[d][4 * g4 + 3] * inv));
          __builtin_memcpy(orow + col, &v, 8);       // output rows at element alignment
        }
      }
  }
}

template <typename T, int DHP, int W, bool CAUSAL>
int32_t launch_stream(AttnParams p, hipStream_t st) {
  p.q_tiles = static_cast<int>(cdiv(p.sq, W * 32));
  const int64_t blocks = static_cast<int64_t>(p.nb) * p.heads * p.q_tiles;
  if (blocks >= 0x7fffffffll) return set_error(WC_ERR_LIMIT, "wc_attention: too many tiles");
  attn_stream_kernel<T, DHP, W, CAUSAL><<<dim3(static_cast<uint32_t>(blocks)), dim3(W * 64), 0, st>>>(p);
  return check_launch("wc_attention");
}

// Four waves (128 queries) per workgroup, or eight, which read each K / V tile half as often, for
// full attention where 256-query tiles cover the CUs with little padding (64 x 2048 x 64 heads x
// tokens x head dim: 95.5 us against 102; 128 x 512 x 64 has no preference, 19.4 against 19.9;
// 256 x 333 x 64 pads, 23.2 against 20.6).  Causal tiles are better short (55.9 against 53.5),
// and at head dims past 96 the registers of eight waves leave one workgroup per CU.
template <typename T, int DHP>
int32_t stream_dh(const AttnParams& p, hipStream_t st) {
  if (p.causal) return launch_stream<T, DHP, 4, true>(p, st);
  if constexpr (DHP <= 96) {
    const int64_t tiles = cdiv(p.sq, 256);
    if (tiles * 256 - p.sq <= p.sq / 8 && static_cast<int64_t>(p.nb) * p.heads * tiles >= 256)
      return launch_stream<T, DHP, 8, false>(p, st);
  }
  return launch_stream<T, DHP, 4, false>(p, st);
}

}  // namespace

template <typename T>
int32_t attn_stream(const AttnParams& p, hipStream_t st) {
  if (p.dh % 8 != 0 || p.dh > 128 || p.mask || !(p.scale_log2 > 0.f && p.scale_log2 < INFINITY)) return 1;
  if (p.dh <= 32) return stream_dh<T, 32>(p, st);
  if (p.dh <= 64) return stream_dh<T, 64>(p, st);
  if (p.dh <= 96) return stream_dh<T, 96>(p, st);
  return stream_dh<T, 128>(p, st);
}

template int32_t attn_stream<bf16>(const AttnParams&, hipStream_t);
template int32_t attn_stream<f16>(const AttnParams&, hipStream_t);

}  // namespace wc
