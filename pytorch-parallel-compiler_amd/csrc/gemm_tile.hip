// Grouped GEMM for problems between the latency-bound small ones and the persistent XL kernel
// (both in gemm.hip):
//   C[i][m][o] = act( sum_k A[i][m][k] * W[i][o][k] + bias[i][o] + R[i][m][o] )
//
// A workgroup of four waves (2 x 2) computes a BM x BN tile of C on 32x32x16 MFMAs.  K advances
// 128 bytes of a row at a time (32 fp32 or 64 16-bit values): the next step's operands are loaded
// into registers while the current one feeds the MFMAs, then written to LDS.  Two or more
// workgroups share a CU, so one's loads, conversions and barriers run beside another's MFMAs.
//
// fp32 operands are split on their way into LDS into three bf16 planes,
//   v = v0 + v1 + v2,   v0 = bf16(v), v1 = bf16(v - v0), v2 = v - v0 - v1,
// which holds every bit of a normal fp32 value (8 + 8 + 8 mantissa bits, round to nearest), and
// the product is the sum of the six plane products of at most second order, accumulated in fp32.
// The dropped terms are below 2^-26 of a product.  The bf16 MFMA does 16 times the fp32 one's
// work per cycle, so six of them still take 2.7 times less, and each rounds its accumulator once
// for 16 values of k: measured against fp64 the result is closer than the fp32 MFMA's.
// Infinities and NaN (and values that round up to infinity in bf16) leave a NaN or an infinity
// in the accumulator; a wave that finds one recomputes its tile with the fp32 MFMA from memory,
// so such inputs give exactly what fp32 arithmetic gives.  Operands under 2^-110 the planes hold in
// fewer bits.  That can show in a result under kPlaneSmall, or beside an operand of kPlaneBig or more: a
// workgroup with either looks for such operands (its staged rows once more, a fifth of a tile's time) and
// if it finds one recomputes too.  Tracking the largest operand costs 1-2 %; testing each for being
// small instead cost 2-4, and 4-7 where zeros are common.
//
// What bounds it, in fp32: the MFMAs (42 % of the cycles at k = 256) and the VALU work of splitting the
// operands (about as many), which overlap only between waves; a large bf16 product reaches 1.25 PFLOP/s on
// this chip at the clock that random operands allow, a sixth of which is 208 TFLOP/s.  In 16 bits, and for
// short k, the latency of the first loads and the epilogue of each tile (MFMAs 13 % at k = 300).  Measured (us, before: the 16x16x4 fp32 MFMA and a 16-bit
// kernel with 32-deep K steps whose unaligned rows were loaded one value at a time):
//   fp32  16 x 2048 x 256 x 1024    204   -> 120    (143 TFLOP/s)
//   fp32   2 x 4096 x 2048 x 2048   633   -> 380    (181 TFLOP/s)
//   fp32  16 x 2048 x 257 x 1021    276   -> 137
//   bf16  20 x 800 x 300 x 1000     102   -> 28.5   (rows of 600 bytes)
//   bf16   4 x 4096 x 512 x 512      25.7 -> 17.5   (490 TFLOP/s)
// (models x m x k x o).  Error against fp64, 2-norm, fp32: 2.84e-7 -> 2.46e-7 at k = 256,
// 7.99e-7 -> 6.94e-7 at k = 2048.
#include "wc_gemm.h"

#include <type_traits>

namespace wc {

namespace {

constexpr int kTileThreads = 256;

__device__ __forceinline__ float tile_relu(float v) { return v > 0.f ? v : 0.f; }

// v_mfma_f32_32x32x16 on raw 16-byte fragments of the element type T (fp32: bf16 planes)
template <typename T>
__device__ __forceinline__ f32x16 mma32(bf16x8 a, bf16x8 b, f32x16 c) {
  if constexpr (std::is_same<T, f16>::value)
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0,
                                                  0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

template <typename T> struct Unit;                 // 8 consecutive k values of one row
template <> struct Unit<float> { uint4 v[2]; };
template <> struct Unit<bf16> { uint4 v[1]; };
template <> struct Unit<f16> { uint4 v[1]; };

template <typename TA, int FM, int FN>
struct TileCfg {
  static constexpr int PLANES = sizeof(TA) == 4 ? 3 : 1;
  static constexpr int BK = sizeof(TA) == 4 ? 32 : 64;      // k values per step (128 bytes of a row)
  static constexpr int UPR = BK / 8;                        // units per row
  static constexpr int BM = FM * 64, BN = FN * 64;
  static constexpr int ROWS = BM + BN;                      // A rows, then W rows
  static constexpr int UPT = ROWS * UPR / kTileThreads;     // units per thread
  static constexpr int PLANE = ROWS * BK;                   // 16-bit elements per plane
  static constexpr int STAGE_BYTES = PLANES * PLANE * 2;
  static constexpr int EPI_PITCH = FN * 32 + 4;             // floats per epilogue strip row
  static constexpr int EPI_BYTES = 4 * 32 * EPI_PITCH * 4;  // one 32-row strip per wave
  static constexpr int LDS = STAGE_BYTES > EPI_BYTES ? STAGE_BYTES : EPI_BYTES;
};

// At least two waves per SIMD (registers), so that two workgroups share a CU; three and, for the 64 x 64
// tile, five in fp32, which the compiler misses by a few registers if left alone.
template <typename TA, typename TC, typename TB, int FM, int FN>
__global__ __launch_bounds__(kTileThreads)
__attribute__((amdgpu_waves_per_eu(sizeof(TA) != 4 ? 2 : FM * FN == 1 ? 5 : 3)))
void gemm_tile_kernel(GemmParams p) {
  using C = TileCfg<TA, FM, FN>;
  constexpr int PLANES = C::PLANES, BK = C::BK, UPR = C::UPR, BM = C::BM, BN = C::BN, UPT = C::UPT;
  __shared__ __attribute__((aligned(16))) char smem[C::LDS];
  uint16_t* const lds = reinterpret_cast<uint16_t*>(smem);
  __shared__ int flags[2];                           // fp32: look at the operands again; compute again

  // tile coordinates (XCD-aware: consecutive tiles, which share operands, run on one XCD)
  const int tiles_per_model = p.tiles_m * p.tiles_o;
  const int nblk = p.n * tiles_per_model;
  int bid = blockIdx.x;
  if (p.remap) bid = (blockIdx.x & 7) * (nblk >> 3) + (blockIdx.x >> 3);
  const int mdl = bid / tiles_per_model;
  const int rem = bid - mdl * tiles_per_model;
  const int to = rem / p.tiles_m;
  const int m0 = (rem - to * p.tiles_m) * BM, o0 = to * BN;

  const int tid = threadIdx.x;
  const int wave = tid >> 6, lane = tid & 63;
  const int l32 = lane & 31, hf = lane >> 5;
  const int mw = (wave >> 1) * FM * 32, ow = (wave & 1) * FN * 32;   // the wave's corner of the tile

  const TA* const abase = static_cast<const TA*>(p.a) + static_cast<int64_t>(mdl) * p.a_sn;
  const TA* const wbase = gemm_w<TA>(p, mdl, o0);
  auto a_row = [&](int m) {
    m = m < p.m ? m : p.m - 1;                       // rows past the end repeat the last one (not stored)
    const uint32_t outer = fdiv(static_cast<uint32_t>(m), p.a_ri);
    return abase + static_cast<int64_t>(outer) * p.a_so + static_cast<int64_t>(m - outer * p.a_ri.d) * p.a_si;
  };
  auto w_row = [&](int o) { return wbase + static_cast<int64_t>(o < p.o ? o : p.o - 1) * p.k; };

  // staging: thread t moves unit t % UPR of rows t / UPR + q * (256 / UPR)
  constexpr int RPQ = kTileThreads / UPR;
  const int su = tid % UPR, sr = tid / UPR;
  const TA* src[UPT];
#pragma unroll
  for (int q = 0; q < UPT; ++q) {
    const int r = sr + q * RPQ;
    src[q] = (r < BM ? a_row(m0 + r) : w_row(o0 + r - BM)) + su * 8;
  }
  // LDS rows of BK 16-bit values; unit u of row r sits at u ^ ((r >> 1) % UPR), which keeps the
  // fragment reads (32 rows x 2 units) free of bank conflicts
  auto lds_at = [&](int plane, int row, int u) {
    return lds + plane * C::PLANE + row * BK + ((u ^ ((row >> 1) & (UPR - 1))) * 8);
  };

  Unit<TA> reg[UPT];
  auto fetch = [&](int k0) {
    if (k0 + BK <= p.k) {
      // 16-byte loads at element alignment (rows of any length)
#pragma unroll
      for (int q = 0; q < UPT; ++q) __builtin_memcpy(&reg[q], src[q] + k0, sizeof(Unit<TA>));
    } else {
      const int left = p.k - k0 - su * 8;            // values of this unit that exist
#pragma unroll
      for (int q = 0; q < UPT; ++q) {
        if (left >= 8) {
          __builtin_memcpy(&reg[q], src[q] + k0, sizeof(Unit<TA>));
        } else {
          TA t[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) t[e] = e < left ? src[q][k0 + e] : from_f32<TA>(0.f);
          __builtin_memcpy(&reg[q], t, sizeof(Unit<TA>));
        }
      }
    }
  };
  float top = 0.f;                                   // fp32: the largest operand this thread has staged
  auto stash = [&]() {
#pragma unroll
    for (int q = 0; q < UPT; ++q) {
      const int r = sr + q * RPQ;
      if constexpr (PLANES == 1) {
        *reinterpret_cast<uint4*>(lds_at(0, r, su)) = reg[q].v[0];
      } else {
        float f[8];
        __builtin_memcpy(f, &reg[q], sizeof(f));
        top = abs_max8(f, top);
        uint4 pl[3];
        split_planes(f, pl);
#pragma unroll
        for (int z = 0; z < 3; ++z) *reinterpret_cast<uint4*>(lds_at(z, r, su)) = pl[z];
      }
    }
  };

  // lane holds, for MFMA tile (i, j): row m = 32 i + l32, columns o = 32 j + 8 (r / 4) + 4 hf + r % 4
  f32x16 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
  // fp32, 64 x 64 tile: acc takes the largest plane product and low the five small ones, whose
  // roundings are 2^-8 of acc's, so a k-step of 16 rounds the sum about once (2-norm error at k = 16
  // 4.0e-8; 8.5e-8 with one accumulator, 7.8e-8 on the fp32 MFMA).  The 128 x 128 tile has no
  // registers for it (it costs the third wave per SIMD and 8 %) and takes k >= 64 only, where one
  // accumulator is closer than the fp32 MFMA too (1.35e-7 against 1.43e-7).
  constexpr bool LOW = PLANES == 3 && FM * FN == 1;
  f32x16 low;
#pragma unroll
  for (int e = 0; e < 16; ++e) low[e] = 0.f;

  if (PLANES == 3 && tid < 2) flags[tid] = 0;
  const int ksteps = (p.k + BK - 1) / BK;
  if (ksteps > 0) {
    fetch(0);
    stash();
  }
  __syncthreads();
  for (int kt = 0; kt < ksteps; ++kt) {
    if (kt + 1 < ksteps) fetch((kt + 1) * BK);
#pragma unroll
    for (int ks = 0; ks < BK / 16; ++ks) {
      bf16x8 am[FM][PLANES], wo[FN][PLANES];
#pragma unroll
      for (int pl = 0; pl < PLANES; ++pl) {
#pragma unroll
        for (int i = 0; i < FM; ++i)
          am[i][pl] = *reinterpret_cast<const bf16x8*>(lds_at(pl, mw + i * 32 + l32, 2 * ks + hf));
#pragma unroll
        for (int j = 0; j < FN; ++j)
          wo[j][pl] = *reinterpret_cast<const bf16x8*>(lds_at(pl, BM + ow + j * 32 + l32, 2 * ks + hf));
      }
      // plane products, largest order first; all tiles of one product before the next, so that
      // consecutive MFMAs are independent
#pragma unroll
      for (int order = 0; order < PLANES; ++order)
#pragma unroll
        for (int pa = 0; pa <= order; ++pa)
#pragma unroll
          for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) {
              f32x16& c = LOW && order > 0 ? low : acc[i][j];
              c = mma32<TA>(wo[j][order - pa], am[i][pa], c);
            }
    }
    __syncthreads();
    if (kt + 1 < ksteps) {
      stash();
      __syncthreads();
    }
  }

  if constexpr (PLANES == 3) {
    if constexpr (LOW) acc[0][0] += low;
    // what the planes do not carry: the wave's tile again, with the fp32 MFMA straight from memory
    bool bad = false;
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) bad |= !(__builtin_fabsf(acc[i][j][e]) <= 3.402823466e38f);
    float least = INFINITY;
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) least = abs_min16(acc[i][j], least);
    if (top >= kPlaneBig || least < kPlaneSmall) flags[0] = 1;     // an operand under kPlaneMin could show
    __syncthreads();
    if (flags[0] != 0) {
      bool below = false;
      for (int kt = 0; kt < ksteps; ++kt) {
        fetch(kt * BK);
#pragma unroll
        for (int q = 0; q < UPT; ++q) {
          float f[8];
          __builtin_memcpy(f, &reg[q], sizeof(f));
          below |= below_planes(f);
        }
      }
      if (below) flags[1] = 1;
      __syncthreads();
      bad |= flags[1] != 0;
    }
    if (__builtin_amdgcn_ballot_w64(bad) != 0) {
      const TA* ar[FM];
      const TA* wr[FN];
#pragma unroll
      for (int i = 0; i < FM; ++i) ar[i] = a_row(m0 + mw + i * 32 + l32);
#pragma unroll
      for (int j = 0; j < FN; ++j) wr[j] = w_row(o0 + ow + j * 32 + l32);
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
          for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
      // 8 values of k at a time, 4 of each lane half: a step pairs k and k + 4
      auto load4 = [&](const TA* row, int k) {
        f32x4 v = {0.f, 0.f, 0.f, 0.f};
        if (k + 4 <= p.k) {
          __builtin_memcpy(&v, row + k, 16);         // element alignment
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (k + e < p.k) v[e] = to_f32(row[k + e]);
        }
        return v;
      };
      for (int k0 = 0; k0 < p.k; k0 += 8) {
        f32x4 av[FM], wv[FN];
#pragma unroll
        for (int i = 0; i < FM; ++i) av[i] = load4(ar[i], k0 + 4 * hf);
#pragma unroll
        for (int j = 0; j < FN; ++j) wv[j] = load4(wr[j], k0 + 4 * hf);
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j)
              acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(wv[j][e], av[i][e], acc[i][j], 0, 0, 0);
      }
    }
  }

  // ---- epilogue: 32-row strips through LDS (the last step's barrier has freed it), so that
  // stores and residual loads run along rows ----
  const TB* const bias = gemm_bias<TB>(p, mdl, o0);
  TC* const cbase = static_cast<TC*>(p.c) + static_cast<int64_t>(mdl) * p.c_sn;
  const TC* const rbase = p.r ? static_cast<const TC*>(p.r) + static_cast<int64_t>(mdl) * p.r_sn : nullptr;
  constexpr int EP = C::EPI_PITCH;
  float* const strip = reinterpret_cast<float*>(smem) + wave * 32 * EP;
  const bool relu = p.act == WC_ACT_RELU;
  constexpr int VE = 16 / sizeof(TC);                // columns per 16-byte store
  constexpr int LPR = FN * 32 / VE;                  // lanes per row
  constexpr int RPI = 64 / LPR;                      // rows per store instruction
#pragma unroll
  for (int i = 0; i < FM; ++i) {
    const int row0 = m0 + mw + i * 32;
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const f32x4 v = {acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
        *reinterpret_cast<f32x4*>(strip + l32 * EP + j * 32 + 8 * q + 4 * hf) = v;
      }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (p.vec_c) {
      const int cl = (lane % LPR) * VE;
      const int col = o0 + ow + cl;
      if (col < p.o) {
        float bv[VE];
#pragma unroll
        for (int e = 0; e < VE; ++e) bv[e] = bias ? to_f32(bias[col + e]) : 0.f;
#pragma unroll
        for (int s = 0; s < 32 / RPI; ++s) {
          const int lr = s * RPI + lane / LPR;
          const int row = row0 + lr;
          if (row < p.m) {
            const uint32_t outer = fdiv(static_cast<uint32_t>(row), p.c_ri);
            const uint32_t inner = row - outer * p.c_ri.d;
            float v[VE];
#pragma unroll
            for (int e = 0; e < VE; e += 4) {
              const f32x4 t = *reinterpret_cast<const f32x4*>(strip + lr * EP + cl + e);
#pragma unroll
              for (int z = 0; z < 4; ++z) v[e + z] = t[z] + bv[e + z];
            }
            if (rbase) {
              TC r[VE];
              __builtin_memcpy(r, __builtin_assume_aligned(rbase + static_cast<int64_t>(outer) * p.r_so +
                                                           static_cast<int64_t>(inner) * p.r_si + col, 16), 16);
#pragma unroll
              for (int e = 0; e < VE; ++e) v[e] += to_f32(r[e]);
            }
            TC out[VE];
#pragma unroll
            for (int e = 0; e < VE; ++e) out[e] = from_f32<TC>(relu ? tile_relu(v[e]) : v[e]);
            __builtin_memcpy(__builtin_assume_aligned(cbase + static_cast<int64_t>(outer) * p.c_so +
                                                      static_cast<int64_t>(inner) * p.c_si + col, 16), out, 16);
          }
        }
      }
    } else {
      // rows or widths that 16-byte stores do not fit: one column per lane
      for (int c0 = 0; c0 < FN * 32; c0 += 64) {
        const int cl = c0 + (FN * 32 >= 64 ? lane : l32);
        const int col = o0 + ow + cl;
        constexpr int RS = FN * 32 >= 64 ? 1 : 2;     // rows per pass
        if (col < p.o) {
          const float bv = bias ? to_f32(bias[col]) : 0.f;
          for (int lr = RS == 1 ? 0 : hf; lr < 32 && row0 + lr < p.m; lr += RS) {
            const int row = row0 + lr;
            const uint32_t outer = fdiv(static_cast<uint32_t>(row), p.c_ri);
            const uint32_t inner = row - outer * p.c_ri.d;
            float v = strip[lr * EP + cl] + bv;
            if (rbase)
              v += to_f32(rbase[static_cast<int64_t>(outer) * p.r_so + static_cast<int64_t>(inner) * p.r_si + col]);
            if (relu) v = tile_relu(v);
            cbase[static_cast<int64_t>(outer) * p.c_so + static_cast<int64_t>(inner) * p.c_si + col] =
                from_f32<TC>(v);
          }
        }
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
}

template <typename TA, typename TC, typename TB, int FM, int FN>
int32_t launch_tile(GemmParams p, hipStream_t st) {
  using C = TileCfg<TA, FM, FN>;
  p.tiles_m = static_cast<int>(cdiv(p.m, C::BM));
  p.tiles_o = static_cast<int>(cdiv(p.o, C::BN));
  const int64_t nblk = static_cast<int64_t>(p.n) * p.tiles_m * p.tiles_o;
  if (nblk >= 0x7fffffffll) return set_error(WC_ERR_LIMIT, "wc_grouped_gemm: too many tiles");
  p.remap = (nblk % 8 == 0) ? 1 : 0;
  const int ce = sizeof(TC);
  p.vec_c = p.o % (16 / ce) == 0 &&
            common_vec_bytes({reinterpret_cast<uintptr_t>(p.c), ubytes(p.c_sn, ce), ubytes(p.c_so, ce),
                              ubytes(p.c_si, ce)}) >= 16 &&
            (!p.r || common_vec_bytes({reinterpret_cast<uintptr_t>(p.r), ubytes(p.r_sn, ce), ubytes(p.r_so, ce),
                                       ubytes(p.r_si, ce)}) >= 16);
  gemm_tile_kernel<TA, TC, TB, FM, FN><<<dim3(static_cast<uint32_t>(nblk)), dim3(kTileThreads), 0, st>>>(p);
  return check_launch("wc_grouped_gemm");
}

}  // namespace

template <typename TA, typename TC, typename TB>
int32_t gemm_tile(const GemmParams& p, int bm, hipStream_t st) {
  return bm == 128 ? launch_tile<TA, TC, TB, 2, 2>(p, st) : launch_tile<TA, TC, TB, 1, 1>(p, st);
}

#define WC_TILE(TA, TC, TB) template int32_t gemm_tile<TA, TC, TB>(const GemmParams&, int, hipStream_t);
WC_TILE(float, float, float)
WC_TILE(bf16, bf16, bf16) WC_TILE(bf16, bf16, float) WC_TILE(bf16, float, bf16) WC_TILE(bf16, float, float)
WC_TILE(f16, f16, f16) WC_TILE(f16, f16, float) WC_TILE(f16, float, f16) WC_TILE(f16, float, float)
#undef WC_TILE

}  // namespace wc
