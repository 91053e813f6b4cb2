// Streaming attention in fp32 (softmax(Q K^T * scale) V per (model, batch, head), causal or full),
// head dims up to 64: the structure of attention_stream.hip on bf16 planes.
//
// Q, K, V and P are split into three bf16 planes (v = v0 + v1 + v2, every bit of a value from 2^-110 on) and
// multiplied as the six plane products of at most second order, the largest in one accumulator and
// the five small ones in another, so a step of 16 rounds the sum about once.  Six 32x32x16 bf16
// MFMAs take 3/8 of the fp32 MFMA's time.  K and V tiles of 64 keys are loaded one tile ahead,
// split on their way into LDS, and V^T comes from the row-major planes through
// ds_read_b64_tr_b16.  Softmax, maxima and row sums are fp32 as before.
//
// What the planes do not carry: a workgroup that met a Q or K of 2^56 or more, where a score could overflow
// or the planes' absolute error could count, or a V of 2^100 or more, where a sum could, or a non-zero V under
// 2^-110, computes its queries again on the fp32 MFMA, straight from memory.
//
// Bound by the VALU (softmax, splitting P: about 2,000 cycles per wave and tile against 1,536 of
// MFMAs at head dim 32; at 128 tokens MFMAs take 25 % of the cycles, other VALU instructions 45 %) and, for
// short sequences, by the latency of the first loads.  Measured (us,
// heads x tokens x head dim; before: 16x16x4 fp32 MFMAs, V transposed one value at a time; 2-norm
// error against fp64 in brackets):
//   2048 x 128 x 32            60 -> 40.5  [2.9e-7 -> 1.3e-7]
//     64 x 2048 x 64          653 -> 383   [8.7e-7 -> 3.5e-7]  (179 TFLOP/s)
//     64 x 2048 x 64 causal   538 -> 217   [4.0e-7 -> 1.7e-7]
//    512 x 512 x 32           179 -> 109
// With the fp32 pass 64 x 2048 x 64 takes 990 us (small V), 2,150 (infinite keys); the general kernel 653.
// Registers: no scratch at head dims up to 32, 7 (causal 10) spilled at 64; head dims past 64 (Q and O planes of
// 128 columns) would spill far more and keep the general kernel.
#include "wc_attn.h"

namespace wc {
namespace {

typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef short i16x8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) i16x4 lds_i16x4;

constexpr int kS32Threads = 256;       // four waves of 32 queries
constexpr float kBigV = 0x1p100f;      // below it no sum of 2^27 values overflows

template <int DHP, bool CAUSAL>
__global__ __launch_bounds__(kS32Threads) __attribute__((amdgpu_waves_per_eu(DHP == 32 ? 3 : 2)))
void attn_stream32_kernel(AttnParams p) {
  constexpr int NT = kS32Threads;
  constexpr int NKS = DHP / 16, DT = DHP / 32;
  constexpr int UPR = DHP / 8;                       // 8-value units per row
  constexpr int UN = kStBK * UPR;                    // units of a K (or V) tile
  constexpr int PT = 2 * UN / NT;                    // units per thread
  constexpr int TILE = kStBK * DHP;                  // 16-bit elements of one plane of a tile
  constexpr int NBUF = DHP == 32 ? 2 : 1;            // what leaves three workgroups per CU their LDS
  static_assert(2 * UN % NT == 0 && UN % NT == 0, "units divide evenly");
  __shared__ __attribute__((aligned(16))) uint16_t lds[NBUF][2][3][TILE];   // K planes, V planes
  __shared__ int odd_flag;

  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int l32 = lane & 31, hf = lane >> 5;
  int bh, qt;
  stream_tile<CAUSAL>(p, bh, qt);
  const int nb = bh / p.heads, h = bh - (bh / p.heads) * p.heads;
  const int dh = p.dh;
  const float* qb = static_cast<const float*>(p.q) + nb * p.q_sb + static_cast<int64_t>(h) * dh;
  const float* kb = static_cast<const float*>(p.k) + nb * p.k_sb + static_cast<int64_t>(h) * dh;
  const float* vb = static_cast<const float*>(p.v) + nb * p.v_sb + static_cast<int64_t>(h) * dh;
  float* ob = static_cast<float*>(p.o) + nb * p.o_sb + static_cast<int64_t>(h) * dh;
  const int q0 = qt * 128 + wave * 32;               // the wave's first query
  const int q = q0 + l32;                            // the lane's query
  if (tid == 0) odd_flag = 0;
  __syncthreads();

  bool odd = false;                                  // met what the planes do not carry
  // 8 values from src, those at column c and past it that exist
  auto load8 = [&](const float* src, int c, float (&v)[8]) {
    f32x4 a = {0.f, 0.f, 0.f, 0.f}, b = a;
    if (c < dh) a = *reinterpret_cast<const f32x4*>(src + c);
    if (c + 4 < dh) b = *reinterpret_cast<const f32x4*>(src + c + 4);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v[e] = a[e];
      v[4 + e] = b[e];
    }
  };
  // ---- Q^T planes (B operand of S^T): query l32, dims 16 k + 8 hf .. + 8 ----
  bf16x8 qf[NKS][3];
  {
    const float* qr = qb + static_cast<int64_t>(q < p.sq ? q : p.sq - 1) * p.q_ss;
#pragma unroll
    for (int k = 0; k < NKS; ++k) {
      float v[8];
      load8(qr, 16 * k + 8 * hf, v);
      odd |= abs_max8(v) >= kPlaneSafe;
      uint4 pl[3];
      split_planes(v, pl);
#pragma unroll
      for (int z = 0; z < 3; ++z) qf[k][z] = __builtin_bit_cast(bf16x8, pl[z]);
    }
  }

  // ---- staging: unit tid + u * NT of K (u < PT / 2), then of V ----
  float reg[PT][8];
  auto fetch = [&](int k0) {
#pragma unroll
    for (int u = 0; u < PT; ++u) {
      const bool isv = u >= PT / 2;
      const int e = tid + (isv ? u - PT / 2 : u) * NT;
      const int key = k0 + e / UPR, c = (e % UPR) * 8;
#pragma unroll
      for (int z = 0; z < 8; ++z) reg[u][z] = 0.f;
      if (key < p.skv)
        load8(isv ? vb + static_cast<int64_t>(key) * p.v_ss : kb + static_cast<int64_t>(key) * p.k_ss, c, reg[u]);
    }
  };
  auto stash = [&](int buf) {
#pragma unroll
    for (int u = 0; u < PT; ++u) {
      const bool isv = u >= PT / 2;
      const int e = tid + (isv ? u - PT / 2 : u) * NT;
      const int key = e / UPR, c = e % UPR;
      odd |= abs_max8(reg[u]) >= (isv ? kBigV : kPlaneSafe);
      if (isv && __builtin_amdgcn_ballot_w64(abs_min8(reg[u]) < kPlaneMin) != 0) odd |= below_planes(reg[u]);
      uint4 pl[3];
      split_planes(reg[u], pl);
      const int at = isv ? v_at<DHP>(key, c * 8) : k_at<DHP>(key, c);
#pragma unroll
      for (int z = 0; z < 3; ++z) *reinterpret_cast<uint4*>(&lds[buf][isv ? 1 : 0][z][at]) = pl[z];
    }
  };

  f32x16 oacc[DT];
#pragma unroll
  for (int d = 0; d < DT; ++d)
#pragma unroll
    for (int e = 0; e < 16; ++e) oacc[d][e] = 0.f;
  const float c = p.scale_log2;
  float base = 0.f, lrun = 0.f;                      // base: 0 until the first tile sets it

  int kend = p.skv;
  if (CAUSAL) {
    int qlast = qt * 128 + 127;
    qlast = qlast < p.sq ? qlast : p.sq - 1;
    kend = qlast + 1 < kend ? qlast + 1 : kend;
  }
  const int ntiles = (kend + kStBK - 1) / kStBK;
  fetch(0);
  stash(0);
  __syncthreads();

  // one tile: as in the 16-bit kernel, both 32-key blocks (keys past the diagonal or the last are masked)
  auto tile = [&](int buf, int k0) {
    f32x16 s[2];
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      f32x16 lo;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        s[b][e] = 0.f;
        lo[e] = 0.f;
      }
#pragma unroll
      for (int k = 0; k < NKS; ++k) {
        bf16x8 kf[3];
#pragma unroll
        for (int z = 0; z < 3; ++z)
          kf[z] = *reinterpret_cast<const bf16x8*>(&lds[buf][0][z][k_at<DHP>(32 * b + l32, 2 * k + hf)]);
        s[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[0], qf[k][0], s[b], 0, 0, 0);
#pragma unroll
        for (int order = 1; order < 3; ++order)
#pragma unroll
          for (int z = 0; z <= order; ++z)
            lo = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[order - z], qf[k][z], lo, 0, 0, 0);
      }
      s[b] += lo;
    }
    if (k0 + 64 > p.skv || (CAUSAL && k0 + 63 > q0)) {
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int key = k0 + 32 * b + (r >> 2) * 8 + 4 * hf + (r & 3);
          if (key >= p.skv || (CAUSAL && key > q)) s[b][r] = -INFINITY;
        }
    }
    float bm = -INFINITY;
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const float m0 = __builtin_fmaxf(__builtin_fmaxf(s[b][0], s[b][1]), s[b][2]);
      const float m1 = __builtin_fmaxf(__builtin_fmaxf(s[b][3], s[b][4]), s[b][5]);
      const float m2 = __builtin_fmaxf(__builtin_fmaxf(s[b][6], s[b][7]), s[b][8]);
      const float m3 = __builtin_fmaxf(__builtin_fmaxf(s[b][9], s[b][10]), s[b][11]);
      const float m4 = __builtin_fmaxf(__builtin_fmaxf(s[b][12], s[b][13]), s[b][14]);
      bm = __builtin_fmaxf(bm, __builtin_fmaxf(__builtin_fmaxf(__builtin_fmaxf(m0, m1), m2),
                                               __builtin_fmaxf(__builtin_fmaxf(m3, m4), s[b][15])));
    }
    bm *= c;
    const bool first = k0 == 0;
    if (__builtin_amdgcn_ballot_w64(first || bm > base) != 0) {
      bm = __builtin_fmaxf(bm, __shfl_xor(bm, 32, 64));
      const float nbase = (first || bm > base) && bm > -INFINITY ? bm : base;
      if (!first) {
        const float alpha = __builtin_amdgcn_exp2f(base - nbase);
#pragma unroll
        for (int d = 0; d < DT; ++d) oacc[d] *= alpha;
        lrun *= alpha;
      }
      base = nbase;
    }
    f32x16 olo[DT];
#pragma unroll
    for (int d = 0; d < DT; ++d)
#pragma unroll
      for (int e = 0; e < 16; ++e) olo[d][e] = 0.f;
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      float l0 = 0.f, l1 = 0.f;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        float pv[8];
#pragma unroll
        for (int r = 0; r < 8; ++r) {
          // one rounding of the argument (the largest P is 1 to within that of the scaled maximum)
          pv[r] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[b][8 * j + r], c, -base));
          if (r & 1) l1 += pv[r];
          else l0 += pv[r];
        }
        uint4 pu[3];
        split_planes(pv, pu);
#pragma unroll
        for (int d = 0; d < DT; ++d) {
          // keys 32 b + 16 j + 8 piece + 4 hf + (0 .. 3), columns 32 d + 16 (lane / 16 % 2) + (0 .. 15)
          const int row = 32 * b + 16 * j + 4 * hf + ((lane & 15) >> 2);
          const int col = 32 * d + (lane & 16) + 4 * (lane & 3);
          bf16x8 vf[3];
#pragma unroll
          for (int z = 0; z < 3; ++z) {
            const uint16_t* vs = lds[buf][1][z];
            const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(vs + v_at<DHP>(row, col)));
            const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(vs + v_at<DHP>(row + 8, col)));
            const i16x8 v8 = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
            vf[z] = __builtin_bit_cast(bf16x8, v8);
          }
          oacc[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[0], __builtin_bit_cast(bf16x8, pu[0]), oacc[d], 0, 0, 0);
#pragma unroll
          for (int order = 1; order < 3; ++order)
#pragma unroll
            for (int z = 0; z <= order; ++z)
              olo[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[order - z], __builtin_bit_cast(bf16x8, pu[z]), olo[d],
                                                               0, 0, 0);
        }
      }
      lrun += l0 + l1;
    }
#pragma unroll
    for (int d = 0; d < DT; ++d) oacc[d] += olo[d];
  };

  for (int kt = 0; kt < ntiles; ++kt) {
    const int k0 = kt * kStBK;
    if (kt + 1 < ntiles) fetch(k0 + kStBK);
    if (q0 < p.sq && !(CAUSAL && k0 > q0 + 31)) tile(kt % NBUF, k0);
    if (kt + 1 < ntiles) {
      if (NBUF == 1) __syncthreads();                // everyone has read the tile
      stash((kt + 1) % NBUF);                        // NBUF 2: last read before the previous barrier
      __syncthreads();
    }
  }

  // the lane's coordinates anew: the key loop then keeps no registers for them
  int ln = 0;
  asm volatile("" : "+v"(ln));
  ln = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, ln));
  const int el = ln & 31, eh = ln >> 5, eq0 = __builtin_amdgcn_readfirstlane(q0), eq = eq0 + el;

  // ---- again in fp32: each wave its 32 queries, 32 keys at a time, operands from memory.  k-steps pair
  // dims d and d + 4 (dh % 4 == 0), keys key and key + 4. ----
  if (odd) odd_flag = 1;
  __syncthreads();
  if (odd_flag != 0 && eq0 < p.sq) {
#pragma unroll
    for (int d = 0; d < DT; ++d)
#pragma unroll
      for (int e = 0; e < 16; ++e) oacc[d][e] = 0.f;
    base = lrun = 0.f;
    bool fresh = true;                               // no score above -infinity yet
    const float* const qr = qb + static_cast<int64_t>(eq < p.sq ? eq : p.sq - 1) * p.q_ss;
    const int kw = CAUSAL && eq0 + 32 < kend ? eq0 + 32 : kend;
    for (int k0 = 0; k0 < kw; k0 += 32) {
      f32x16 s;
#pragma unroll
      for (int e = 0; e < 16; ++e) s[e] = 0.f;
      const int krow = k0 + el < p.skv ? k0 + el : p.skv - 1;       // past the last: masked below
      const float* const kr = kb + static_cast<int64_t>(krow) * p.k_ss;
      for (int d0 = 0; d0 < dh; d0 += 8) {
        f32x4 kv = {0.f, 0.f, 0.f, 0.f}, qv = kv;
        if (d0 + 4 * eh < dh) {
          kv = *reinterpret_cast<const f32x4*>(kr + d0 + 4 * eh);
          qv = *reinterpret_cast<const f32x4*>(qr + d0 + 4 * eh);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) s = __builtin_amdgcn_mfma_f32_32x32x2f32(kv[e], qv[e], s, 0, 0, 0);
      }
      float bm = -INFINITY;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int key = k0 + (r >> 2) * 8 + 4 * eh + (r & 3);
        if (key >= p.skv || (CAUSAL && key > eq)) s[r] = -INFINITY;
        bm = __builtin_fmaxf(bm, s[r]);
      }
      bm *= c;
      bm = __builtin_fmaxf(bm, __shfl_xor(bm, 32, 64));
      const bool up = (fresh || bm > base) && bm > -INFINITY;
      const float nbase = up ? bm : base;
      const float alpha = fresh ? 1.0f : __builtin_amdgcn_exp2f(base - nbase);
#pragma unroll
      for (int d = 0; d < DT; ++d) oacc[d] *= alpha;
      base = nbase;
      fresh = fresh && !up;
      float l0 = 0.f, l1 = 0.f;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float pr = __builtin_amdgcn_exp2f(__builtin_fmaf(s[r], c, -base));
        if (r & 1) l1 += pr;
        else l0 += pr;
        const int key = k0 + (r >> 2) * 8 + 4 * eh + (r & 3);
        const float* const vr = vb + static_cast<int64_t>(key < p.skv ? key : p.skv - 1) * p.v_ss;
#pragma unroll
        for (int d = 0; d < DT; ++d) {
          const float v = key < p.skv && 32 * d + el < dh ? vr[32 * d + el] : 0.f;
          oacc[d] = __builtin_amdgcn_mfma_f32_32x32x2f32(v, pr, oacc[d], 0, 0, 0);
        }
      }
      lrun = lrun * alpha + (l0 + l1);
    }
  }

  // ---- O = (O^T / l)^T: lane holds query el, dims 32 d + 8 (r / 4) + 4 eh + r % 4 ----
  const float lt = lrun + __shfl_xor(lrun, 32, 64);
  if (eq < p.sq) {
    float* const orow = ob + static_cast<int64_t>(eq) * p.o_ss;
    const float inv = lt > 0.f ? 1.0f / lt : (lt == 0.f ? 0.f : lt);      // NaN stays NaN
#pragma unroll
    for (int d = 0; d < DT; ++d)
#pragma unroll
      for (int g4 = 0; g4 < 4; ++g4) {
        const int col = 32 * d + 8 * g4 + 4 * eh;
        if (col < dh) {                              // dh % 4 == 0: whole groups of 4
          const f32x4 v = {oacc[d][4 * g4] * inv, oacc[d][4 * g4 + 1] * inv, oacc[d][4 * g4 + 2] * inv,
                           oacc[d][4 * g4 + 3] * inv};
          __builtin_memcpy(orow + col, &v, 16);      // output rows at element alignment
        }
      }
  }
}

template <int DHP>
int32_t launch_s32(AttnParams p, hipStream_t st) {
  p.q_tiles = static_cast<int>(cdiv(p.sq, 128));
  const int64_t blocks = static_cast<int64_t>(p.nb) * p.heads * p.q_tiles;
  if (blocks >= 0x7fffffffll) return set_error(WC_ERR_LIMIT, "wc_attention: too many tiles");
  auto kernel = p.causal ? attn_stream32_kernel<DHP, true> : attn_stream32_kernel<DHP, false>;
  kernel<<<dim3(static_cast<uint32_t>(blocks)), dim3(kS32Threads), 0, st>>>(p);
  return check_launch("wc_attention");
}

}  // namespace

int32_t attn_stream32(const AttnParams& p, hipStream_t st) {
  // a scale of 2^30 could lift what the planes lose of a score (kPlaneSafe) to what counts
  if (p.dh % 4 != 0 || p.dh > 64 || p.mask || !(p.scale_log2 > 0.f && p.scale_log2 < 0x1p30f)) return 1;
  return p.dh <= 32 ? launch_s32<32>(p, st) : launch_s32<64>(p, st);
}

}  // namespace wc
