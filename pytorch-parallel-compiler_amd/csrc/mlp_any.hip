// Two chained per-model Linear layers in one launch (the contract of mlp.hip's wc_mlp2) for any
// widths and alignments, fp32, bf16 and fp16.
//
// A workgroup of eight waves owns 16 rows of one model, or 32 once 32-row workgroups cover the
// compute units (a weight fragment then feeds two MFMAs).  Its x rows and h stay in LDS, zero-padded
// to whole 32-wide k-steps; the weights go from memory straight into MFMA operands, 8 consecutive k
// values per lane at element alignment, because a workgroup uses each of them once: wave w computes
// the 16-column tiles w, w + 8, ... of a layer, its next 128 (fp32) or 256 (16-bit) k values of weights
// in flight while the current ones are multiplied, and the second layer's first ones are requested
// before the first layer starts.  Rows of LDS are 16 bytes longer than a multiple of 64, so that 16
// rows' fragment reads cover all banks.
//
// Each lane ends with 4 consecutive columns of one row (the weights are the MFMA's first operand).
// h is rounded to the element type, as a separate first layer would store it.  fp32 uses the fp32 MFMA.
// What bounds it: the latency of its loads, and for wide layers their layout, 16 rows of weights to a
// load instruction, which takes the address unit 64 cycles (15 bytes a cycle and compute unit).
// Whole-line loads through LDS bring 512-wide layers in 1.2-1.4 times faster, but took 1.3-1.6
// times longer at widths that are no multiple of the block; the rule below keeps such sizes on the GEMMs.
// Measured (us for a whole traced forward, host included; models x rows, widths; before: two GEMMs):
//   fp32    8 x 4    176 ->  48 ->  16   28.6 -> 9.8
//   fp32  100 x 2     82 ->  96 ->  16   28.4 -> 10.0
//   fp32  100 x 32    64 -> 300 ->  64   28.8 -> 10.3
//   fp32  128 x 16   256 -> 256 -> 256   28.7 -> 19.5
//   bf16   45 x 108   32 -> 208 ->  31   28.8 -> 9.1
// The GPU's part alone: 8.1 -> 4.8, 8.3 -> 5.3, 13.1 -> 9.8, 22.5 -> 19.7, 13.0 -> 7.8.
#include "wc_common.h"

namespace wc {
namespace {

constexpr int kAnyThreads = 512, kAnyWaves = kAnyThreads / 64;
constexpr int kAnyLds = 160 * 1024;

struct MlpAnyParams {
  int n, m, in, hid, out;
  int act1, act2;
  int pitch1, pitch2;                            // bytes per LDS row of x and of h
  int row_blocks;
  const void* x;
  int64_t x_sn, x_so, x_si;
  FastDiv x_ri;
  const void* w1;
  const void* b1;
  const void* w2;
  const void* b2;
  void* y;
  int64_t y_sn, y_so, y_si;
  FastDiv y_ri;
};

template <typename T> struct AnyFrag { uint4 v[sizeof(T) / 2]; };      // 8 consecutive k values of a row

template <typename T>
__device__ __forceinline__ f32x4 any_mma(const AnyFrag<T>& w, const AnyFrag<T>& a, f32x4 acc) {
  if constexpr (sizeof(T) == 4) {
    float wv[8], av[8];
    __builtin_memcpy(wv, &w, 32);
    __builtin_memcpy(av, &a, 32);
#pragma unroll
    for (int s = 0; s < 8; ++s) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[s], av[s], acc, 0, 0, 0);
    return acc;
  } else {
    return mma16<T>(__builtin_bit_cast(bf16x8, w.v[0]), __builtin_bit_cast(bf16x8, a.v[0]), acc);
  }
}

// 8 values from src, those past `left` zero
template <typename T>
__device__ __forceinline__ AnyFrag<T> any_load(const T* src, int left) {
  AnyFrag<T> f;
  if (left >= 8) {
    __builtin_memcpy(&f, src, sizeof(f));
  } else {
    T t[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) t[e] = e < left ? src[e] : from_f32<T>(0.f);
    __builtin_memcpy(&f, t, sizeof(f));
  }
  return f;
}

// k-steps of 32 that a wave multiplies at a time, and the k values they cover
template <typename T> struct AnyCfg { static constexpr int U = sizeof(T) == 4 ? 4 : 8, BK = 32 * U; };

// A layer's weights [cols][k]; `avail`: elements from w to the end of the whole tensor (at least 8).
template <typename T> struct AnyW { const T* w; int cols, k, avail; };

// A lane's 8 values of row j * 16 + lane % 16 for the k-steps of block kb.  Loads are unconditional (a
// branch around them would have the wave wait where it joins): a unit that crosses the end of its
// row reads on into the next (any_trim clears that), and one that would cross the end of the tensor
// is moved back to end there.
template <typename T>
__device__ __forceinline__ void any_fetch(AnyFrag<T> (&f)[AnyCfg<T>::U], const AnyW<T>& w, int j, int kb) {
  const int lane = threadIdx.x & 63, g8 = (lane >> 4) * 8;
  const int row = min(j * 16 + (lane & 15), w.cols - 1);     // columns past the last repeat it (dropped)
  const int at = row * w.k + kb + g8;
#pragma unroll
  for (int u = 0; u < AnyCfg<T>::U; ++u)
    __builtin_memcpy(&f[u], w.w + static_cast<uint32_t>(min(at + 32 * u, w.avail - 8)), sizeof(f[u]));
}

// The unit at k-step kk: values past the row's end become zero, a unit that was moved back is put right.
template <typename T>
__device__ __forceinline__ void any_trim(AnyFrag<T>& f, const AnyW<T>& w, int j, int kk) {
  using E = typename std::conditional<sizeof(T) == 4, uint32_t, uint16_t>::type;
  const int lane = threadIdx.x & 63, g8 = (lane >> 4) * 8;
  const int row = min(j * 16 + (lane & 15), w.cols - 1);
  const int back = max(row * w.k + kk + g8 + 8 - w.avail, 0); // places it was moved back
  const int left = w.k - kk - g8;                             // its values that exist
  E t[8];
  __builtin_memcpy(t, &f, sizeof(t));
  if (__builtin_amdgcn_ballot_w64(back > 0) != 0) {
#pragma unroll
    for (int s = 4; s > 0; s >>= 1)
#pragma unroll
      for (int e = 0; e + s < 8; ++e) t[e] = (back & s) ? t[e + s] : t[e];
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) t[e] = e < left ? t[e] : E(0);
  __builtin_memcpy(&f, t, sizeof(t));
}

// The wave's column tiles of a[rows][k] (LDS) x w^T; `cur` holds the first tile's first weights.
// sink(j, rb, acc) takes columns 16 j + 4 (lane / 16) + (0 .. 3) of row 16 rb + lane % 16.
template <typename T, int RB, typename Sink>
__device__ __forceinline__ void any_layer(const char* a, int pitch, const AnyW<T>& w, AnyFrag<T> (&cur)[AnyCfg<T>::U],
                                          Sink sink) {
  constexpr int U = AnyCfg<T>::U, BK = AnyCfg<T>::BK;
  const int lane = threadIdx.x & 63;
  const int tiles = (w.cols + 15) >> 4, k = w.k;
  int j = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6), kb = 0;
  if (j >= tiles) return;
  const char* const ab = a + (lane & 15) * pitch + (lane >> 4) * 8 * static_cast<int>(sizeof(T));
  f32x4 acc[RB][2];                              // two chains: even and odd k-steps
  auto clear = [&]() {
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) acc[rb][0] = acc[rb][1] = f32x4{0.f, 0.f, 0.f, 0.f};
  };
  clear();
  // multiplies `f` while `next` is loaded; false after the last tile
  auto step = [&](AnyFrag<T> (&f)[U], AnyFrag<T> (&next)[U]) {
    const bool last = kb + BK >= k;
    const int nj = last ? j + kAnyWaves : j, nk = last ? 0 : kb + BK;
    any_fetch<T>(next, w, nj, nk);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (kb + 32 * u >= k) break;
      if (kb + 32 * u + 32 > k) any_trim<T>(f[u], w, j, kb + 32 * u);
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {
        AnyFrag<T> av;
        const char* const src = ab + rb * 16 * pitch + (kb + 32 * u) * static_cast<int>(sizeof(T));
        __builtin_memcpy(&av, __builtin_assume_aligned(src, 16), sizeof(av));
        acc[rb][u & 1] = any_mma<T>(f[u], av, acc[rb][u & 1]);
      }
    }
    if (last) {
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) sink(j, rb, acc[rb][0] + acc[rb][1]);
      clear();
    }
    j = nj;
    kb = nk;
    return j < tiles;
  };
  AnyFrag<T> other[U];
  while (step(cur, other) && step(other, cur)) {
  }
}

template <typename T, int RB>
__global__ __launch_bounds__(kAnyThreads) void mlp2_any_kernel(MlpAnyParams p) {
  constexpr int ROWS = 16 * RB, U = AnyCfg<T>::U;
  extern __shared__ __attribute__((aligned(16))) char any_smem[];
  char* const xs = any_smem;                                     // [ROWS][pitch1]
  char* const hs = xs + ROWS * p.pitch1;                         // [ROWS][pitch2]
  float* const bs1 = reinterpret_cast<float*>(hs + ROWS * p.pitch2);
  const int cp1 = (p.hid + 15) & ~15, cp2 = (p.out + 15) & ~15;
  float* const bs2 = bs1 + cp1;

  // a model's row blocks run on one XCD, whose L2 then serves its weights
  int blk = static_cast<int>(blockIdx.x);
  if ((gridDim.x & 7) == 0) blk = (blk & 7) * static_cast<int>(gridDim.x >> 3) + (blk >> 3);
  const int mdl = blk / p.row_blocks;
  const int m0 = (blk - mdl * p.row_blocks) * ROWS;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int fr = lane & 15, g4 = (lane >> 4) * 4;

  const int64_t s1 = static_cast<int64_t>(p.hid) * p.in, s2 = static_cast<int64_t>(p.out) * p.hid;
  auto avail = [&](int64_t s) { return static_cast<int>(min((p.n - mdl) * s, static_cast<int64_t>(1) << 30)); };
  const AnyW<T> w1 = {static_cast<const T*>(p.w1) + mdl * s1, p.hid, p.in, avail(s1)};
  const AnyW<T> w2 = {static_cast<const T*>(p.w2) + mdl * s2, p.out, p.hid, avail(s2)};
  AnyFrag<T> f1[U], f2[U];
  any_fetch<T>(f1, w1, wave, 0);

  // ---- x rows (rows past the last are zero), biases, the columns of h that pad its last k-step ----
  {
    const T* const b1 = p.b1 ? static_cast<const T*>(p.b1) + static_cast<int64_t>(mdl) * p.hid : nullptr;
    const T* const b2 = p.b2 ? static_cast<const T*>(p.b2) + static_cast<int64_t>(mdl) * p.out : nullptr;
    auto bias = [](const T* b, int e, int cols) { return b && e < cols ? to_f32(b[e]) : 0.f; };
    const float bv1 = bias(b1, tid, p.hid), bv2 = bias(b2, tid, p.out);
    const T* const xb = static_cast<const T*>(p.x) + static_cast<int64_t>(mdl) * p.x_sn;
    const int upr = ((p.in + 31) & ~31) / 8;                     // units of 8 values per row
    for (int e = tid; e < ROWS * upr; e += kAnyThreads) {
      const int r = e / upr, c = (e - r * upr) * 8;
      AnyFrag<T> v = any_load<T>(xb, 0);
      if (m0 + r < p.m && c < p.in) {
        const uint32_t gm = static_cast<uint32_t>(m0 + r);
        const uint32_t outer = fdiv(gm, p.x_ri);
        v = any_load<T>(xb + static_cast<int64_t>(outer) * p.x_so +
                            static_cast<int64_t>(gm - outer * p.x_ri.d) * p.x_si + c, p.in - c);
      }
      __builtin_memcpy(__builtin_assume_aligned(xs + r * p.pitch1 + c * sizeof(T), 16), &v, sizeof(v));
    }
    for (int e = tid; e < cp1; e += kAnyThreads) bs1[e] = e == tid ? bv1 : bias(b1, e, p.hid);
    for (int e = tid; e < cp2; e += kAnyThreads) bs2[e] = e == tid ? bv2 : bias(b2, e, p.out);
    if (cp1 & 16)
      for (int e = tid; e < ROWS * 16; e += kAnyThreads)
        reinterpret_cast<T*>(hs + (e >> 4) * p.pitch2)[cp1 + (e & 15)] = from_f32<T>(0.f);
  }
  any_fetch<T>(f2, w2, wave, 0);
  __syncthreads();

  // ---- h = act1(x W1^T + b1), to LDS ----
  any_layer<T, RB>(xs, p.pitch1, w1, f1, [&](int j, int rb, f32x4 acc) {
    const int col = 16 * j + g4;
    T o[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float v = acc[e] + bs1[col + e];
      if (p.act1 == WC_ACT_RELU) v = fmaxf(v, 0.f);
      o[e] = from_f32<T>(col + e < p.hid ? v : 0.f);
    }
    __builtin_memcpy(__builtin_assume_aligned(hs + (16 * rb + fr) * p.pitch2 + col * sizeof(T), 4 * sizeof(T)), o,
                     sizeof(o));
  });
  __syncthreads();

  // ---- y = act2(h W2^T + b2) ----
  T* yrow[RB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    const int gm = min(m0 + 16 * rb + fr, p.m - 1);
    const uint32_t outer = fdiv(static_cast<uint32_t>(gm), p.y_ri);
    yrow[rb] = static_cast<T*>(p.y) + static_cast<int64_t>(mdl) * p.y_sn + static_cast<int64_t>(outer) * p.y_so +
               static_cast<int64_t>(gm - outer * p.y_ri.d) * p.y_si;
  }
  any_layer<T, RB>(hs, p.pitch2, w2, f2, [&](int j, int rb, f32x4 acc) {
    const int col = 16 * j + g4;
    if (m0 + 16 * rb + fr >= p.m) return;
    T o[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float v = acc[e] + bs2[col + e];
      if (p.act2 == WC_ACT_RELU) v = fmaxf(v, 0.f);
      o[e] = from_f32<T>(v);
    }
    if (col + 4 <= p.out) {
      __builtin_memcpy(yrow[rb] + col, o, sizeof(o));            // element alignment
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (col + e < p.out) yrow[rb][col + e] = o[e];
    }
  });
}

inline int any_pitch(int es, int64_t k) { return static_cast<int>((k + 31) / 32 * 32) * es + 16; }

inline int64_t any_lds(int es, int rows, int64_t in, int64_t hid, int64_t out) {
  return static_cast<int64_t>(rows) * (any_pitch(es, in) + any_pitch(es, hid)) +
          4 * ((hid + 15) / 16 + (out + 15) / 16) * 16;
}

// a whole 8-value unit must exist in either weight tensor
inline bool any_weights(int64_t in, int64_t hid, int64_t out) { return in * hid >= 8 && hid * out >= 8; }

// rows per workgroup: 32 once 32-row workgroups cover the compute units
inline int any_rows(int es, int64_t n, int64_t m, int64_t in, int64_t hid, int64_t out, int cus) {
  return mul_sat({n, cdiv(m, 32)}) >= cus && any_lds(es, 32, in, hid, out) <= kAnyLds ? 32 : 16;
}

template <typename T, int RB>
int32_t launch_any(const MlpAnyParams& p, uint32_t blocks, size_t lds, hipStream_t st) {
  auto kern = mlp2_any_kernel<T, RB>;
  if (lds > 64 * 1024) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
    if (e != hipSuccess)
      return set_error(static_cast<int32_t>(e), "wc_mlp2_any: LDS of %zu bytes refused: %s", lds, hipGetErrorString(e));
  }
  kern<<<dim3(blocks), dim3(kAnyThreads), lds, st>>>(p);
  return check_launch("wc_mlp2_any");
}

}  // namespace
}  // namespace wc

using namespace wc;

// Where one launch pays.  A workgroup takes about 3 us and 2 for each block of weights (8 waves x 16
// columns x BK values of k), in as many rounds as there are workgroups for the compute units; two GEMM
// launches take 28 us or more of host time, and spread a model's columns over the chip.  Measured on both
// sides of the line (us; one launch / two): 128 x 16 rows of 256 -> 256 -> 256, estimate 19: 19.5 / 28.7;
// 32 x 64 of 256 -> 512 -> 256, estimate 35: 33.2 / 28.7; 128 x 256 of 64 -> 96 -> 100, estimate 28:
// 29.3 / 28.9.
extern "C" int32_t wc_mlp2_any_supported(int32_t dtype, int64_t n, int64_t m, int64_t in_features, int64_t hidden,
                                         int64_t out_features) {
  const int es = dtype_size(dtype);
  if (es == 0 || n <= 0 || m <= 0 || in_features <= 0 || hidden <= 0 || out_features <= 0) return 0;
  if (in_features > 4096 || hidden > 4096 || out_features > 4096 || n >= 0x7fffffffll || m >= 0x7fffffffll) return 0;
  if (any_lds(es, 16, in_features, hidden, out_features) > kAnyLds || !any_weights(in_features, hidden, out_features))
    return 0;
  int cus = device_cu_count();
  if (cus <= 0) cus = 256;
  const int rows = any_rows(es, n, m, in_features, hidden, out_features, cus);
  const int64_t blocks = mul_sat({n, cdiv(m, rows)});
  const int bk = es == 4 ? AnyCfg<float>::BK : AnyCfg<bf16>::BK;
  auto steps = [&](int64_t k, int64_t cols) { return static_cast<double>(cdiv(cols, 16 * kAnyWaves) * cdiv(k, bk)); };
  const double rounds = blocks > cus ? static_cast<double>(blocks) / cus : 1.0;
  return rounds * (3.0 + 2.0 * (steps(in_features, hidden) + steps(hidden, out_features))) <= 20.0 ? 1 : 0;
}

extern "C" int32_t wc_mlp2_any(const wc_mlp2_args* a, void* stream) {
  clear_error();
  WC_REQUIRE(a != nullptr, WC_ERR_NULL, "wc_mlp2_any: null args");
  const int es = dtype_size(a->dtype);
  WC_REQUIRE(es != 0, WC_ERR_DTYPE, "wc_mlp2_any: unsupported dtype %d", a->dtype);
  WC_REQUIRE(a->n >= 0 && a->m >= 0 && a->in_features > 0 && a->hidden > 0 && a->out_features > 0, WC_ERR_SHAPE,
             "wc_mlp2_any: bad size");
  WC_REQUIRE(a->in_features <= 4096 && a->hidden <= 4096 && a->out_features <= 4096 &&
                 any_lds(es, 16, a->in_features, a->hidden, a->out_features) <= kAnyLds &&
                 any_weights(a->in_features, a->hidden, a->out_features),
             WC_ERR_LIMIT, "wc_mlp2_any: sizes %lld -> %lld -> %lld (%s) not supported", (long long)a->in_features,
             (long long)a->hidden, (long long)a->out_features, dtype_name(a->dtype));
  WC_REQUIRE(a->act1 == WC_ACT_NONE || a->act1 == WC_ACT_RELU, WC_ERR_ARG, "wc_mlp2_any: bad act1");
  WC_REQUIRE(a->act2 == WC_ACT_NONE || a->act2 == WC_ACT_RELU, WC_ERR_ARG, "wc_mlp2_any: bad act2");
  if (a->n == 0 || a->m == 0) return WC_OK;
  WC_REQUIRE(a->x && a->w1 && a->w2 && a->y, WC_ERR_NULL, "wc_mlp2_any: null pointer");
  WC_REQUIRE(a->x_rows_inner > 0 && a->y_rows_inner > 0, WC_ERR_ARG, "wc_mlp2_any: rows_inner must be positive");
  WC_REQUIRE(a->x_rows_inner < 0x7fffffffll && a->y_rows_inner < 0x7fffffffll && a->m < 0x7fffffffll &&
                 a->n < 0x7fffffffll, WC_ERR_LIMIT, "wc_mlp2_any: sizes too large");
  WC_REQUIRE(aligned(a->x, es) && aligned(a->w1, es) && aligned(a->w2, es) && aligned(a->y, es) &&
                 (!a->b1 || aligned(a->b1, es)) && (!a->b2 || aligned(a->b2, es)),
             WC_ERR_ALIGN, "wc_mlp2_any: pointers must be aligned to the element size");
  MlpAnyParams p;
  p.n = (int)a->n;
  p.m = (int)a->m;
  p.in = (int)a->in_features;
  p.hid = (int)a->hidden;
  p.out = (int)a->out_features;
  p.act1 = a->act1;
  p.act2 = a->act2;
  p.pitch1 = any_pitch(es, p.in);
  p.pitch2 = any_pitch(es, p.hid);
  p.x = a->x;
  p.x_sn = a->x_stride_n;
  p.x_so = a->x_stride_outer;
  p.x_si = a->x_stride_inner;
  p.x_ri = make_fastdiv(static_cast<uint32_t>(a->x_rows_inner));
  p.w1 = a->w1;
  p.b1 = a->b1;
  p.w2 = a->w2;
  p.b2 = a->b2;
  p.y = a->y;
  p.y_sn = a->y_stride_n;
  p.y_so = a->y_stride_outer;
  p.y_si = a->y_stride_inner;
  p.y_ri = make_fastdiv(static_cast<uint32_t>(a->y_rows_inner));
  const int rows = any_rows(es, a->n, a->m, p.in, p.hid, p.out, device_cu_count());
  p.row_blocks = static_cast<int>(cdiv(p.m, rows));
  const int64_t blocks = a->n * p.row_blocks;
  WC_REQUIRE(blocks < 0x7fffffffll, WC_ERR_LIMIT, "wc_mlp2_any: too many workgroups");
  const size_t lds = static_cast<size_t>(any_lds(es, rows, p.in, p.hid, p.out));
  hipStream_t st = as_stream(stream);
  const uint32_t nb = static_cast<uint32_t>(blocks);
  if (a->dtype == WC_F32) return rows == 32 ? launch_any<float, 2>(p, nb, lds, st) : launch_any<float, 1>(p, nb, lds, st);
  if (a->dtype == WC_F16) return rows == 32 ? launch_any<f16, 2>(p, nb, lds, st) : launch_any<f16, 1>(p, nb, lds, st);
  return rows == 32 ? launch_any<bf16, 2>(p, nb, lds, st) : launch_any<bf16, 1>(p, nb, lds, st);
}
