// Partitioned persistent recurrence in fp32: LSTM and GRU, hidden sizes above 128 up to 384 that
// are a multiple of 32.
//
// W_hh of one model (G x H fp32, 1 MB for an LSTM at H = 256) exceeds a compute unit's registers,
// so P = H / (16 TPW) workgroups share a unit of (model, up to 16 batch rows), one per compute
// unit, for all T steps.  A workgroup owns 16 TPW hidden units and holds the rows of W_hh of
// their gates in registers for the whole sequence, split into three bf16 planes
// (v = v0 + v1 + v2; the products of at most second order in fp32, as in the tile GEMM).
//
// Per step: gates = h_{t-1} W_hh^T as 16x16x32 MFMAs (A = W_hh planes, B = h planes from LDS),
// the cell update in registers (the fp32 state never leaves the chip), h_t into its place in the
// output, a flag per workgroup, and once all P flags of the unit show step t, the whole h_t row
// back from the output through L2 into LDS planes.
//
// Lane layout (wave w of 4, lane = 16 g + fr): row rho of MFMA tile j is gate slot rho & 3 of unit
// 4 TPW w + TPW (rho >> 2) + j, so lane (g, fr) accumulates the four gate slots of unit
// 4 TPW w + TPW g + j for batch row fr and the cell update needs no lane exchange.  GRU slots are
// r, z, n and a fourth that repeats n's rows and whose result is never read.
//
// Exchange.  When all parts of a unit run on one XCD (HW_REG_XCC_ID, compared at the start)
// the h_t stores and the flag are plain: they write through the L1 into that XCD's L2, in order
// (the stores' vmcnt, then a barrier, then the flag), and the readers' device-scope loads find
// them there.  Otherwise stores are device-scope and an agent release precedes the flag.  Flags
// and XCD entries are zeroed by a small kernel before each launch.  Every wait is bounded: past
// the limit (poll rounds) the workgroup records 1 in the status word and leaves, and its outputs
// are invalid.  The host launches the grid cooperatively (all workgroups co-resident, or the
// launch fails); a captured stream takes the one-launch-per-step kernel instead.
//
// What the planes do not carry: a workgroup whose W_hh rows, or a step whose h, hold a value of 2^56 or more
// (kPlaneSafe) or an infinity computes its gates with fp32 multiply-adds from memory instead.  Below it no gate
// sum overflows, and what the planes lose of a value under 2^-110 stays 2^-60 of a gate's range.  (An infinite
// weight in every model: LSTM 16 x 16 x 64 x 256 whole forward 1,090 us against 222; per-step launches 625.)
//
// Bound by the step's serial chain: MFMAs (and the LDS reads that feed them), the store, flag and
// load latencies of the exchange.  Measured (us; before: one launch per step, streaming W_hh):
//   LSTM 16 models x 16 rows x 64 steps x 256    559 -> 165  (2.3 per step and a launch of 20)
//   LSTM 64 x 16 x 32 x 256                      555 -> 229
//   GRU  16 x 16 x 64 x 256                      746 -> 162
//   GRU  32 x 8 x 32 x 384                       497 -> 277
#include <type_traits>

#include "wc_rnn.h"

namespace wc {
namespace {

constexpr int kThreads = 256;
constexpr int kSyncInts = 64;          // one 256-byte block per unit:
constexpr int kSyncStatus = 31;        //   [0, 31): steps finished, per part; status (unit 0's)
constexpr int kSyncXcc = 32;           //   [32, 64): XCD + 1, per part
constexpr int kSc1 = 16;               // buffer-op cache policy: device scope

struct P32Params {
  int rows, chunks, unit0, units, steps, hid, parts, spin_limit;   // units: of this launch
  const float* gx;       // [n, rows, steps, G]: x W_ih^T + b_ih
  const float* w_hh;     // [n, G, H]
  const float* b_hh;     // [n, G] or null
  const float* h0;       // [n, rows, H] or null
  const float* c0;       // LSTM: [n, rows, H] or null
  float* out;            // [n, rows, steps, H]
  float* hn;             // [n, rows, H] or null
  float* cn;             // LSTM: [n, rows, H] or null
  int* sync;             // [units][kSyncInts]
  int* status;           // set to 1 when a wait gave up
};

__device__ __forceinline__ int sync_load(const int* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void sync_store(int* p, int v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// 8 floats as planes; true when one is kPlaneSafe or more (NaN stays NaN in the planes)
__device__ __forceinline__ bool split8(const float (&v)[8], bf16x8 (&pl)[3]) {
  bool big = false;
#pragma unroll
  for (int e = 0; e < 8; ++e) big |= __builtin_fabsf(v[e]) >= kPlaneSafe;
  uint4 u[3];
  split_planes(v, u);
#pragma unroll
  for (int q = 0; q < 3; ++q) pl[q] = __builtin_bit_cast(bf16x8, u[q]);
  return big;
}

template <int KS, int TPW, int CELL>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(1, 1)))
void part32_kernel(P32Params p) {
  constexpr bool GRU = CELL == WC_CELL_GRU;
  constexpr int NG = GRU ? 3 : 4;
  constexpr int UP = 16 * TPW;                       // hidden units per workgroup
  constexpr int K = KS * 32, HP = K + 8;             // padded k, LDS pitch of an h row (bf16 elements)
  constexpr int NA = 6 / TPW;                        // accumulator chains per tile
  constexpr int NU = 16 * K / 8;                     // 8-value pieces of an h block
  constexpr int UPT = (NU + kThreads - 1) / kThreads;
  __shared__ __attribute__((aligned(16))) uint16_t hs[3][16 * HP];
  __shared__ int flags[4];                           // abort, W_hh not carried, h not carried (by step parity)

  const int H = p.hid, G = NG * H, P = p.parts;
  // workgroups go to the 8 XCDs in turn: a unit's parts take consecutive places of one XCD
  const int slot_x = blockIdx.x >> 3;
  const int lu = (slot_x / P) * 8 + (blockIdx.x & 7), part = slot_x % P;
  if (lu >= p.units) return;                         // padding of the last round of units
  const int unit = p.unit0 + lu;
  const int mdl = unit / p.chunks, chk = unit - mdl * p.chunks;
  const int row0 = chk * 16;
  const int nrows = p.rows - row0 < 16 ? p.rows - row0 : 16;
  const int64_t mb = static_cast<int64_t>(mdl) * p.rows + row0;
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63, g = lane >> 4, fr = lane & 15;
  const int ul = part * UP + w * 4 * TPW + g * TPW;  // the lane's first unit
  const bool brow = fr < nrows;
  const int64_t wrow0 = static_cast<int64_t>(mdl) * G;
  int* const my_sync = p.sync + static_cast<int64_t>(unit) * kSyncInts;

  if (tid < 4) flags[tid] = 0;
  __syncthreads();

  // ---- W_hh rows of this workgroup's units, as planes ----
  bf16x8 wp[KS][TPW][3];
  {
    bool bad = false;
    const int slot = GRU && (fr & 3) == 3 ? 2 : (fr & 3);
#pragma unroll
    for (int j = 0; j < TPW; ++j) {
      const int u = part * UP + w * 4 * TPW + (fr >> 2) * TPW + j;
      const float* row = p.w_hh + (wrow0 + static_cast<int64_t>(slot) * H + u) * H + g * 8;
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = 0.f;
        if (32 * s < H) __builtin_memcpy(v, __builtin_assume_aligned(row + 32 * s, 16), 32);
        bad |= split8(v, wp[s][j]);
      }
    }
    if (bad) flags[1] = 1;
  }
  // ---- h_{-1} planes into LDS (rows >= nrows and columns >= H stay zero) ----
  {
    bool bad = false;
#pragma unroll
    for (int q = 0; q < UPT; ++q) {
      const int e = tid + q * kThreads;
      if (e >= NU) continue;
      const int b = e / (K / 8), c = (e - b * (K / 8)) * 8;
      float v[8];
#pragma unroll
      for (int z = 0; z < 8; ++z) v[z] = 0.f;
      if (p.h0 && b < nrows && c < H) __builtin_memcpy(v, __builtin_assume_aligned(p.h0 + (mb + b) * H + c, 16), 32);
      bf16x8 pl[3];
      bad |= split8(v, pl);
#pragma unroll
      for (int z = 0; z < 3; ++z) *reinterpret_cast<bf16x8*>(&hs[z][b * HP + c]) = pl[z];
    }
    if (bad) flags[2] = 1;
  }
  // ---- state, recurrent bias, gates_x of step 0 ----
  float st[TPW], bh[TPW][NG];
#pragma unroll
  for (int j = 0; j < TPW; ++j) {
    const float* s0 = GRU ? p.h0 : p.c0;
    st[j] = s0 && brow ? s0[(mb + fr) * H + ul + j] : 0.f;
#pragma unroll
    for (int q = 0; q < NG; ++q) bh[j][q] = p.b_hh ? p.b_hh[wrow0 + static_cast<int64_t>(q) * H + ul + j] : 0.f;
  }
  const __amdgpu_buffer_rsrc_t ors = __builtin_amdgcn_make_buffer_rsrc(
      p.out + mb * p.steps * H, 0, static_cast<int>(static_cast<uint32_t>(nrows) * p.steps * H * 4), 0x00020000);
  const float* const gxl = p.gx + ((mb + (brow ? fr : 0)) * p.steps) * G + ul;
  float gxn[TPW][NG];
  auto load_gx = [&](int t) {
#pragma unroll
    for (int q = 0; q < NG; ++q)
#pragma unroll
      for (int j = 0; j < TPW; ++j) gxn[j][q] = gxl[static_cast<int64_t>(t) * G + q * H + j];
  };
  load_gx(0);

  // ---- are all parts of this unit on one XCD? ----
  if (tid == 0) {
    const uint32_t xcc = __builtin_amdgcn_s_getreg((3 << 11) | (0 << 6) | 20) & 0xFu;   // HW_REG_XCC_ID
    sync_store(my_sync + kSyncXcc + part, static_cast<int>(xcc + 1));
  }
  bool ok = true;
  int got = 0;
  if (lane < P) {
    int spins = 0;
    while (true) {
      if (spins++ >= p.spin_limit) {
        ok = false;
        break;
      }
      got = sync_load(my_sync + kSyncXcc + lane);
      if (got != 0) break;
      __builtin_amdgcn_s_sleep(1);
    }
  }
  const int first = __shfl(got, 0, 64);
  const bool local = __all(lane >= P || got == first);
  if (!ok) flags[0] = 1;
  __syncthreads();
  bool aborted = flags[0] != 0;
  const bool badw = flags[1] != 0;

  const uint16_t* const hl = &hs[0][fr * HP + g * 8];
  const uint32_t orow = static_cast<uint32_t>(brow ? fr : 0) * p.steps;
  float hv[TPW];
#pragma unroll
  for (int j = 0; j < TPW; ++j) hv[j] = 0.f;
  for (int t = 0; t < p.steps && !aborted; ++t) {
    // gates_x one step ahead, issued before the MFMAs: loads retire in order, so one issued later
    // would hold up the exchange's polls
    float gxv[TPW][NG];
#pragma unroll
    for (int j = 0; j < TPW; ++j)
#pragma unroll
      for (int q = 0; q < NG; ++q) gxv[j][q] = gxn[j][q];
    if (t + 1 < p.steps) load_gx(t + 1);
    // ---- gates_h = h_{t-1} W_hh^T ----
    float gh[TPW][4];
    if (!(badw || flags[2 + (t & 1)])) {
      f32x4 acc[TPW][NA];
#pragma unroll
      for (int j = 0; j < TPW; ++j)
#pragma unroll
        for (int a = 0; a < NA; ++a) acc[j][a] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        bf16x8 hb[3];
#pragma unroll
        for (int z = 0; z < 3; ++z) hb[z] = *reinterpret_cast<const bf16x8*>(hl + z * 16 * HP + 32 * s);
        // the six products, over independent chains: one per order (TPW = 2) or product (TPW = 1)
#pragma unroll
        for (int order = 0, prod = 0; order < 3; ++order)
#pragma unroll
          for (int a = 0; a <= order; ++a, ++prod)
#pragma unroll
            for (int j = 0; j < TPW; ++j) {
              const int ch = TPW == 2 ? order : prod;
              acc[j][ch] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wp[s][j][order - a], hb[a], acc[j][ch], 0, 0, 0);
            }
      }
#pragma unroll
      for (int j = 0; j < TPW; ++j) {
        f32x4 sum;
        if constexpr (TPW == 2) sum = (acc[j][2] + acc[j][1]) + acc[j][0];
        else sum = ((acc[j][5] + acc[j][4]) + acc[j][3]) + (acc[j][2] + acc[j][1]) + acc[j][0];
#pragma unroll
        for (int q = 0; q < 4; ++q) gh[j][q] = sum[q];
      }
    } else {
#pragma unroll
      for (int j = 0; j < TPW; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) gh[j][q] = 0.f;
      if (t > 0 || p.h0) {
        const float* const h0r = t == 0 ? p.h0 + (mb + (brow ? fr : 0)) * H : nullptr;
        const float* const wr = p.w_hh + (wrow0 + ul) * H;
        for (int k = 0; k < H; k += 4) {
          f32x4 hk;
          if (t == 0) hk = *reinterpret_cast<const f32x4*>(h0r + k);
          else
            hk = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(ors, ((orow + t - 1) * H + k) * 4, 0,
                                                                                 kSc1));
#pragma unroll
          for (int j = 0; j < TPW; ++j)
#pragma unroll
            for (int q = 0; q < NG; ++q) {
              const f32x4 w = *reinterpret_cast<const f32x4*>(wr + (static_cast<int64_t>(q) * H + j) * H + k);
#pragma unroll
              for (int e = 0; e < 4; ++e) gh[j][q] += hk[e] * w[e];
            }
        }
      }
    }
    // ---- cell update of the lane's units ----
#pragma unroll
    for (int j = 0; j < TPW; ++j) {
      if constexpr (GRU) {
        const float rg = sigmoid_f(gxv[j][0] + (gh[j][0] + bh[j][0]));
        const float zg = sigmoid_f(gxv[j][1] + (gh[j][1] + bh[j][1]));
        const float nn = tanh_f(gxv[j][2] + rg * (gh[j][2] + bh[j][2]));
        st[j] = (1.0f - zg) * nn + zg * st[j];
        hv[j] = st[j];
      } else {
        const float ig = sigmoid_f(gxv[j][0] + (gh[j][0] + bh[j][0]));
        const float fg = sigmoid_f(gxv[j][1] + (gh[j][1] + bh[j][1]));
        const float gg = tanh_f(gxv[j][2] + (gh[j][2] + bh[j][2]));
        const float og = sigmoid_f(gxv[j][3] + (gh[j][3] + bh[j][3]));
        st[j] = fg * st[j] + ig * gg;
        hv[j] = og * tanh_f(st[j]);
      }
    }
    // ---- h_t to the output ----
    const uint32_t oo = ((orow + t) * H + ul) * 4;
    if (brow) {
      if constexpr (TPW == 2) {
        const i32x2 v = {__builtin_bit_cast(int, hv[0]), __builtin_bit_cast(int, hv[1])};
        if (local) __builtin_amdgcn_raw_buffer_store_b64(v, ors, oo, 0, 0);
        else __builtin_amdgcn_raw_buffer_store_b64(v, ors, oo, 0, kSc1);
      } else {
        if (local) __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(int, hv[0]), ors, oo, 0, 0);
        else __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(int, hv[0]), ors, oo, 0, kSc1);
      }
    }
    if (t + 1 == p.steps) break;
    // ---- publish: this wave's stores have reached L2, then every wave's, then the flag ----
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();                                 // also: every wave has read h_{t-1}
    if (tid == 0) {
      if (local) {
        __hip_atomic_store(my_sync + part, t + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      } else {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
        sync_store(my_sync + part, t + 1);
      }
      flags[2 + (t & 1)] = 0;                        // set again, if at all, for step t + 2
    }
    // ---- wait for every part's h_t ----
    {
      int spins = 0;
      bool done = lane >= P;
      while (true) {
        if (!done) done = sync_load(my_sync + lane) > t;
        if (__all(done)) break;
        if (spins++ >= p.spin_limit) {
          flags[0] = 1;
          break;
        }
        __builtin_amdgcn_s_sleep(1);
      }
    }
    if (!local) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    asm volatile("" ::: "memory");
    // ---- h_t planes into LDS ----
    {
      i32x4 v[UPT][2];
#pragma unroll
      for (int q = 0; q < UPT; ++q) {
        const int e = tid + q * kThreads;
        const int b = e / (K / 8), c = (e - b * (K / 8)) * 8;
        v[q][0] = i32x4{0, 0, 0, 0};
        v[q][1] = i32x4{0, 0, 0, 0};
        if (e < NU && b < nrows && c < H) {
          const uint32_t off = ((static_cast<uint32_t>(b) * p.steps + t) * H + c) * 4;
          v[q][0] = __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(ors, off, 0, kSc1));
          v[q][1] = __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(ors, off + 16, 0, kSc1));
        }
      }
      bool bad = false;
#pragma unroll
      for (int q = 0; q < UPT; ++q) {
        const int e = tid + q * kThreads;
        const int b = e / (K / 8), c = (e - b * (K / 8)) * 8;
        if (e < NU && b < nrows && c < H) {
          float f[8];
          __builtin_memcpy(f, &v[q], 32);
          bf16x8 pl[3];
          bad |= split8(f, pl);
#pragma unroll
          for (int z = 0; z < 3; ++z) *reinterpret_cast<bf16x8*>(&hs[z][b * HP + c]) = pl[z];
        }
      }
      if (bad) flags[2 + ((t + 1) & 1)] = 1;
    }
    __syncthreads();
    aborted = flags[0] != 0;
  }

  if (aborted) {
    if (tid == 0) sync_store(p.status, 1);
    return;
  }
  if (brow) {
#pragma unroll
    for (int j = 0; j < TPW; ++j) {
      const int64_t so = (mb + fr) * H + ul + j;
      if (p.hn) p.hn[so] = hv[j];
      if (!GRU && p.cn) p.cn[so] = st[j];
    }
  }
}

__global__ void part32_zero_kernel(int* p, int64_t n) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) sync_store(p + i, 0);
}

inline int64_t p32_units(const wc_rnn_args* a) { return a->n * ((a->batch + 15) / 16); }

// units of one launch: as many per XCD as have all their workgroups on compute units of their own
inline int p32_per_launch(int hidden, int tpw, int cus) { return (cus / 8) / (hidden / (16 * tpw)) * 8; }

// Microseconds of the whole recurrence with 16 * tpw hidden units per workgroup: 1 halves the
// MFMAs of a step, 2 the workgroups of a unit.  A launch costs about 20 us (cooperative dispatch,
// loading and splitting W_hh), a step 2.3 or, with two, 2.85 (4.3 past 256 columns, where W_hh
// fills the AGPRs), times the launches that the units need (measured, 16 rows).
inline double p32_cost(const wc_rnn_args* a, int tpw, int cus) {
  const int64_t launches = cdiv(p32_units(a), p32_per_launch(static_cast<int>(a->hidden), tpw, cus));
  const double step = tpw == 1 ? 2.3 : a->hidden <= 256 ? 2.85 : 4.3;
  return static_cast<double>(launches) * (20.0 + step * static_cast<double>(a->steps));
}
inline int p32_tpw(const wc_rnn_args* a, int cus) { return p32_cost(a, 1, cus) <= p32_cost(a, 2, cus) ? 1 : 2; }

// The same for one launch per step: 7 us, or 4 and the time to stream every model's W_hh from
// memory at 5 TB/s, once per 16 batch rows.  Measured (us per step): LSTM 16 models x 256 hidden
// 8.7, 64 models 17.4, with 32 rows 30.8; GRU 32 x 384 15.5; LSTM 64 x 384 29.4.
inline double step_cost(const wc_rnn_args* a) {
  const double bytes = static_cast<double>(a->n) * (a->cell == WC_CELL_GRU ? 3.0 : 4.0) *
                       static_cast<double>(a->hidden) * static_cast<double>(a->hidden) * 4.0;
  const double us = 4.0 + static_cast<double>(cdiv(a->batch, 16)) * bytes / 5.0e6;
  return static_cast<double>(a->steps) * (us < 7.0 ? 7.0 : us);
}

inline int64_t p32_sync_offset(const wc_rnn_args* a) {
  return a->n * a->batch * a->steps * (a->cell == WC_CELL_GRU ? 3 : 4) * a->hidden * 4;
}

template <int KS, int TPW, int CELL>
int32_t launch_p32(P32Params p, int units_total, int cus, hipStream_t st) {
  const void* fn = reinterpret_cast<const void*>(part32_kernel<KS, TPW, CELL>);
  const bool cooperative = part_cooperative();
  const int per_launch = p32_per_launch(p.hid, TPW, cus);
  for (int u = 0; u < units_total; u += per_launch) {
    p.unit0 = u;
    p.units = units_total - u < per_launch ? units_total - u : per_launch;
    const int nwg = (p.units + 7) / 8 * 8 * p.parts;
    if (cooperative) {
      void* args[] = {&p};
      const hipError_t e = hipLaunchCooperativeKernel(fn, dim3(nwg), dim3(kThreads), args, 0, st);
      if (e != hipSuccess)
        return set_error(static_cast<int32_t>(e), "wc_rnn_recurrence: cooperative launch of %d workgroups "
                         "failed: %s", nwg, hipGetErrorString(e));
    } else {
      part32_kernel<KS, TPW, CELL><<<dim3(nwg), dim3(kThreads), 0, st>>>(p);
      const int32_t rc = check_launch("wc_rnn_recurrence(partitioned fp32)");
      if (rc) return rc;
    }
  }
  return WC_OK;
}

template <int CELL>
int32_t p32_dispatch(const P32Params& p, int tpw, int units, int cus, hipStream_t st) {
  const int ks = p.hid <= 192 ? 6 : p.hid <= 256 ? 8 : 12;
  if (ks == 6) return tpw == 1 ? launch_p32<6, 1, CELL>(p, units, cus, st) : launch_p32<6, 2, CELL>(p, units, cus, st);
  if (ks == 8) return tpw == 1 ? launch_p32<8, 1, CELL>(p, units, cus, st) : launch_p32<8, 2, CELL>(p, units, cus, st);
  return tpw == 1 ? launch_p32<12, 1, CELL>(p, units, cus, st) : launch_p32<12, 2, CELL>(p, units, cus, st);
}

}  // namespace

bool part32_plan(const wc_rnn_args* a) {
  if ((a->cell != WC_CELL_LSTM && a->cell != WC_CELL_GRU) || a->dtype != WC_F32 || a->n < 1 || a->batch < 1 ||
      a->steps < 1 || a->hidden <= 128 || a->hidden > 384 || a->hidden % 32 != 0)
    return false;
  const int cus = device_cu_count();
  if (cus <= 0 || p32_per_launch(static_cast<int>(a->hidden), 1, cus) < 8) return false;
  // a unit's block of the output (16 rows) is addressed with 32-bit byte offsets
  if (mul_sat({16, a->steps, a->hidden, 4}) >= 0x7fffffffll || p32_units(a) >= 0x7fffffffll / kSyncInts) return false;
  for (const void* q : {a->w_hh, a->h0, static_cast<const void*>(a->out)})
    if (q && !aligned(q, 16)) return false;
  // short sequences do not earn the launch, and very many units take too many of them (GRU 64
  // models x 2 rows x 8 steps x 160: 80 us against 62)
  return p32_cost(a, p32_tpw(a, cus), cus) <= 0.9 * step_cost(a);
}

int64_t part32_status_offset(const wc_rnn_args* a) { return p32_sync_offset(a) + kSyncStatus * 4; }

int32_t part32_clear_status(const wc_rnn_args* a, hipStream_t st) {
  part32_zero_kernel<<<dim3(1), dim3(64), 0, st>>>(
      reinterpret_cast<int*>(static_cast<char*>(a->workspace) + part32_status_offset(a)), 1);
  return check_launch("wc_rnn_recurrence(status)");
}

int32_t part32_recurrence(const wc_rnn_args* a, hipStream_t st) {
  const int cus = device_cu_count();
  const int tpw = p32_tpw(a, cus);
  const int units = static_cast<int>(p32_units(a));
  P32Params p;
  p.rows = static_cast<int>(a->batch);
  p.chunks = (p.rows + 15) / 16;
  p.steps = static_cast<int>(a->steps);
  p.hid = static_cast<int>(a->hidden);
  p.parts = p.hid / (16 * tpw);
  p.spin_limit = part_spin_limit();
  p.gx = static_cast<const float*>(a->workspace);
  p.w_hh = static_cast<const float*>(a->w_hh);
  p.b_hh = static_cast<const float*>(a->b_hh);
  p.h0 = static_cast<const float*>(a->h0);
  p.c0 = a->cell == WC_CELL_LSTM ? static_cast<const float*>(a->c0) : nullptr;
  p.out = static_cast<float*>(a->out);
  p.hn = static_cast<float*>(a->h_n);
  p.cn = a->cell == WC_CELL_LSTM ? static_cast<float*>(a->c_n) : nullptr;
  // the streamed kernel's cell state (n * batch * hidden floats) is not used by this plan, and holds
  // the counters: 64 ints per unit of up to 16 rows, at least 160 floats per row
  p.sync = reinterpret_cast<int*>(static_cast<char*>(a->workspace) + p32_sync_offset(a));
  p.status = a->status ? static_cast<int*>(a->status) : p.sync + kSyncStatus;
  const int64_t nsync = static_cast<int64_t>(units) * kSyncInts;
  part32_zero_kernel<<<dim3(static_cast<uint32_t>(cdiv(nsync, 256))), dim3(256), 0, st>>>(p.sync, nsync);
  const int32_t rc = check_launch("wc_rnn_recurrence(counters)");
  if (rc) return rc;
  return a->cell == WC_CELL_GRU ? p32_dispatch<WC_CELL_GRU>(p, tpw, units, cus, st)
                                : p32_dispatch<WC_CELL_LSTM>(p, tpw, units, cus, st);
}

}  // namespace wc
