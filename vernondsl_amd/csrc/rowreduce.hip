// Op class 3: row reductions (sum, max) + softmax, and column reductions, on gfx950.
//
// No reference code (the north-star op class).  Semantics, shared with the CPU oracle:
//   row_sum = sum_j x[j] accumulated in f64, rounded once to f32;
//   row_max = max_j x[j] (exact);
//   softmax[j] = e[j] / s,  e[j] = exp(x[j] - row_max) in f32,  s = f64 sum of e rounded to f32.
// (The register-resident kernels evaluate exp with the branch-free exp_fast of fmath.h, in its
// form for arguments <= 0, within a few ulp of the library expf that the streaming kernel and the
// oracle use.)
// The register-resident kernels multiply by 1/s instead of dividing (within one ulp of e/s) and
// form their sums as f32 partials of 4 or 8 elements added into f64 accumulators (f32 rows) or,
// for bf16 rows, as f32 sums across the wave (DPP) added in f64 across waves: sums within a few
// ulp of the f64 accumulation, far inside the op's 1e-5 (f32) / 1e-2 (bf16) tolerances, for less
// VALU work per element, which bounds the bf16 kernels.
//
// Mapping: one 64-lane wavefront owns one row and keeps it in VGPRs, so x is read from HBM once
// and softmax written once (the HBM roofline's minimum traffic).  Lane l holds the 16-byte
// vectors v*64 + l, v < NV, so every load/store instruction of a wave covers 1 KiB contiguous.
// Reductions stay inside the wave (xor butterflies), so a 256-thread block is 4 independent
// rows and needs no LDS and no barrier.  Other widths are held in registers too, masked at their
// ends (row_softmax_any); only rows wider than 8192 vectors and few narrow rows use a 3-pass streaming
// kernel (max/sum, exp-sum, write).

#include <type_traits>

#include "common.h"

namespace vdsl {
namespace {

__device__ __forceinline__ double wave_sum_f64(double v) {
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) v += __shfl_xor(v, m, 64);
  return v;
}

// Wave reductions through DPP (no LDS round trip): a butterfly inside each row of 16 lanes
// (quad_perm [1,0,3,2], [2,3,0,1], row_half_mirror, row_mirror), then the four rows' values read
// as scalars and combined.  Every lane gets the result.
template <int CTRL>
__device__ __forceinline__ float dpp_f32(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, false));
}
__device__ __forceinline__ float row_lane(float v, int lane) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane));
}
__device__ __forceinline__ float wave_sum_dpp(float v) {
  v += dpp_f32<0xB1>(v);
  v += dpp_f32<0x4E>(v);
  v += dpp_f32<0x141>(v);
  v += dpp_f32<0x140>(v);
  return (row_lane(v, 0) + row_lane(v, 16)) + (row_lane(v, 32) + row_lane(v, 48));
}
__device__ __forceinline__ float wave_max_dpp(float v) {
  v = fmaxf(v, dpp_f32<0xB1>(v));
  v = fmaxf(v, dpp_f32<0x4E>(v));
  v = fmaxf(v, dpp_f32<0x141>(v));
  v = fmaxf(v, dpp_f32<0x140>(v));
  return fmaxf(fmaxf(row_lane(v, 0), row_lane(v, 16)), fmaxf(row_lane(v, 32), row_lane(v, 48)));
}

// exp_fast for n <= 0 (softmax's x - max): 2^t cannot overflow there, so only a non-finite t
// (n = -inf or NaN) skips the correction.  The same value as exp_fast for every such n.
__device__ __forceinline__ float exp_nonpos(float n) {
  const float t = n * 1.4426950408889634f;
  float r = __builtin_fmaf(n, 1.4426950408889634f, -t);
  r = __builtin_fmaf(n, 1.92596299e-08f, r);  // log2(e) - fl(log2(e))
  const float e = __builtin_amdgcn_exp2f(t);
  const float c = __builtin_fmaf(e, r * 0.6931471805599453f, e);
  return __builtin_isfinite(t) ? c : e;
}

// A wave's partial sum: f64 butterflies for f32 rows; for bf16 rows (outputs with 8 significant
// bits, bound by VALU work rather than HBM) the lanes' f32 partials meet in f32 through DPP.
template <int DT>
__device__ __forceinline__ double wave_partial_sum(float lane_part, double lane_part64) {
  if constexpr (DT == VDSL_BF16) return static_cast<double>(wave_sum_dpp(lane_part));
  else return wave_sum_f64(lane_part64);
}
template <int DT>
__device__ __forceinline__ float wave_partial_max(float v) {
  if constexpr (DT == VDSL_BF16) return wave_max_dpp(v);
  else return wave_max(v);
}

template <int DT>
struct Elem;
template <>
struct Elem<VDSL_F32> {
  static constexpr int kPerVec = 4;  // elements per 16-byte vector
  __device__ static __forceinline__ void unpack(const uint4& v, float (&o)[4]) {
    o[0] = __uint_as_float(v.x); o[1] = __uint_as_float(v.y); o[2] = __uint_as_float(v.z); o[3] = __uint_as_float(v.w);
  }
  __device__ static __forceinline__ uint4 pack(const float (&o)[4]) {
    return make_uint4(__float_as_uint(o[0]), __float_as_uint(o[1]), __float_as_uint(o[2]), __float_as_uint(o[3]));
  }
  __device__ static __forceinline__ float load1(const void* p, int64_t i) { return static_cast<const float*>(p)[i]; }
  __device__ static __forceinline__ void store1(void* p, int64_t i, float v) { static_cast<float*>(p)[i] = v; }
};
template <>
struct Elem<VDSL_BF16> {
  static constexpr int kPerVec = 8;
  __device__ static __forceinline__ void unpack(const uint4& v, float (&o)[8]) {
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      o[2 * k] = __uint_as_float(w[k] << 16);
      o[2 * k + 1] = __uint_as_float(w[k] & 0xFFFF0000u);
    }
  }
  __device__ static __forceinline__ uint4 pack(const float (&o)[8]) {
    return make_uint4(pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3]), pack_bf16x2(o[4], o[5]), pack_bf16x2(o[6], o[7]));
  }
  __device__ static __forceinline__ float load1(const void* p, int64_t i) {
    return bf16_to_f32(static_cast<const uint16_t*>(p)[i]);
  }
  __device__ static __forceinline__ void store1(void* p, int64_t i, float v) { static_cast<uint16_t*>(p)[i] = f32_to_bf16(v); }
};

// Register-resident row: NV 16-byte vectors per lane, cols = 64 * NV * E::kPerVec.
template <int DT, int NV>
__global__ __launch_bounds__(256) void row_softmax_resident(const void* __restrict__ x, float* __restrict__ row_sum,
                                                            float* __restrict__ row_max, void* __restrict__ sm,
                                                            int64_t rows) {
  using E = Elem<DT>;
  constexpr int PV = E::kPerVec;
  constexpr int64_t cols = 64 * NV * PV;
  const int lane = threadIdx.x & 63;
  const int64_t row = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  const uint4* src = reinterpret_cast<const uint4*>(static_cast<const char*>(x) + row * cols * (DT == VDSL_F32 ? 4 : 2));

  float v[NV][PV];
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const u32x4 r = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(src + k * 64 + lane));
    E::unpack(make_uint4(r[0], r[1], r[2], r[3]), v[k]);
  }
  double s = 0.0;
  float fs = 0.0f;
  float m = -INFINITY;
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    float part = 0.0f;
#pragma unroll
    for (int e = 0; e < PV; ++e) {
      part += v[k][e];
      m = fmaxf(m, v[k][e]);
    }
    s += static_cast<double>(part);
    fs += part;
  }
  s = wave_partial_sum<DT>(fs, s);
  m = wave_partial_max<DT>(m);
  if (lane == 0) {
    if (row_sum) row_sum[row] = static_cast<float>(s);
    if (row_max) row_max[row] = m;
  }
  if (!sm) return;
  double es = 0.0;
  float fes = 0.0f;
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    float part = 0.0f;
#pragma unroll
    for (int e = 0; e < PV; ++e) {
      v[k][e] = exp_nonpos(v[k][e] - m);
      part += v[k][e];
    }
    es += static_cast<double>(part);
    fes += part;
  }
  const float inv = 1.0f / static_cast<float>(wave_partial_sum<DT>(fes, es));
  uint4* dst = reinterpret_cast<uint4*>(static_cast<char*>(sm) + row * cols * (DT == VDSL_F32 ? 4 : 2));
#pragma unroll
  for (int k = 0; k < NV; ++k) {
#pragma unroll
    for (int e = 0; e < PV; ++e) v[k][e] = v[k][e] * inv;
    const uint4 w = E::pack(v[k]);
    const u32x4 wv = {w.x, w.y, w.z, w.w};
    __builtin_nontemporal_store(wv, reinterpret_cast<u32x4*>(dst + k * 64 + lane));
  }
}

// Wide rows, one block per row: cols = 64 * WPR * NV * PV, the row held in the registers of WPR
// waves (NV 16-byte vectors per lane, lane l of wave w holding vectors (w NV + k) 64 + l).  Each
// wave reduces its part; the WPR partial sums (f64) and maxima meet in LDS and every wave adds
// them in the same order.  Against one wave per row (all of a 4096-wide f32 row in one wave's
// registers, 88 VGPRs, 5 waves per SIMD) the smaller per-lane share runs at full occupancy and a
// row's load-reduce-store chain is 8 times shorter: [16384][4096] f32 84 us against 93-96 us.
template <int DT, int NV, int WPR>
__global__ __launch_bounds__(64 * WPR) void row_softmax_split(const void* __restrict__ x, float* __restrict__ row_sum,
                                                              float* __restrict__ row_max, void* __restrict__ sm,
                                                              int64_t rows) {
  using E = Elem<DT>;
  constexpr int PV = E::kPerVec;
  constexpr int64_t cols = 64 * WPR * NV * PV;
  __shared__ double part_sum[WPR];
  __shared__ float part_max[WPR];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t row = blockIdx.x;
  const uint4* src = reinterpret_cast<const uint4*>(static_cast<const char*>(x) + row * cols * (DT == VDSL_F32 ? 4 : 2)) +
                     wave * NV * 64 + lane;

  float v[NV][PV];
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const u32x4 r = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(src + k * 64));
    E::unpack(make_uint4(r[0], r[1], r[2], r[3]), v[k]);
  }
  double s = 0.0;
  float fs = 0.0f;
  float m = -INFINITY;
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    float part = 0.0f;
#pragma unroll
    for (int e = 0; e < PV; ++e) {
      part += v[k][e];
      m = fmaxf(m, v[k][e]);
    }
    s += static_cast<double>(part);
    fs += part;
  }
  s = wave_partial_sum<DT>(fs, s);
  m = wave_partial_max<DT>(m);
  if (lane == 0) {
    part_sum[wave] = s;
    part_max[wave] = m;
  }
  __syncthreads();
  s = 0.0;
  m = -INFINITY;
#pragma unroll
  for (int w = 0; w < WPR; ++w) {
    s += part_sum[w];
    m = fmaxf(m, part_max[w]);
  }
  if (threadIdx.x == 0) {
    if (row_sum) row_sum[row] = static_cast<float>(s);
    if (row_max) row_max[row] = m;
  }
  if (!sm) return;
  double es = 0.0;
  float fes = 0.0f;
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    float part = 0.0f;
#pragma unroll
    for (int e = 0; e < PV; ++e) {
      v[k][e] = exp_nonpos(v[k][e] - m);
      part += v[k][e];
    }
    es += static_cast<double>(part);
    fes += part;
  }
  es = wave_partial_sum<DT>(fes, es);
  __syncthreads();  // every wave has read part_sum
  if (lane == 0) part_sum[wave] = es;
  __syncthreads();
  es = 0.0;
#pragma unroll
  for (int w = 0; w < WPR; ++w) es += part_sum[w];
  const float inv = 1.0f / static_cast<float>(es);
  uint4* dst = reinterpret_cast<uint4*>(static_cast<char*>(sm) + row * cols * (DT == VDSL_F32 ? 4 : 2)) + wave * NV * 64 + lane;
#pragma unroll
  for (int k = 0; k < NV; ++k) {
#pragma unroll
    for (int e = 0; e < PV; ++e) v[k][e] = v[k][e] * inv;
    const uint4 w = E::pack(v[k]);
    const u32x4 wv = {w.x, w.y, w.z, w.w};
    __builtin_nontemporal_store(wv, reinterpret_cast<u32x4*>(dst + k * 64));
  }
}

// exp of n[0 .. PV) <= 0, the steps of exp_fast.  Where some lane of the wave has an n below -87, whose
// exp2 would be flushed or whose exponent may be infinite, the wave takes the form that keeps
// subnormal results: the power is formed 2^32 higher (t + 32 is exact there) and scaled back once.
// NaN becomes 0 there: the caller gives a row with a NaN or an infinite maximum NaN.
template <int PV>
__device__ __forceinline__ void exp_nonpos_vec(float (&n)[PV]) {
  float low = n[0];
#pragma unroll
  for (int e = 1; e < PV; ++e) low = fminf(low, n[e]);
  if (__any(low < -87.0f)) {
#pragma unroll
    for (int e = 0; e < PV; ++e) {
      const float c = fmaxf(n[e], -200.0f);
      const float t = c * 1.4426950408889634f;
      float r = __builtin_fmaf(c, 1.4426950408889634f, -t);
      r = __builtin_fmaf(c, 1.92596299e-08f, r);  // log2(e) - fl(log2(e))
      const bool up = t < -100.0f;
      const float x = __builtin_amdgcn_exp2f(up ? t + 32.0f : t);
      n[e] = __builtin_ldexpf(__builtin_fmaf(x, r * 0.6931471805599453f, x), up ? -32 : 0);
    }
  } else {
#pragma unroll
    for (int e = 0; e < PV; ++e) {
      const float t = n[e] * 1.4426950408889634f;
      float r = __builtin_fmaf(n[e], 1.4426950408889634f, -t);
      r = __builtin_fmaf(n[e], 1.92596299e-08f, r);
      const float x = __builtin_amdgcn_exp2f(t);
      n[e] = __builtin_fmaf(x, r * 0.6931471805599453f, x);
    }
  }
}

// e / s from i = 1 / s (correctly rounded): the rounded product corrected once by its exact
// residual (Markstein), which rounds normal results correctly in 3 operations.
__device__ __forceinline__ float quotient(float e, float s, float i) {
  const float q = e * i;
  return __builtin_fmaf(__builtin_fmaf(-q, s, e), i, q);
}

// Any width up to NV 16-byte vectors per lane: the row is read once, in the aligned vectors that
// cover it (a row of an odd width starts anywhere in its first vector), and held in registers.
// Elements of the first and last vector that belong to the neighbouring rows are read with it,
// replaced by -inf and never stored; only the tensor's very last vector is read by elements.  BLOCK:
// a block per row, its waves meeting in LDS; else groups of 1 << lg_lanes <= 64 lanes take a row
// each and reduce by butterflies.  Sums are f64 sums of every element, as in the streaming kernel.
// Bound by HBM for f32 and by VALU work (the f64 sums and the exponential) for bf16.  [3000][5003]
// f32: 99.4 us with the streaming kernel (three passes of 4-byte loads, one wave per row), 23.3 us
// (5.16 TB/s) here; bf16 76 -> 20 us; [16384][1000] f32 58.8 -> 26 us.
template <int DT, int NV, bool BLOCK>
__global__ __launch_bounds__(BLOCK ? 1024 : 256) void row_softmax_any(const void* __restrict__ x, float* __restrict__ row_sum,
                                                                      float* __restrict__ row_max, void* __restrict__ sm,
                                                                      int64_t rows, int64_t cols, int lg_lanes) {
  using E = Elem<DT>;
  constexpr int PV = E::kPerVec;
  __shared__ double part_sum[BLOCK ? 16 : 1];
  __shared__ float part_max[BLOCK ? 16 : 1];
  const int lanes = BLOCK ? static_cast<int>(blockDim.x) : 1 << lg_lanes;  // per row
  const int at = BLOCK ? static_cast<int>(threadIdx.x) : static_cast<int>(threadIdx.x) & (lanes - 1);
  const int64_t row = BLOCK ? static_cast<int64_t>(blockIdx.x)
                            : static_cast<int64_t>(blockIdx.x) * (256 >> lg_lanes) + (threadIdx.x >> lg_lanes);
  const bool live = row < rows;  // groups past the last row take part in the wave's butterflies
  const int64_t begin = row * cols, end = begin + cols, total = rows * cols;
  const int64_t first = begin / PV;
  const int waves = lanes >> 6, wave = threadIdx.x >> 6;

  float v[NV][PV];
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const int64_t i = first + at + static_cast<int64_t>(k) * lanes, e0 = i * PV;
    if (live && e0 < end) {
      if (e0 + PV <= total) {
        const u32x4 r = __builtin_nontemporal_load(static_cast<const u32x4*>(x) + i);
        E::unpack(make_uint4(r[0], r[1], r[2], r[3]), v[k]);
      } else {
#pragma unroll
        for (int e = 0; e < PV; ++e) v[k][e] = e0 + e < total ? E::load1(x, e0 + e) : 0.0f;
      }
    } else {
#pragma unroll
      for (int e = 0; e < PV; ++e) v[k][e] = 0.0f;
    }
  }
  double s = 0.0;
  float m = -INFINITY;
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const int64_t e0 = (first + at + static_cast<int64_t>(k) * lanes) * PV;
    if (e0 >= begin && e0 + PV <= end) {
#pragma unroll
      for (int e = 0; e < PV; ++e) {
        s += static_cast<double>(v[k][e]);
        m = fmaxf(m, v[k][e]);
      }
    } else {
#pragma unroll
      for (int e = 0; e < PV; ++e) {
        const bool in = e0 + e >= begin && e0 + e < end;
        s += static_cast<double>(in ? v[k][e] : 0.0f);
        v[k][e] = in ? v[k][e] : -INFINITY;
        m = fmaxf(m, v[k][e]);
      }
    }
  }
  // The row's f64 sum of one value per lane, on every lane; the same order on each.
  const auto row_total = [&](double t) -> double {
    for (int d = (BLOCK ? 64 : lanes) >> 1; d >= 1; d >>= 1) t += __shfl_xor(t, d, 64);
    if constexpr (BLOCK) {
      if ((threadIdx.x & 63) == 0) part_sum[wave] = t;
      __syncthreads();
      t = 0.0;
      for (int w = 0; w < waves; ++w) t += part_sum[w];
    }
    return t;
  };
  for (int d = (BLOCK ? 64 : lanes) >> 1; d >= 1; d >>= 1) m = fmaxf(m, __shfl_xor(m, d, 64));
  if constexpr (BLOCK) {
    if ((threadIdx.x & 63) == 0) part_max[wave] = m;
  }
  s = row_total(s);
  if constexpr (BLOCK) {
    for (int w = 0; w < waves; ++w) m = fmaxf(m, part_max[w]);
  }
  if (live && at == 0) {
    if (row_sum) row_sum[row] = static_cast<float>(s);
    if (row_max) row_max[row] = m;
  }
  if (!sm) return;
  double es = 0.0;
#pragma unroll
  for (int k = 0; k < NV; ++k) {
#pragma unroll
    for (int e = 0; e < PV; ++e) v[k][e] = v[k][e] - m;
    exp_nonpos_vec<PV>(v[k]);
#pragma unroll
    for (int e = 0; e < PV; ++e) es += static_cast<double>(v[k][e]);
  }
  if constexpr (BLOCK) __syncthreads();  // every wave has read part_sum
  // A NaN element (its sum is NaN), +inf or a row of -inf: every quotient is NaN.
  const bool nan_row = __builtin_isnan(s) || __builtin_isinf(m);
  es = row_total(es);
  const float sum = nan_row ? __builtin_nanf("") : static_cast<float>(es), inv = 1.0f / sum;
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const int64_t i = first + at + static_cast<int64_t>(k) * lanes, e0 = i * PV;
    if (!live || e0 >= end) continue;
#pragma unroll
    for (int e = 0; e < PV; ++e) v[k][e] = quotient(v[k][e], sum, inv);
    if (e0 >= begin && e0 + PV <= end) {
      const uint4 w = E::pack(v[k]);
      const u32x4 wv = {w.x, w.y, w.z, w.w};
      __builtin_nontemporal_store(wv, static_cast<u32x4*>(sm) + i);
    } else {
#pragma unroll
      for (int e = 0; e < PV; ++e)
        if (e0 + e >= begin && e0 + e < end) E::store1(sm, e0 + e, v[k][e]);
    }
  }
}

// Rows wider than row_softmax_any holds, and few narrow rows: three streaming passes with the same arithmetic.
template <int DT>
__global__ __launch_bounds__(256) void row_softmax_generic(const void* __restrict__ x, float* __restrict__ row_sum,
                                                           float* __restrict__ row_max, void* __restrict__ sm,
                                                           int64_t rows, int64_t cols) {
  using E = Elem<DT>;
  const int lane = threadIdx.x & 63;
  const int64_t row = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  const int64_t base = row * cols;
  double s = 0.0;
  float m = -INFINITY;
  for (int64_t c = lane; c < cols; c += 64) {
    const float v = E::load1(x, base + c);
    s += static_cast<double>(v);
    m = fmaxf(m, v);
  }
  s = wave_sum_f64(s);
  m = wave_max(m);
  if (lane == 0) {
    if (row_sum) row_sum[row] = static_cast<float>(s);
    if (row_max) row_max[row] = m;
  }
  if (!sm) return;
  double es = 0.0;
  for (int64_t c = lane; c < cols; c += 64) es += static_cast<double>(expf(E::load1(x, base + c) - m));
  const float esf = static_cast<float>(wave_sum_f64(es));
  for (int64_t c = lane; c < cols; c += 64) E::store1(sm, base + c, expf(E::load1(x, base + c) - m) / esf);
}

// Column reductions.  A block owns a strip of L * VEC columns (L a power of two, VEC elements per
// load) and a range of rows: its 1024 lanes are L column lanes x 1024 / L row lanes, each adding
// its rows in f64 in row order; the row lanes then meet in a fixed order (butterflies in the wave,
// the 16 waves in LDS), so results do not depend on scheduling.  With one range the block stores
// the result; with several it stores f64 sums and f32 maxima to scratch memory and
// col_finish_kernel adds the ranges in order.
constexpr int kColThreads = 1024, kColBatch = 8;

// VEC consecutive elements of a row from one load (16 bytes, a bf16 pair or one element).
template <int DT, int VEC>
struct ColLoad {
  using E = Elem<DT>;
  static constexpr int kBytes = VEC * (DT == VDSL_F32 ? 4 : 2);
  using Raw = std::conditional_t<kBytes == 16, u32x4, std::conditional_t<kBytes == 4, uint32_t, uint16_t>>;
  __device__ static __forceinline__ void unpack(const Raw& r, float (&o)[VEC]) {
    if constexpr (kBytes == 16) {
      E::unpack(make_uint4(r[0], r[1], r[2], r[3]), o);
    } else if constexpr (DT == VDSL_F32) {
      o[0] = __uint_as_float(r);
    } else if constexpr (VEC == 2) {
      o[0] = __uint_as_float(r << 16);
      o[1] = __uint_as_float(r & 0xFFFF0000u);
    } else {
      o[0] = bf16_to_f32(r);
    }
  }
};

template <int DT, int VEC, int THREADS>
__global__ __launch_bounds__(THREADS) void col_reduce_kernel(const void* __restrict__ x, float* __restrict__ col_sum,
                                                                 float* __restrict__ col_max, double* __restrict__ part_sum,
                                                                 float* __restrict__ part_max, int64_t all_rows, int64_t per_range,
                                                                 int64_t cols, int lg_lanes) {
  using LD = ColLoad<DT, VEC>;
  using Raw = typename LD::Raw;
  extern __shared__ __align__(16) char col_smem[];  // [waves][L * VEC] f64 sums, then as many f32 maxima
  const int L = 1 << lg_lanes, width = VEC << lg_lanes, R = THREADS >> lg_lanes;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t strip = blockIdx.x, first = static_cast<int64_t>(blockIdx.y) * per_range;
  const int64_t rows = all_rows - first < per_range ? all_rows - first : per_range;  // of this range
  const int cl = threadIdx.x & (L - 1);
  const int64_t rl = threadIdx.x >> lg_lanes;
  const int64_t c = strip * width + cl * VEC;
  const int64_t pitch = cols / VEC;  // cols % VEC == 0
  const Raw* src = reinterpret_cast<const Raw*>(x) + first * pitch + c / VEC;
  double s[VEC];
  float m[VEC];
#pragma unroll
  for (int e = 0; e < VEC; ++e) s[e] = 0.0, m[e] = -INFINITY;
  if (c < cols) {
    int64_t r = rl;
    for (; r + static_cast<int64_t>(kColBatch - 1) * R < rows; r += static_cast<int64_t>(kColBatch) * R) {
      Raw v[kColBatch];
#pragma unroll
      for (int u = 0; u < kColBatch; ++u) v[u] = src[(r + static_cast<int64_t>(u) * R) * pitch];
#pragma unroll
      for (int u = 0; u < kColBatch; ++u) {
        float f[VEC];
        LD::unpack(v[u], f);
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
          s[e] += static_cast<double>(f[e]);
          m[e] = fmaxf(m[e], f[e]);
        }
      }
    }
    if (r < rows) {  // the last, partial batch: rows past the end read the last row and add nothing
      Raw v[kColBatch];
#pragma unroll
      for (int u = 0; u < kColBatch; ++u) {
        const int64_t ru = r + static_cast<int64_t>(u) * R;
        v[u] = src[(ru < rows ? ru : rows - 1) * pitch];
      }
#pragma unroll
      for (int u = 0; u < kColBatch; ++u) {
        if (r + static_cast<int64_t>(u) * R < rows) {  // a branch: few rows skip the f64 work of the rest
          float f[VEC];
          LD::unpack(v[u], f);
#pragma unroll
          for (int e = 0; e < VEC; ++e) {
            s[e] += static_cast<double>(f[e]);
            m[e] = fmaxf(m[e], f[e]);
          }
        }
      }
    }
  }
  for (int k = 32; k >= L; k >>= 1) {
#pragma unroll
    for (int e = 0; e < VEC; ++e) {
      s[e] += __shfl_xor(s[e], k, 64);
      m[e] = fmaxf(m[e], __shfl_xor(m[e], k, 64));
    }
  }
  double* const ssum = reinterpret_cast<double*>(col_smem);
  float* const smax = reinterpret_cast<float*>(ssum + (THREADS / 64) * width);
  if (lane < L) {
#pragma unroll
    for (int e = 0; e < VEC; ++e) {
      ssum[wave * width + cl * VEC + e] = s[e];
      smax[wave * width + cl * VEC + e] = m[e];
    }
  }
  __syncthreads();
  for (int k = threadIdx.x; k < width; k += THREADS) {
    const int64_t col = strip * width + k;
    if (col >= cols) break;
    double t = ssum[k];
    float mm = smax[k];
#pragma unroll
    for (int w = 1; w < THREADS / 64; ++w) {
      t += ssum[w * width + k];
      mm = fmaxf(mm, smax[w * width + k]);
    }
    if (part_sum) {
      part_sum[blockIdx.y * cols + col] = t;
      part_max[blockIdx.y * cols + col] = mm;
    } else {
      if (col_sum) col_sum[col] = static_cast<float>(t);
      if (col_max) col_max[col] = mm;
    }
  }
}

// Few rows: a lane per VEC columns takes all of them, 8 rows' loads at a time; nothing to combine.  Up to 8
// rows, or 16 of small tensors; us with the lanes of a block split over rows (most of them idle, then LDS
// and butterflies) and here: [1][1000000] f32 47.6, 4.7 bf16 27.4, 3.7; [2][3000001] f32 143, 9.9; [8][1048576]
// bf16 24.1, 6.7; [16][30000] f32 5.0, 2.6; but [16][2000000] bf16 18.0 in blocks of 256 lanes split over rows, 21.7.
template <int DT, int VEC>
__global__ __launch_bounds__(256) void col_few_kernel(const void* __restrict__ x, float* __restrict__ col_sum,
                                                      float* __restrict__ col_max, int rows, int64_t pitch) {
  using LD = ColLoad<DT, VEC>;
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;  // of the row's loads
  if (i >= pitch) return;
  const typename LD::Raw* src = reinterpret_cast<const typename LD::Raw*>(x) + i;
  double s[VEC];
  float m[VEC];
#pragma unroll
  for (int e = 0; e < VEC; ++e) s[e] = 0.0, m[e] = -INFINITY;
  for (int r = 0; r < rows; r += kColBatch) {
    std::conditional_t<LD::kBytes == 2, uint32_t, typename LD::Raw> v[kColBatch];  // (no halves of one register)
#pragma unroll
    for (int u = 0; u < kColBatch; ++u)
      if (r + u < rows) v[u] = src[(r + u) * pitch];
#pragma unroll
    for (int u = 0; u < kColBatch; ++u) {
      if (r + u >= rows) break;
      float f[VEC];
      LD::unpack(static_cast<typename LD::Raw>(v[u]), f);
#pragma unroll
      for (int e = 0; e < VEC; ++e) {
        s[e] += static_cast<double>(f[e]);
        m[e] = fmaxf(m[e], f[e]);
      }
    }
  }
  struct __attribute__((packed, aligned(4))) Out {
    float v[VEC];
  };
  if (col_sum) {
    Out o;
#pragma unroll
    for (int e = 0; e < VEC; ++e) o.v[e] = static_cast<float>(s[e]);
    reinterpret_cast<Out*>(col_sum)[i] = o;
  }
  if (col_max) {
    Out o;
#pragma unroll
    for (int e = 0; e < VEC; ++e) o.v[e] = m[e];
    reinterpret_cast<Out*>(col_max)[i] = o;
  }
}

// Adds the row ranges' partial results: 64 columns per block, its 16 waves taking every 16th range
// of them and meeting in LDS, both in a fixed order.
__global__ __launch_bounds__(kColThreads) void col_finish_kernel(const double* __restrict__ part_sum,
                                                                 const float* __restrict__ part_max,
                                                                 float* __restrict__ col_sum, float* __restrict__ col_max,
                                                                 int64_t cols, int ranges) {
  constexpr int W = kColThreads / 64;
  __shared__ double ssum[W][64];
  __shared__ float smax[W][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t c = static_cast<int64_t>(blockIdx.x) * 64 + lane;
  double s = 0.0;
  float m = -INFINITY;
  if (c < cols) {
#pragma unroll 4
    for (int k = wave; k < ranges; k += W) {
      s += part_sum[k * cols + c];
      m = fmaxf(m, part_max[k * cols + c]);
    }
  }
  ssum[wave][lane] = s;
  smax[wave][lane] = m;
  __syncthreads();
  if (wave == 0 && c < cols) {
#pragma unroll
    for (int w = 1; w < W; ++w) {
      s += ssum[w][lane];
      m = fmaxf(m, smax[w][lane]);
    }
    if (col_sum) col_sum[c] = static_cast<float>(s);
    if (col_max) col_max[c] = m;
  }
}

// The strip's width (log2 of its column lanes) and the row ranges.  A CU misses its L1 at about one
// 128-byte line per 4 cycles whatever part of the line is used, so strips of 256 bytes of a row are
// read best, and row ranges make them cover the CUs: [16384][4096] f32 1627 us with one block of
// 256 lanes per 64 columns, 70.3-78.5 us in one launch with 64- or 128-byte strips, 47.8 us (5616
// GB/s) with 256-byte strips in 8 ranges (512 blocks; 256 blocks 51.1, 1024 49.1); bf16 27.2 us
// with 256 blocks (512: 30.0); [16384][256] f32 8.5 us against 31 us in one launch.  For less the
// second launch costs more than the strips' latency ([700][700] f32 6.8 us a call against 5.4; but
// [16384][64] 7.2 against 21.7, hence the row count): one range, and strips narrowed to 16 bytes
// while they do not cover the CUs and a row lane has more than half a batch of rows.  Up to 64 rows
// such a block has 256 lanes (of 1024 most have no row: [20][262144] f32 10.5 us against 6.2,
// [64][1048576] bf16 46.2 against 32.2).  Small tensors are read an element or a bf16 pair per lane
// (col_small): with 16 bytes per lane the f64 adds and butterflies of few blocks take longer than the
// loads ([100][16384] bf16 5.1 us a call against 4.1).
bool col_small(int64_t rows, int64_t bytes) {
  return !(bytes >= (int64_t{4} << 20) || (bytes >= (int64_t{1} << 20) && rows >= 4096));
}

template <int DT, int VEC>
int launch_cols(vdsl_queue q, const void* x, float* cs, float* cm, int64_t rows, int64_t cols) {
  constexpr int kBytes = ColLoad<DT, VEC>::kBytes;
  const auto strips = [&](int l) { return (cols + (int64_t{VEC} << l) - 1) / (int64_t{VEC} << l); };
  const int64_t bytes = rows * cols * (DT == VDSL_F32 ? 4 : 2);  // fits: checked by the caller
  if (rows <= (col_small(rows, bytes) ? 16 : 8)) {
    const int64_t pitch = cols / VEC, threads = pitch < 256 * 256 ? 64 : 256, blocks = (pitch + threads - 1) / threads;
    if (blocks > 0x7fffffff) return fail(VDSL_ERR_UNSUPPORTED, "too many columns");
    hipLaunchKernelGGL((col_few_kernel<DT, VEC>), dim3(static_cast<unsigned>(blocks)), dim3(static_cast<unsigned>(threads)), 0,
                       q->stream, x, cs, cm, static_cast<int>(rows), pitch);
    return check_launch("col_few_kernel");
  }
  int lg = kBytes == 16 ? 4 : 6, ranges = 1;
  int64_t per_range = rows;
  double* part = nullptr;
  if (!col_small(rows, bytes)) {
    const int64_t by_blocks = (DT == VDSL_F32 && bytes >= (int64_t{128} << 20) ? 512 : 256) / strips(lg);
    const int64_t by_rows = rows / (kColBatch / 2 * (kColThreads >> lg));
    const int64_t want = by_blocks < by_rows ? by_blocks : by_rows;
    if (want > 1) {
      per_range = (rows + want - 1) / want;
      ranges = static_cast<int>((rows + per_range - 1) / per_range);
      part = static_cast<double*>(queue_scratch(q, nbytes(ranges, cols, 12)));
    }
  }
  const bool few = !part && rows <= 64;
  const int threads = few ? 256 : kColThreads;
  if (!part) {
    ranges = 1, per_range = rows, lg = 6;
    while (lg > 0 && (kBytes << (lg - 1)) >= 16 && strips(lg) < 256 && rows > (kColBatch / 2) * (threads >> lg)) --lg;
  }
  const int64_t blocks = strips(lg);
  if (blocks > 0x7fffffff) return fail(VDSL_ERR_UNSUPPORTED, "too many columns");
  float* pmax = part ? reinterpret_cast<float*>(part + static_cast<int64_t>(ranges) * cols) : nullptr;
  const unsigned lds = static_cast<unsigned>((threads / 64) * (VEC << lg) * 12);
  hipLaunchKernelGGL((few ? col_reduce_kernel<DT, VEC, 256> : col_reduce_kernel<DT, VEC, kColThreads>),
                     dim3(static_cast<unsigned>(blocks), static_cast<unsigned>(ranges)), dim3(threads), lds, q->stream, x, cs, cm, part,
                     pmax, rows, per_range, cols, lg);
  VDSL_TRY(check_launch("col_reduce_kernel"));
  if (!part) return VDSL_OK;
  hipLaunchKernelGGL(col_finish_kernel, dim3(static_cast<unsigned>((cols + 63) / 64)), dim3(kColThreads), 0, q->stream, part, pmax,
                     cs, cm, cols, ranges);
  return check_launch("col_finish_kernel");
}

template <int DT>
int launch_rows(const void* x, float* rs, float* rm, void* sm, int64_t rows, int64_t cols, hipStream_t st) {
  constexpr int PV = Elem<DT>::kPerVec;
  // Rows of 8, 16 or 32 vectors per 64 lanes: one block per row.  f32: 4 waves of 2 vectors per
  // lane or 8 waves of 2 or 4; bf16 (VALU-bound): 4 vectors per lane in 2, 4 or 8 waves, which
  // halves the reductions per element at 4096 columns (42.9 us against 45.7 for 2 vectors in 4
  // waves on [16384][4096], with the DPP reductions).
  if (cols == 64 * 8 * PV || cols == 64 * 16 * PV || cols == 64 * 32 * PV) {
    if (rows > 0x7fffffff) return fail(VDSL_ERR_UNSUPPORTED, "too many rows");
    const dim3 g(static_cast<unsigned>(rows));
    if constexpr (DT == VDSL_BF16) {
      if (cols == 64 * 8 * PV) hipLaunchKernelGGL((row_softmax_split<DT, 4, 2>), g, dim3(128), 0, st, x, rs, rm, sm, rows);
      else if (cols == 64 * 16 * PV) hipLaunchKernelGGL((row_softmax_split<DT, 4, 4>), g, dim3(256), 0, st, x, rs, rm, sm, rows);
      else hipLaunchKernelGGL((row_softmax_split<DT, 4, 8>), g, dim3(512), 0, st, x, rs, rm, sm, rows);
    } else {
      if (cols == 64 * 8 * PV) hipLaunchKernelGGL((row_softmax_split<DT, 2, 4>), g, dim3(256), 0, st, x, rs, rm, sm, rows);
      else if (cols == 64 * 16 * PV) hipLaunchKernelGGL((row_softmax_split<DT, 2, 8>), g, dim3(512), 0, st, x, rs, rm, sm, rows);
      else hipLaunchKernelGGL((row_softmax_split<DT, 4, 8>), g, dim3(512), 0, st, x, rs, rm, sm, rows);
    }
    return check_launch("row_softmax_split");
  }
  const int64_t blocks = (rows + 3) / 4;
  if (blocks > 0x7fffffff) return fail(VDSL_ERR_UNSUPPORTED, "too many rows");
  const dim3 grid(static_cast<unsigned>(blocks)), block(256);
  switch (cols) {
#define VDSL_ROW_CASE(NV) \
  case 64 * NV * PV: \
    hipLaunchKernelGGL((row_softmax_resident<DT, NV>), grid, block, 0, st, x, rs, rm, sm, rows); \
    return check_launch("row_softmax");
    VDSL_ROW_CASE(1)
    VDSL_ROW_CASE(2)
    VDSL_ROW_CASE(4)
#undef VDSL_ROW_CASE
    default: break;
  }
  // Other widths: the vectors that cover a row (one more than its width where rows start anywhere).
  const int64_t nvec = (cols + PV - 1) / PV + (cols % PV ? 1 : 0);
  constexpr int64_t kBlockMax = 1024 * 8;
  // Few rows of up to 256 columns are a matter of latency, where an element per lane comes sooner than a
  // vector per lane: [300][33] bf16 3.3 us against 4.1 in masked vectors, [2000][60] 3.6, 4.4, [1000][129] f32
  // 4.2, 4.5; but [4000][100] bf16 4.9, 4.7, [1000][200] (aligned rows) 4.5, 4.3, [300][16] 3.4, 3.1.
  const bool narrow = rows <= 2000 && cols > 16 && (cols <= 128 || (cols <= 256 && cols % PV != 0));
  if (narrow || nvec > kBlockMax || rows > 0x7fffffff) {
    hipLaunchKernelGGL((row_softmax_generic<DT>), grid, block, 0, st, x, rs, rm, sm, rows, cols);
    return check_launch("row_softmax");
  }
  // Waves per row: the fewest whose lanes hold the row in kMost vectors each.  More vectors per lane
  // mean fewer reductions and barriers per element, until their registers leave too few waves; wave
  // counts that are no multiple of 4 load a CU's SIMDs unevenly (9 waves of 94 registers: one block
  // per CU instead of two, [4000][16383] f32 152 us against 100).  f32 [3000][5003]: 4 waves of 5
  // vectors 24.0 us, 3 of 8 25.5, 5 of 4 25.7, 10 of 2 31; bf16 [8000][7000]: 4 of 4 55 us, 7 of 2 60,
  // 2 of 8 73; bf16 [4000][12000]: 8 of 3 47 us, 6 of 4 65, 3 of 8 65.
  constexpr int kWaves[] = {1, 2, 4, 8, 12, 16};
  constexpr int kMostF32[] = {4, 5, 5, 6, 6, 8}, kMostBf16[] = {5, 5, 4, 3, 3, 8};
  const int* most = DT == VDSL_F32 ? kMostF32 : kMostBf16;
  int w = 0;
  while (nvec > int64_t{64} * kWaves[w] * most[w]) ++w;  // ends: nvec <= kBlockMax
  if (w == 0) {
    int lg = 6;
    while (lg > 0 && nvec <= (int64_t{1} << (lg - 1))) --lg;
    const dim3 g(static_cast<unsigned>((rows + (256 >> lg) - 1) / (256 >> lg)));
    switch ((nvec + 63) / 64) {
#define VDSL_ANY_CASE(NV) \
  case NV: hipLaunchKernelGGL((row_softmax_any<DT, NV, false>), g, block, 0, st, x, rs, rm, sm, rows, cols, lg); break;
      VDSL_ANY_CASE(1)
      VDSL_ANY_CASE(2)
      VDSL_ANY_CASE(3)
      VDSL_ANY_CASE(4)
      default: hipLaunchKernelGGL((row_softmax_any<DT, 5, false>), g, block, 0, st, x, rs, rm, sm, rows, cols, lg);
#undef VDSL_ANY_CASE
    }
    return check_launch("row_softmax_any");
  }
  const dim3 g(static_cast<unsigned>(rows)), bl(static_cast<unsigned>(64 * kWaves[w]));
  switch ((nvec + 64 * kWaves[w] - 1) / (64 * kWaves[w])) {
#define VDSL_ANY_CASE(NV) \
  case NV: hipLaunchKernelGGL((row_softmax_any<DT, NV, true>), g, bl, 0, st, x, rs, rm, sm, rows, cols, 6); break;
    case 1:
    VDSL_ANY_CASE(2)
    VDSL_ANY_CASE(3)
    VDSL_ANY_CASE(4)
    VDSL_ANY_CASE(5)
    VDSL_ANY_CASE(6)
    default: hipLaunchKernelGGL((row_softmax_any<DT, 8, true>), g, bl, 0, st, x, rs, rm, sm, rows, cols, 6);
#undef VDSL_ANY_CASE
  }
  return check_launch("row_softmax_any");
}

}  // namespace
}  // namespace vdsl

using namespace vdsl;

extern "C" int vdsl_op_row_reduce_softmax(vdsl_queue q, int64_t rows, int64_t cols, int32_t dtype, vdsl_buffer x,
                                          vdsl_buffer row_sum, vdsl_buffer row_max, vdsl_buffer softmax) {
  VDSL_TRY(enter_queue(q));
  if (rows < 0 || cols < 0) return fail(VDSL_ERR_INVALID_ARG, "negative shape");
  if (dtype != VDSL_F32 && dtype != VDSL_BF16) return fail(VDSL_ERR_UNSUPPORTED, "softmax dtype must be f32 or bf16");
  const size_t es = dtype_size(dtype);
  VDSL_TRY(check_buffer(q, x, nbytes(rows, cols, es), "x", false));
  if (row_sum) VDSL_TRY(check_buffer(q, row_sum, nbytes(rows, 4), "row_sum", true));
  if (row_max) VDSL_TRY(check_buffer(q, row_max, nbytes(rows, 4), "row_max", true));
  if (softmax) VDSL_TRY(check_buffer(q, softmax, nbytes(rows, cols, es), "softmax", true));
  if (rows == 0) return VDSL_OK;
  if (cols == 0) {
    // sum of an empty row is 0 and its max is -inf; nothing else to write
    if (row_sum) VDSL_TRY(vdsl_buffer_fill_u32(q, row_sum, 0, static_cast<size_t>(rows) * 4, 0u));
    if (row_max) VDSL_TRY(vdsl_buffer_fill_u32(q, row_max, 0, static_cast<size_t>(rows) * 4, 0xFF800000u));
    return VDSL_OK;
  }
  float* rs = row_sum ? static_cast<float*>(row_sum->ptr) : nullptr;
  float* rm = row_max ? static_cast<float*>(row_max->ptr) : nullptr;
  void* sm = softmax ? softmax->ptr : nullptr;
  if (dtype == VDSL_F32) return launch_rows<VDSL_F32>(x->ptr, rs, rm, sm, rows, cols, q->stream);
  return launch_rows<VDSL_BF16>(x->ptr, rs, rm, sm, rows, cols, q->stream);
}

extern "C" int vdsl_op_col_reduce(vdsl_queue q, int64_t rows, int64_t cols, int32_t dtype, vdsl_buffer x,
                                  vdsl_buffer col_sum, vdsl_buffer col_max) {
  VDSL_TRY(enter_queue(q));
  if (rows < 0 || cols < 0) return fail(VDSL_ERR_INVALID_ARG, "negative shape");
  if (dtype != VDSL_F32 && dtype != VDSL_BF16) return fail(VDSL_ERR_UNSUPPORTED, "col_reduce dtype must be f32 or bf16");
  VDSL_TRY(check_buffer(q, x, nbytes(rows, cols, dtype_size(dtype)), "x", false));
  if (col_sum) VDSL_TRY(check_buffer(q, col_sum, nbytes(cols, 4), "col_sum", true));
  if (col_max) VDSL_TRY(check_buffer(q, col_max, nbytes(cols, 4), "col_max", true));
  if (cols == 0) return VDSL_OK;
  float* cs = col_sum ? static_cast<float*>(col_sum->ptr) : nullptr;
  float* cm = col_max ? static_cast<float*>(col_max->ptr) : nullptr;
  // 16-byte loads need rows of whole 16-byte units (hipMalloc bases are aligned).
  const bool wide = !col_small(rows, static_cast<int64_t>(nbytes(rows, cols, dtype_size(dtype))));
  if (dtype == VDSL_F32) {
    if (wide && cols % 4 == 0) return launch_cols<VDSL_F32, 4>(q, x->ptr, cs, cm, rows, cols);
    return launch_cols<VDSL_F32, 1>(q, x->ptr, cs, cm, rows, cols);
  }
  if (wide && cols % 8 == 0) return launch_cols<VDSL_BF16, 8>(q, x->ptr, cs, cm, rows, cols);
  if (cols % 2 == 0) return launch_cols<VDSL_BF16, 2>(q, x->ptr, cs, cm, rows, cols);
  return launch_cols<VDSL_BF16, 1>(q, x->ptr, cs, cm, rows, cols);
}
