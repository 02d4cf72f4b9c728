// Op class 4: dense bf16 x bf16 -> f32-accumulate GEMM on gfx950 MFMA, with fused epilogues.
//
// No reference code (the north-star op class: the dense matmuls of the MLP graph, forward and
// autodiff-generated backward).
//
// Native layout "NT": C[m][n] = sum_k A[m][k] * B[n][k], both operands K-contiguous (B is a
// weight in [out][in] form).  The other layouts are read as stored (gemm_any.h, gemm_dma.h's K-major
// forms) or, large, reduced to it by transposing the strided operand into caller-provided workspace
// first (vdsl_gemm_bf16_workspace_bytes).  The main loops are gemm_dma.h, gemm_bpk.h (packed
// weights), gemm_skinny.h (a short side), gemm_any.h (any layout and extents) and gemm_mfma.h; this
// file adds the epilogue (GELU / ReLU, optional f32 pre-activation, f32 or bf16 C) and the choice of
// loop and tile configuration per shape.

#include <atomic>
#include <cstdlib>

#include "gemm_mfma.h"
#include "gemm_bpk.h"
#include "gemm_any.h"
#include "gemm_dma.h"
#include "gemm_skinny.h"

namespace vdsl {

// Defined in layout.hip.
int launch_transpose(const void* src, void* dst, int64_t rows, int64_t cols, int dtype, hipStream_t s);
// Defined in autodiff.hip: the one-block, fixed-order sum of MSE partials into the loss.
int launch_mse_finish(const double* partials, int64_t n_partials, float* loss, double inv_n, hipStream_t s);

namespace {
std::atomic<int> g_gemm_config{-2};  // -2: not yet read from the environment
}  // namespace

int gemm_config_override() {
  int v = g_gemm_config.load(std::memory_order_relaxed);
  if (v == -2) {
    const char* e = std::getenv("VDSL_GEMM_CONFIG");
    g_gemm_config.compare_exchange_strong(v, e ? std::atoi(e) : -1);
    v = g_gemm_config.load(std::memory_order_relaxed);
  }
  return v;
}

namespace {


// Tile configurations (block M x N, K bytes per stage, wave grid).
using Bf0 = GemmConfig<MfmaBf16, 128, 128, 128, 2, 2>;  // wave tile 64x64
using Bf1 = GemmConfig<MfmaBf16, 256, 128, 128, 2, 2>;  // wave tile 128x64
using Bf2 = GemmConfig<MfmaBf16, 128, 256, 128, 2, 2>;  // wave tile 64x128
using Bf3 = GemmConfig<MfmaBf16, 64, 64, 128, 2, 2>;    // wave tile 32x32: small outputs
using Bf4 = GemmConfig<MfmaBf16, 256, 256, 64, 4, 2>;   // 8 waves, wave tile 64x128
using Bf5 = GemmConfig<MfmaBf16, 256, 128, 128, 4, 2>;  // 8 waves, wave tile 64x64
using Bf6 = GemmConfig<MfmaBf16, 128, 128, 256, 2, 2>;  // 128 bf16 of K per stage
using Bf7 = GemmConfig<MfmaBf16, 128, 64, 128, 2, 2>;   // wave tile 64x32: twice the blocks of 128x128
using Bf8 = GemmConfig<MfmaBf16, 64, 128, 128, 2, 2>;   // wave tile 32x64
using Bf9 = GemmConfig<MfmaBf16, 128, 128, 64, 2, 2>;   // 64 K bytes per stage: 3 blocks per CU fit in LDS
using Bf10 = GemmConfig<MfmaBf16, 256, 128, 64, 2, 2>;  // wave tile 128x64, 2 blocks per CU
using Bf11 = GemmConfig<MfmaBf16, 128, 256, 64, 2, 2>;  // wave tile 64x128, 2 blocks per CU
using Bf12 = GemmConfig<MfmaBf16, 256, 256, 64, 2, 4>;  // 8 waves, wave tile 128x64
using Bf13 = GemmConfig<MfmaBf16, 256, 128, 64, 4, 2>;  // 8 waves, wave tile 64x64, 2 blocks per CU
// Direct-to-LDS loop (gemm_dma.h), configurations 14..: <BM, BN, WGM, WGN, LDS stages>
using Dm14 = DmaConfig<MfmaBf16, 128, 256, 2, 4, 4>;  // 8 waves of 64x64
using Dm15 = DmaConfig<MfmaBf16, 256, 256, 2, 4, 3>;  // 8 waves of 128x64
using Dm16 = DmaConfig<MfmaBf16, 128, 256, 2, 4, 3>;  // 8 waves of 64x64, 3 LDS stages
using Dm17 = DmaConfig<MfmaBf16, 128, 128, 2, 2, 4>;  // 4 waves of 64x64, 2 blocks per CU
using Dm18 = DmaConfig<MfmaBf16, 128, 256, 2, 4, 5>;  // 8 waves of 64x64, 5 LDS stages
using Dm19 = DmaConfig<MfmaBf16, 256, 128, 2, 2, 4>;  // 4 waves of 128x64
using Dm20 = DmaConfig<MfmaBf16, 128, 256, 2, 2, 4>;  // 4 waves of 64x128
using Dm21 = DmaConfig<MfmaBf16, 128, 256, 2, 2, 3>;  // 4 waves of 64x128, 3 LDS stages
using Dm22 = DmaConfig<MfmaBf16, 128, 256, 2, 2, 5>;  // 4 waves of 64x128, 5 LDS stages
// 128-byte stages (one barrier per 64 bf16 of K); need K % 64 == 0
using Dm23 = DmaConfig<MfmaBf16, 128, 256, 2, 4, 3, 128>;  // 8 waves of 64x64
using Dm24 = DmaConfig<MfmaBf16, 128, 256, 2, 2, 3, 128>;  // 4 waves of 64x128
using Dm25 = DmaConfig<MfmaBf16, 128, 128, 2, 2, 4, 128>;  // 4 waves of 64x64
using Dm26 = DmaConfig<MfmaBf16, 256, 128, 2, 2, 3, 128>;  // 4 waves of 128x64
constexpr int kNumConfigs = 27;
constexpr int kFirstDma = 14, kFirstDma128 = 23;

// Internal epilogue code of vdsl_op_gemm_bf16_gelu_bwd: C (bf16) = v * GELU'(pre) with `pre` an
// input, and the same values transposed into `ctr` ([N][M], optional).
constexpr int kEpiGeluBwd = 100;
// OR-ed into a kernel's `epi` argument when its f32 output is bound as VDSL_BIND_OUTPUT (a result
// for the host that no later device work reads soon): the LDS-staged epilogue then stores it with
// non-temporal hints.  In the config-4 step the weight gradients (2 x 64 MB of f32) stored that way
// no longer leave dirty lines for the next GEMMs to write back: step 372-376 -> 355-358 us.
constexpr int kEpiStreamOut = 0x1000;

// Backward epilogue modes (template argument BWD): 0 = forward (epi selects it), 1 = C = v *
// GELU'(pre) (vdsl_op_gemm_bf16_gelu_bwd), 2 = C = v * g with the factor g given in `pre`
// (vdsl_op_gemm_bf16_mul_packed).  With g = GELU'(pre) from the forward epilogue
// VDSL_EPI_GELU_DERIV, modes 1 and 2 compute the same product and round it the same way.
template <int BWD>
__device__ __forceinline__ float bwd_factor(float p) {
  if constexpr (BWD == 2) return p;
  else return gelu_grad_f(p);
}

// Epilogue of one accumulator element at (row, col), shared by both main loops.  DERIV: the
// kernel runs VDSL_EPI_GELU_DERIV only (a separate instantiation: in the shared forward kernels
// its code made the register allocator spill).
template <int BWD, bool DERIV = false>
__device__ __forceinline__ void bf16_epilogue(float v, int row, int col, int M, int N, void* __restrict__ C,
                                              float* __restrict__ pre, int epi, int c_dtype, uint16_t* __restrict__ ctr) {
  if (row < M && col < N) {
    const size_t o = static_cast<size_t>(row) * N + col;
    if constexpr (BWD != 0) {
      const uint16_t h = f32_to_bf16(v * bwd_factor<BWD>(pre[o]));
      static_cast<uint16_t*>(C)[o] = h;
      if (ctr) ctr[static_cast<size_t>(col) * M + row] = h;
      return;
    }
    if constexpr (DERIV) {
      pre[o] = gelu_grad_f(v);
      static_cast<uint16_t*>(C)[o] = f32_to_bf16(gelu_f(v));
      return;
    }
    if (pre) pre[o] = v;
    float y = v;
    if (epi == VDSL_EPI_GELU) y = gelu_f(v);
    else if (epi == VDSL_EPI_RELU) y = v > 0.0f ? v : 0.0f;
    if (c_dtype == VDSL_F32) static_cast<float*>(C)[o] = y;
    else static_cast<uint16_t*>(C)[o] = f32_to_bf16(y);
  }
}

// Whole-tile epilogue with the variant fixed at compile time: no bounds checks and no per-element
// branches (the generic per-element form costs ~6000 instructions of branchy code per tile).
// Variants: 0 = f32 C, no activation, no pre-activation; 1 = bf16 C = GELU(v) with f32 pre-activation.
template <class Cfg, int VARIANT>
__device__ __forceinline__ void bf16_epilogue_tile(const f32x16 (&acc)[Cfg::FM][Cfg::FN], int m0, int n0, int N,
                                                   void* __restrict__ C, float* __restrict__ pre) {
#pragma unroll
  for (int i = 0; i < Cfg::FM; ++i)
#pragma unroll
    for (int j = 0; j < Cfg::FN; ++j) {
      const int col = acc_col<Cfg>(n0, j);
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const size_t o = static_cast<size_t>(acc_row<Cfg>(m0, i, r)) * N + col;
        const float v = acc[i][j][r];
        if (VARIANT == 0) {
          static_cast<float*>(C)[o] = v;
        } else {
          pre[o] = v;
          static_cast<uint16_t*>(C)[o] = f32_to_bf16(gelu_f(v));
        }
      }
    }
}

// Picks the whole-tile variant when one applies, else the generic per-element epilogue.
template <class Cfg, int BWD, bool DERIV = false>
__device__ __forceinline__ void bf16_store_tile(const f32x16 (&acc)[Cfg::FM][Cfg::FN], int m0, int n0, int M, int N,
                                                void* __restrict__ C, float* __restrict__ pre, int epi, int c_dtype,
                                                uint16_t* __restrict__ ctr) {
  const bool whole = m0 + Cfg::BM <= M && n0 + Cfg::BN <= N;
  if (DERIV) {
#pragma unroll
    for (int i = 0; i < Cfg::FM; ++i)
#pragma unroll
      for (int j = 0; j < Cfg::FN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          bf16_epilogue<0, true>(acc[i][j][r], acc_row<Cfg>(m0, i, r), acc_col<Cfg>(n0, j), M, N, C, pre, epi, c_dtype, ctr);
  } else if (BWD != 0) {
#pragma unroll
    for (int i = 0; i < Cfg::FM; ++i)
#pragma unroll
      for (int j = 0; j < Cfg::FN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          bf16_epilogue<BWD>(acc[i][j][r], acc_row<Cfg>(m0, i, r), acc_col<Cfg>(n0, j), M, N, C, pre, epi, c_dtype, ctr);
  } else if (whole && epi == VDSL_EPI_NONE && c_dtype == VDSL_F32 && !pre) {
    bf16_epilogue_tile<Cfg, 0>(acc, m0, n0, N, C, pre);
  } else if (whole && epi == VDSL_EPI_GELU && c_dtype == VDSL_BF16 && pre) {
    bf16_epilogue_tile<Cfg, 1>(acc, m0, n0, N, C, pre);
  } else {
#pragma unroll
    for (int i = 0; i < Cfg::FM; ++i)
#pragma unroll
      for (int j = 0; j < Cfg::FN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          bf16_epilogue<0>(acc[i][j][r], acc_row<Cfg>(m0, i, r), acc_col<Cfg>(n0, j), M, N, C, pre, epi, c_dtype, ctr);
  }
}

// Whole-tile epilogue staged through LDS (after the main loop, when the block's LDS is free):
// each wave writes one 32-row block of its accumulators to a private LDS area (row stride WTN + 8
// floats: the lanes of one accumulator store, 32 columns x rows 4 apart, hit 64 distinct banks),
// reads it back as 4 consecutive columns per lane and stores 16-byte runs of the f32 output (or
// of the pre-activation) and 8-byte runs of the bf16 output, instead of one 4- or 2-byte store
// per accumulator element.  Needs N % 4 == 0 (aligned runs) and NW * 32 * (WTN + 8) floats of
// LDS; the caller has synchronised the block after the main loop.
template <class Cfg>
constexpr bool kLdsEpilogue = Cfg::NW * 32 * (Cfg::WTN + 8) * 4 <= Cfg::LDS_BYTES;


template <class Cfg, int VARIANT>
__device__ __forceinline__ void bf16_epilogue_tile_lds(const f32x16 (&acc)[Cfg::FM][Cfg::FN], int m0, int n0, int N,
                                                       void* __restrict__ C, float* __restrict__ pre, char* smem) {
  constexpr int WTN = Cfg::WTN, LD = WTN + 8;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave / Cfg::WGN, wn = wave % Cfg::WGN;
  float* const area = reinterpret_cast<float*>(smem) + wave * 32 * LD;
  const int row0 = m0 + wm * Cfg::WTM, col0 = n0 + wn * WTN;
#pragma unroll
  for (int i = 0; i < Cfg::FM; ++i) {
#pragma unroll
    for (int j = 0; j < Cfg::FN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) area[(8 * (r >> 2) + 4 * (lane >> 5) + (r & 3)) * LD + 32 * j + (lane & 31)] = acc[i][j][r];
    constexpr int Q = WTN / 4;  // 16-byte units per row
#pragma unroll
    for (int k = 0; k < 32 * Q / 64; ++k) {
      const int u = lane + 64 * k, row = u / Q, c4 = u % Q;
      const f32x4 v = *reinterpret_cast<const f32x4*>(area + row * LD + 4 * c4);
      const size_t o = static_cast<size_t>(row0 + 32 * i + row) * N + col0 + 4 * c4;
      if (VARIANT == 0) {
        *reinterpret_cast<f32x4*>(static_cast<float*>(C) + o) = v;
      } else if (VARIANT == 3) {  // VARIANT 0 with streaming stores (kEpiStreamOut)
        __builtin_nontemporal_store(v, reinterpret_cast<f32x4*>(static_cast<float*>(C) + o));
      } else {
        if (VARIANT == 1) {
          *reinterpret_cast<f32x4*>(pre + o) = v;
        } else {  // GELU'(v) for the backward pass; erfc(-v / sqrt2) is shared with GELU(v) below
          f32x4 d;
#pragma unroll
          for (int e = 0; e < 4; ++e) d[e] = gelu_grad_f(v[e]);
          *reinterpret_cast<f32x4*>(pre + o) = d;
        }
        uint2 h;
        h.x = pack_bf16x2(gelu_f(v[0]), gelu_f(v[1]));
        h.y = pack_bf16x2(gelu_f(v[2]), gelu_f(v[3]));
        *reinterpret_cast<uint2*>(static_cast<uint16_t*>(C) + o) = h;
      }
    }
  }
}

// Whole-tile GELU-backward epilogue (vdsl_op_gemm_bf16_gelu_bwd), also through each wave's LDS
// area: C = bf16(v * GELU'(pre)) stored as 8-byte runs; the f32 products go back into the area and,
// if `ctr` is set, each lane then reads one column of the 32-row block (64 lanes, 64 consecutive
// floats per read: no bank conflict) and writes it as a 64-byte run of the transposed output
// ctr[N][M] (needs M % 8 == 0 and WTN % 64 == 0).  `pre` is usually cold (written by the forward
// pass long before): every load of it for the wave's whole tile is issued first, before the block
// barrier that ends the main loop, so the tile pays one memory latency instead of one per unit
// (in a training step the per-unit form made this GEMM 38 us slower than without the epilogue).
template <class Cfg, int LDS_AVAIL = Cfg::LDS_BYTES, int BWD = 1>
__device__ __forceinline__ void bf16_epilogue_bwd_lds(const f32x16 (&acc)[Cfg::FM][Cfg::FN], int m0, int n0, int M,
                                                      int N, void* __restrict__ C, const float* __restrict__ pre,
                                                      char* smem, uint16_t* __restrict__ ctr) {
  constexpr int WTN = Cfg::WTN, LD = WTN + 8, Q = WTN / 4, UPL = 32 * Q / 64;  // 16-byte units per lane per row block
  // Rows of the wave's area: the whole wave tile when it fits in the block's LDS (LDS_AVAIL bytes;
  // then each lane's transposed run is WTM * 2 bytes, whole 128-byte lines), else 32.
  constexpr int AR = Cfg::NW * Cfg::WTM * LD * 4 <= LDS_AVAIL ? Cfg::WTM : 32;
  static_assert(WTN % 64 == 0, "the transposed store takes whole columns per lane");
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave / Cfg::WGN, wn = wave % Cfg::WGN;
  float* const area = reinterpret_cast<float*>(smem) + wave * AR * LD;
  const int row0 = m0 + wm * Cfg::WTM, col0 = n0 + wn * WTN;
  f32x4 x[Cfg::FM][UPL];
#pragma unroll
  for (int i = 0; i < Cfg::FM; ++i)
#pragma unroll
    for (int k = 0; k < UPL; ++k) {
      const int u = lane + 64 * k, row = u / Q, c4 = u % Q;
      x[i][k] = __builtin_nontemporal_load(
          reinterpret_cast<const f32x4*>(pre + static_cast<size_t>(row0 + 32 * i + row) * N + col0 + 4 * c4));
    }
  dma_barrier();  // every wave's last fragment reads of the main loop are done
  // The transposed output of rows [r0, r0 + AR) of the wave tile: lane c takes column c and writes
  // AR bf16 (AR * 2 bytes) of ctr row col0 + c.
  auto store_transposed = [&](int r0) {
#pragma unroll
    for (int cc = 0; cc < WTN / 64; ++cc) {
      const int c = lane + 64 * cc;
      u32x4* dst = reinterpret_cast<u32x4*>(ctr + static_cast<size_t>(col0 + c) * M + row0 + r0);
#pragma unroll
      for (int q4 = 0; q4 < AR / 8; ++q4) {
        u32x4 w;
#pragma unroll
        for (int e = 0; e < 4; ++e) w[e] = pack_bf16x2(area[(8 * q4 + 2 * e) * LD + c], area[(8 * q4 + 2 * e + 1) * LD + c]);
        dst[q4] = w;
      }
    }
  };
#pragma unroll
  for (int i = 0; i < Cfg::FM; ++i) {
    float* const blk = area + (AR == 32 ? 0 : 32 * i) * LD;  // this 32-row block's rows of the area
#pragma unroll
    for (int j = 0; j < Cfg::FN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) blk[(8 * (r >> 2) + 4 * (lane >> 5) + (r & 3)) * LD + 32 * j + (lane & 31)] = acc[i][j][r];
#pragma unroll
    for (int k = 0; k < UPL; ++k) {
      const int u = lane + 64 * k, row = u / Q, c4 = u % Q;
      const f32x4 v = *reinterpret_cast<const f32x4*>(blk + row * LD + 4 * c4);
      const size_t o = static_cast<size_t>(row0 + 32 * i + row) * N + col0 + 4 * c4;
      f32x4 d;
#pragma unroll
      for (int e = 0; e < 4; ++e) d[e] = v[e] * bwd_factor<BWD>(x[i][k][e]);
      uint2 h;
      h.x = pack_bf16x2(d[0], d[1]);
      h.y = pack_bf16x2(d[2], d[3]);
      *reinterpret_cast<uint2*>(static_cast<uint16_t*>(C) + o) = h;
      if (ctr) *reinterpret_cast<f32x4*>(blk + row * LD + 4 * c4) = d;
    }
    if (AR == 32 && ctr) store_transposed(32 * i);
  }
  if (AR != 32 && ctr) store_transposed(0);
}

// Whole-tile MSE epilogue (vdsl_op_gemm_bf16_mse_packed), through each wave's LDS area like the
// GELU-backward one: with y the accumulator and d = y - t, dy = bf16(d * scale) as 8-byte runs, y
// as 16-byte runs (if wanted), dy^T through the area (each lane one column, AR * 2-byte runs of
// dy_t[N][M]), and the wave's sum of d^2 in f64 (lane order: 32-row block, unit, component; then a
// butterfly over the wave) into *part.  t, like `pre` there, is cold: every load of the wave's
// tile is issued before the block barrier that ends the main loop.  The arithmetic of d, dy and
// its rounding is that of mse_tile_vec (autodiff.hip), so dy and dy_t equal the unfused op's.
template <class Cfg, int LDS_AVAIL>
__device__ __forceinline__ void bf16_epilogue_mse_lds(const f32x16 (&acc)[Cfg::FM][Cfg::FN], int m0, int n0, int M, int N,
                                                      const float* __restrict__ t, float scale, float* __restrict__ y,
                                                      uint16_t* __restrict__ dy, uint16_t* __restrict__ dyt,
                                                      double* __restrict__ part, char* smem) {
  constexpr int WTN = Cfg::WTN, LD = WTN + 8, Q = WTN / 4, UPL = 32 * Q / 64;
  constexpr int AR = Cfg::NW * Cfg::WTM * LD * 4 <= LDS_AVAIL ? Cfg::WTM : 32;
  static_assert(WTN % 64 == 0, "the transposed store takes whole columns per lane");
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave / Cfg::WGN, wn = wave % Cfg::WGN;
  float* const area = reinterpret_cast<float*>(smem) + wave * AR * LD;
  const int row0 = m0 + wm * Cfg::WTM, col0 = n0 + wn * WTN;
  f32x4 x[Cfg::FM][UPL];
#pragma unroll
  for (int i = 0; i < Cfg::FM; ++i)
#pragma unroll
    for (int k = 0; k < UPL; ++k) {
      const int u = lane + 64 * k, row = u / Q, c4 = u % Q;
      x[i][k] = __builtin_nontemporal_load(
          reinterpret_cast<const f32x4*>(t + static_cast<size_t>(row0 + 32 * i + row) * N + col0 + 4 * c4));
    }
  dma_barrier();  // every wave's last fragment reads of the main loop are done
  auto store_transposed = [&](int r0) {
#pragma unroll
    for (int cc = 0; cc < WTN / 64; ++cc) {
      const int c = lane + 64 * cc;
      u32x4* dst = reinterpret_cast<u32x4*>(dyt + static_cast<size_t>(col0 + c) * M + row0 + r0);
#pragma unroll
      for (int q4 = 0; q4 < AR / 8; ++q4) {
        u32x4 w;
#pragma unroll
        for (int e = 0; e < 4; ++e) w[e] = pack_bf16x2(area[(8 * q4 + 2 * e) * LD + c], area[(8 * q4 + 2 * e + 1) * LD + c]);
        dst[q4] = w;
      }
    }
  };
  double s = 0.0;
#pragma unroll
  for (int i = 0; i < Cfg::FM; ++i) {
    float* const blk = area + (AR == 32 ? 0 : 32 * i) * LD;
#pragma unroll
    for (int j = 0; j < Cfg::FN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) blk[(8 * (r >> 2) + 4 * (lane >> 5) + (r & 3)) * LD + 32 * j + (lane & 31)] = acc[i][j][r];
#pragma unroll
    for (int k = 0; k < UPL; ++k) {
      const int u = lane + 64 * k, row = u / Q, c4 = u % Q;
      const f32x4 v = *reinterpret_cast<const f32x4*>(blk + row * LD + 4 * c4);
      const size_t o = static_cast<size_t>(row0 + 32 * i + row) * N + col0 + 4 * c4;
      f32x4 g;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float d = v[e] - x[i][k][e];
        s += static_cast<double>(d) * static_cast<double>(d);
        g[e] = d * scale;
      }
      uint2 h;
      h.x = pack_bf16x2(g[0], g[1]);
      h.y = pack_bf16x2(g[2], g[3]);
      *reinterpret_cast<uint2*>(dy + o) = h;
      if (y) *reinterpret_cast<f32x4*>(y + o) = v;
      if (dyt) *reinterpret_cast<f32x4*>(blk + row * LD + 4 * c4) = g;
    }
    if (AR == 32 && dyt) store_transposed(32 * i);
  }
  if (AR != 32 && dyt) store_transposed(0);
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) s += __shfl_xor(s, m, 64);
  if (lane == 0) *part = s;
}

template <class Cfg, bool EDGE, bool BWD>
__global__ __launch_bounds__(Cfg::NT, Cfg::MIN_BLOCKS) void gemm_bf16_nt(const uint16_t* __restrict__ A, const uint16_t* __restrict__ B,
                                                        void* __restrict__ C, float* __restrict__ pre, int M, int N, int K,
                                                        int epi, int c_dtype, uint16_t* __restrict__ ctr) {
  __shared__ __attribute__((aligned(16))) char smem[Cfg::LDS_BYTES];
  epi &= ~kEpiStreamOut;  // this kernel's epilogue stores per element, with plain stores
  const int tiles_m = (M + Cfg::BM - 1) / Cfg::BM, tiles_n = (N + Cfg::BN - 1) / Cfg::BN;
  int tm, tn;
  tile_coords(xcd_remap(blockIdx.x, gridDim.x), tiles_m, tiles_n, tm, tn);
  const int m0 = tm * Cfg::BM, n0 = tn * Cfg::BN;
  f32x16 acc[Cfg::FM][Cfg::FN];
  gemm_mainloop<MfmaBf16, Cfg, EDGE>(reinterpret_cast<const char*>(A), reinterpret_cast<const char*>(B), M, N, K * 2, 0, K * 2,
                               m0, n0, smem, acc);
  bf16_store_tile<Cfg, BWD>(acc, m0, n0, M, N, C, pre, epi, c_dtype, ctr);
}

// Direct-to-LDS kernel (gemm_dma.h).  Blocks of 8 waves are sized for one block per CU, blocks
// of 4 waves for two.  BKN: B stored [K][N] (the "NN" form, no transpose first; N % 256 == 0).
// AKM: A stored [K][M] (trans_a; M % 256 == 0), read K-major as well.
template <class Cfg, bool BWD, bool BKN = false, bool AKM = false>
__global__ __launch_bounds__(Cfg::NT, Cfg::MIN_BLOCKS) void gemm_bf16_dma(const uint16_t* __restrict__ A,
                                                                               const uint16_t* __restrict__ B,
                                                                               void* __restrict__ C, float* __restrict__ pre,
                                                                               int M, int N, int K, int epi, int c_dtype,
                                                                               uint16_t* __restrict__ ctr) {
  __shared__ __attribute__((aligned(1024))) char smem[Cfg::LDS_BYTES];
  const bool stream = (epi & kEpiStreamOut) != 0;
  epi &= ~kEpiStreamOut;
  const int tiles_m = (M + Cfg::BM - 1) / Cfg::BM, tiles_n = (N + Cfg::BN - 1) / Cfg::BN;
  int tm, tn;
  tile_coords(xcd_remap(blockIdx.x, gridDim.x), tiles_m, tiles_n, tm, tn);
  const int m0 = tm * Cfg::BM, n0 = tn * Cfg::BN;
  f32x16 acc[Cfg::FM][Cfg::FN];
  dma_mainloop<MfmaBf16, Cfg, f32x16, Cfg::FM, Cfg::FN, BKN, AKM>(reinterpret_cast<const char*>(A),
                                                                  reinterpret_cast<const char*>(B), M, N, K * 2, 0, K * 2, m0,
                                                                  n0, smem, acc, N * 2, M * 2);
  if constexpr (kLdsEpilogue<Cfg>) {
    // Block-uniform: the tile is whole, N allows aligned runs, and the epilogue is one the LDS path has.
    const bool whole = m0 + Cfg::BM <= M && n0 + Cfg::BN <= N && N % 4 == 0;
    if constexpr (BWD) {
      if constexpr (Cfg::WTN % 64 == 0 && Cfg::FM * Cfg::WTN / 2 <= 64) {  // pre prefetch: FM * WTN / 2 VGPRs
        if (whole && (!ctr || M % 8 == 0)) {
          bf16_epilogue_bwd_lds<Cfg>(acc, m0, n0, M, N, C, pre, smem, ctr);
          return;
        }
      }
    } else {
      const bool v0 = epi == VDSL_EPI_NONE && c_dtype == VDSL_F32 && !pre;
      const bool v1 = epi == VDSL_EPI_GELU && c_dtype == VDSL_BF16 && pre;
      if (whole && (v0 || v1)) {
        dma_barrier();  // every wave's last fragment reads of the main loop are done
        if (v0 && stream) bf16_epilogue_tile_lds<Cfg, 3>(acc, m0, n0, N, C, pre, smem);
        else if (v0) bf16_epilogue_tile_lds<Cfg, 0>(acc, m0, n0, N, C, pre, smem);
        else bf16_epilogue_tile_lds<Cfg, 1>(acc, m0, n0, N, C, pre, smem);
        return;
      }
    }
  }
  bf16_store_tile<Cfg, BWD>(acc, m0, n0, M, N, C, pre, epi, c_dtype, ctr);
}

// Any K (including K % 8 != 0): one lane per output, f32 accumulate in k order.
__global__ __launch_bounds__(256) void gemm_bf16_nt_simple(const uint16_t* __restrict__ A, const uint16_t* __restrict__ B,
                                                           void* __restrict__ C, float* __restrict__ pre, int M, int N,
                                                           int K, int epi, int c_dtype, uint16_t* __restrict__ ctr) {
  const int64_t idx = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (idx >= static_cast<int64_t>(M) * N) return;
  epi &= ~kEpiStreamOut;
  const int row = static_cast<int>(idx / N), col = static_cast<int>(idx % N);
  float v = 0.0f;
  for (int k = 0; k < K; ++k)
    v = __builtin_fmaf(bf16_to_f32(A[static_cast<size_t>(row) * K + k]), bf16_to_f32(B[static_cast<size_t>(col) * K + k]), v);
  if (epi == kEpiGeluBwd) {
    const uint16_t h = f32_to_bf16(v * gelu_grad_f(pre[idx]));
    static_cast<uint16_t*>(C)[idx] = h;
    if (ctr) ctr[static_cast<size_t>(col) * M + row] = h;
    return;
  }
  if (pre) pre[idx] = v;
  float y = v;
  if (epi == VDSL_EPI_GELU) y = gelu_f(v);
  else if (epi == VDSL_EPI_RELU) y = v > 0.0f ? v : 0.0f;
  if (c_dtype == VDSL_F32) static_cast<float*>(C)[idx] = y;
  else static_cast<uint16_t*>(C)[idx] = f32_to_bf16(y);
}

// The GELU-backward epilogue per element with a 32-row block's loads of `pre` issued before the first is
// used (clamped to the tensor; one load per element and branch waited for each in turn: 300x1000x10 10.0 us, 7.2 here).
template <class Cfg, int BWD>
__device__ __forceinline__ void bf16_store_tile_bwd(const f32x16 (&acc)[Cfg::FM][Cfg::FN], int m0, int n0, int M, int N,
                                                    void* __restrict__ C, const float* __restrict__ pre,
                                                    uint16_t* __restrict__ ctr) {
#pragma unroll
  for (int i = 0; i < Cfg::FM; ++i) {
    float x[Cfg::FN][16];
#pragma unroll
    for (int j = 0; j < Cfg::FN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        x[j][r] = pre[static_cast<size_t>(min(acc_row<Cfg>(m0, i, r), M - 1)) * N + min(acc_col<Cfg>(n0, j), N - 1)];
#pragma unroll
    for (int j = 0; j < Cfg::FN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int row = acc_row<Cfg>(m0, i, r), col = acc_col<Cfg>(n0, j);
        const uint16_t h = f32_to_bf16(acc[i][j][r] * bwd_factor<BWD>(x[j][r]));
        if (row < M && col < N) {
          static_cast<uint16_t*>(C)[static_cast<size_t>(row) * N + col] = h;
          if (ctr) ctr[static_cast<size_t>(col) * M + row] = h;
        }
      }
  }
}

// ---- operands as they are stored, any extents (gemm_any.h) -----------------------------------------
template <class Cfg, bool BWD>
__global__ __launch_bounds__(Cfg::NT) void gemm_bf16_any(const uint16_t* __restrict__ A, const uint16_t* __restrict__ B,
                                                         void* __restrict__ C, float* __restrict__ pre, int M, int N, int K,
                                                         int epi, int c_dtype, uint16_t* __restrict__ ctr) {
  __shared__ __attribute__((aligned(16))) char smem[Cfg::LDS_BYTES];
  const int tiles_m = (M + Cfg::BM - 1) / Cfg::BM, tiles_n = (N + Cfg::BN - 1) / Cfg::BN;
  int tm, tn;
  tile_coords(xcd_remap(blockIdx.x, gridDim.x), tiles_m, tiles_n, tm, tn);
  f32x16 acc[Cfg::FM][Cfg::FN];
  any_mainloop<Cfg>(A, B, M, N, K, tm * Cfg::BM, tn * Cfg::BN, smem, acc);
  if constexpr (BWD) bf16_store_tile_bwd<Cfg, 1>(acc, tm * Cfg::BM, tn * Cfg::BN, M, N, C, pre, ctr);
  else bf16_store_tile<Cfg, 0>(acc, tm * Cfg::BM, tn * Cfg::BN, M, N, C, pre, epi & ~kEpiStreamOut, c_dtype, ctr);
}

int64_t tiles64(int64_t M, int64_t N) { return ((M + 63) / 64) * ((N + 63) / 64); }

// Both operands hold the 16 bytes that its loads take at least, and no configuration is forced.
bool any_runs(int64_t M, int64_t N, int64_t K) { return M * K >= 8 && N * K >= 8 && gemm_config_override() < 0; }

template <bool AKM, bool BKM>
int launch_any_form(const uint16_t* A, const uint16_t* B, void* C, float* pre, int M, int N, int K, int epi, int ct, hipStream_t s,
                    uint16_t* ctr) {
  const auto go = [&](auto cfg) {
    using Cfg = decltype(cfg);
    const int64_t tiles = ((int64_t{M} + Cfg::BM - 1) / Cfg::BM) * ((int64_t{N} + Cfg::BN - 1) / Cfg::BN);
    if (tiles > 0x7fffffff) return fail(VDSL_ERR_UNSUPPORTED, "GEMM: too many tiles");
    if (epi == kEpiGeluBwd)
      hipLaunchKernelGGL((gemm_bf16_any<Cfg, true>), dim3(static_cast<unsigned>(tiles)), dim3(Cfg::NT), 0, s, A, B, C, pre, M, N, K,
                         epi, ct, ctr);
    else
      hipLaunchKernelGGL((gemm_bf16_any<Cfg, false>), dim3(static_cast<unsigned>(tiles)), dim3(Cfg::NT), 0, s, A, B, C, pre, M, N,
                         K, epi, ct, ctr);
    return check_launch("gemm_bf16_any");
  };
  // 64 x 64 tiles below 1024 of them (3000x1000x600 16.3 us against 19.3 with 128 x 128, 512^3 6.4 against
  // 10.4), 128 x 128 from there on (2048^3 31.1 against 35.4, 4000x4000x2000 102 against 181).
  if (tiles64(M, N) < 1024) return go(AnyConfig<64, 64, 2, 2, AKM, BKM>{});
  return go(AnyConfig<128, 128, 2, 2, AKM, BKM>{});
}

// A stored [K][M] if ta, B stored [K][N] if !tb; any_runs(M, N, K).
int launch_any(bool ta, bool tb, const uint16_t* A, const uint16_t* B, void* C, float* pre, int M, int N, int K, int epi, int ct,
               hipStream_t s, uint16_t* ctr = nullptr) {
  if (ta) return tb ? launch_any_form<true, false>(A, B, C, pre, M, N, K, epi, ct, s, ctr)
                    : launch_any_form<true, true>(A, B, C, pre, M, N, K, epi, ct, s, ctr);
  return tb ? launch_any_form<false, false>(A, B, C, pre, M, N, K, epi, ct, s, ctr)
            : launch_any_form<false, true>(A, B, C, pre, M, N, K, epi, ct, s, ctr);
}

// ---- products with a short side (gemm_skinny.h) -----------------------------------------------------
// Epilogue kinds of one kernel: the forward ones (`epi` selects it), the two backward ones and
// VDSL_EPI_GELU_DERIV, as bf16_epilogue's template arguments.
enum { kSkinnyForward = 0, kSkinnyGeluBwd = 1, kSkinnyMul = 2, kSkinnyDeriv = 3 };

// SWAP: the operands are given exchanged (A is the [N][K] one), so that a short N is the side held in
// fragments; row and col are then C's column and row.
template <class Cfg, bool SWAP>
__global__ __launch_bounds__(Cfg::THREADS) void gemm_bf16_skinny(const uint16_t* __restrict__ A, const uint16_t* __restrict__ B,
                                                                 void* __restrict__ C, float* __restrict__ pre, int M, int N,
                                                                 int K, int kind, int epi, int c_dtype,
                                                                 uint16_t* __restrict__ ctr) {
  const int cm = SWAP ? N : M, cn = SWAP ? M : N;  // C's extents
  const unsigned tiles_n = (static_cast<unsigned>(N) + Cfg::BN - 1) / Cfg::BN;
  const int m0 = static_cast<int>(blockIdx.x / tiles_n) * Cfg::BM, n0 = static_cast<int>(blockIdx.x % tiles_n) * Cfg::BN;
  const char *a = reinterpret_cast<const char*>(A), *b = reinterpret_cast<const char*>(B);
  const auto out = [&](int i, int j, float v) {
    const int row = SWAP ? j : i, col = SWAP ? i : j;
    if (kind == kSkinnyForward) bf16_epilogue<0>(v, row, col, cm, cn, C, pre, epi, c_dtype, ctr);
    else if (kind == kSkinnyGeluBwd) bf16_epilogue<1>(v, row, col, cm, cn, C, pre, epi, c_dtype, ctr);
    else if (kind == kSkinnyMul) bf16_epilogue<2>(v, row, col, cm, cn, C, pre, epi, c_dtype, ctr);
    else bf16_epilogue<0, true>(v, row, col, cm, cn, C, pre, epi, c_dtype, ctr);
  };
  if constexpr (Cfg::LDS_BYTES == 0) {
    skinny_direct<Cfg>(a, b, M, N, 2 * K, m0, n0, out);
  } else {
    __shared__ __attribute__((aligned(16))) char smem[Cfg::LDS_BYTES];
    skinny_chain<Cfg>(a, b, M, N, 2 * K, m0, n0, smem, out);
  }
}

// Whether a product takes gemm_skinny.h.  Every path gives the same bits, so the rule is by time alone
// (us, operands rotating).  Packed: up to 16 rows, up to 32 below 16384 columns: [M][4096] x [4096][4096] in
// the tiles of bpk_dispatch and here: M = 1 18.6, 9.3; 8 19.0, 11.1; 16 19.3, 11.9; 32 18.8, 15.2; [20][4096] x
// [16384] 28.8, 31.0; [1000][4096] x [32] 15.6, 18.1.  Row-major, in the tiles of launch_nt and here: a side
// of at most 32 ([8][4096] x [4096] 30.2, 11.2; [300][1000] x [10] 10.8, 4.3), or below 128 while the tiles of
// 64 x 64 leave CUs idle ([64][4000] x [4000] 30.5, 22.4; [127][300] x [500] 6.4, 4.2; [64][200] x [16000] 6.1, 8.4;
// [127][1000] x [8000] 12.2, 15.9); of rows that are not whole 16-byte units, up to 8192 of the long side
// ([8][1001] x [4096] 10.6, 6.8; [31][255] x [10000] 7.1, 10.6), where waves do not load for themselves.
bool skinny_runs(bool packed, int64_t M, int64_t N, int64_t K) {
  const int64_t s = M < N ? M : N, l = M < N ? N : M;
  if (s * K < 8 || l > 0x7fffff00 || gemm_config_override() >= 0) return false;
  if (packed) return M <= 16 || (M <= 32 && (N < 16384 || direct_runs(M, N, K)));
  if (K % 8 != 0 && l > 8192 && !direct_runs(s, l, K)) return false;
  return s <= 32 || (s < 128 && ((s + 63) / 64) * ((l + 31) / 32) <= 256);
}

template <SkinnyForm FORM, bool SWAP>
int launch_skinny_form(const uint16_t* A, const uint16_t* B, void* C, float* pre, int M, int N, int K, int kind, int epi, int ct,
                       hipStream_t s, uint16_t* ctr) {
  return chain_dispatch<FORM>(M, N, K, [&](auto cfg) {
    using Cfg = decltype(cfg);
    const int64_t blocks = ((int64_t{N} + Cfg::BN - 1) / Cfg::BN) * ((int64_t{M} + Cfg::BM - 1) / Cfg::BM);
    if (blocks > 0x7fffffff) return fail(VDSL_ERR_UNSUPPORTED, "GEMM: too many tiles");
    const dim3 g(static_cast<unsigned>(blocks));
    hipLaunchKernelGGL((gemm_bf16_skinny<Cfg, SWAP>), g, dim3(Cfg::THREADS), 0, s, A, B, C, pre, M, N, K, kind,
                       epi & ~kEpiStreamOut, ct, ctr);
    return check_launch("gemm_bf16_skinny");
  });
}

int launch_skinny(bool packed, const uint16_t* A, const uint16_t* B, void* C, float* pre, int M, int N, int K, int kind, int epi,
                  int ct, hipStream_t s, uint16_t* ctr) {
  if (packed) return launch_skinny_form<kSkinnyPacked, false>(A, B, C, pre, M, N, K, kind, epi, ct, s, ctr);
  if (M <= N) return launch_skinny_form<kSkinnyRows, false>(A, B, C, pre, M, N, K, kind, epi, ct, s, ctr);
  return launch_skinny_form<kSkinnyRows, true>(B, A, C, pre, N, M, K, kind, epi, ct, s, ctr);
}

// ---- packed-weight form (gemm_bpk.h main loop): B in MFMA fragment order, A through LDS --------
// For constant weights (forward GEMMs on [out][in] weights): the weight is packed once and each
// wave loads its B fragments straight into registers.  Same k-steps in the same order with the same
// MFMA as every other configuration, so the same results bit for bit.  Measured standalone on
// 2048x4096x4096 (random bf16, f32 out): 61-63 us against 66-68 us for the direct-to-LDS kernel.
using Pb0 = BpkConfig<MfmaBf16, 4, 2, 4, 3>;  // 128 x 256 blocks, 4 waves of 128 x 64
// Smaller tiles for outputs that give 128 x 256 blocks to a part of the CUs.
using Pb1 = BpkConfig<MfmaBf16, 4, 1, 4, 3>;  // 128 x 128 blocks, 4 waves of 128 x 32
using Pb2 = BpkConfig<MfmaBf16, 2, 1, 4, 3>;  // 64 x 128 blocks, 4 waves of 64 x 32
using Pb3 = BpkConfig<MfmaBf16, 2, 1, 2, 3>;  // 64 x 64 blocks, 2 waves of 64 x 32
using Pb4 = BpkConfig<MfmaBf16, 1, 1, 2, 3>;  // 32 x 64 blocks, 2 waves of 32 x 32

// Calls go(Cfg{}, tiles) with the tile of a packed product.  A CU takes in about 55 GB/s of operands
// from its L2, so a launch lasts as long as the operand bytes of its busiest CU: rounds of tiles over
// the 256 CUs times the tile's rows and columns; a smaller tile is taken where that is less by a tenth
// or more.  K = 4096, N = 4096, us for 128 x 256 and the choice: M = 64 47.8, 14.4 (32 x 64); 128 40.6, 15.2
// (32 x 64); 300 46.5, 26.3 (64 x 128); 512 51.5, 28.7 (64 x 128); 2048 65.9 (128 x 256; 128 x 128 78.7);
// [2048][4096] x [1024] 41.7, 22.7 (64 x 128), [512][2048] x [2048] 23.5, 10.9 (64 x 64).  The backward forms gain
// alike, though tiles below 64 columns a wave store their outputs element by element: GELU backward with the
// transposed output, [64][4096] x [4096] 87, 21.7; [300] 123, 34; [2048][4096] x [1024] 69, 36.7; times a factor 81,
// 20.3; 112, 32.9; 60, 35.7.
template <class Go>
int bpk_dispatch(int64_t M, int64_t N, Go&& go) {
  const auto tiles = [&](int bm, int bn) { return ((M + bm - 1) / bm) * ((N + bn - 1) / bn); };
  const int sizes[5][2] = {{128, 256}, {128, 128}, {64, 128}, {64, 64}, {32, 64}};
  int best = 0;
  int64_t cost = 0;
  for (int c = 0; c < 5; ++c) {
    const int64_t t = (tiles(sizes[c][0], sizes[c][1]) + 255) / 256 * (sizes[c][0] + sizes[c][1]);
    if (c == 0 || 10 * t <= 9 * cost) best = c, cost = t;
  }
  const int64_t n = tiles(sizes[best][0], sizes[best][1]);
  if (best == 1) return go(Pb1{}, n);
  if (best == 2) return go(Pb2{}, n);
  if (best == 3) return go(Pb3{}, n);
  if (best == 4) return go(Pb4{}, n);
  return go(Pb0{}, n);
}

// BWD: the backward epilogues (1: vdsl_op_gemm_bf16_gelu_bwd_packed, C = da, pre an input, ctr =
// da^T; 2: vdsl_op_gemm_bf16_mul_packed, the factor given); their LDS is enlarged so the whole wave
// tile stages at once (whole-line transposed stores).
template <class Cfg, bool BWD>
constexpr int bpk_bf16_smem() {
  return BWD && Cfg::NW * Cfg::WTM * (Cfg::WTN + 8) * 4 > Cfg::LDS_BYTES ? Cfg::NW * Cfg::WTM * (Cfg::WTN + 8) * 4
                                                                          : Cfg::LDS_BYTES;
}

// BWD: the backward epilogue mode (bf16_epilogue); DERIV: the forward VDSL_EPI_GELU_DERIV kernel.
template <class Cfg, int BWD, bool DERIV = false>
__global__ __launch_bounds__(Cfg::NT, 1) void gemm_bf16_bpk(const uint16_t* __restrict__ A, const uint16_t* __restrict__ Bp,
                                                         void* __restrict__ C, float* __restrict__ pre, int M, int N, int K,
                                                         int epi, int c_dtype, uint16_t* __restrict__ ctr) {
  // The only __shared__ variable (see gemm_bpk.h); after the main loop it stages the epilogue.
  __shared__ __attribute__((aligned(1024))) char smem[bpk_bf16_smem<Cfg, BWD != 0>()];
  const bool stream = (epi & kEpiStreamOut) != 0;
  epi &= ~kEpiStreamOut;
  // Tiles in groups of 8 tile-rows, walked column-major (tile_coords): the 32 blocks one XCD runs
  // (congruent ids, made consecutive by xcd_remap) then cover 8 row tiles x 4 column panels, so
  // each XCD's L2 fetches 1/2 of A and 1/4 of B (2048x4096x4096: 128 MB fetched in all, against
  // 168 MB when each XCD took 16 row tiles x 2 panels).
  const int tiles_m = (M + Cfg::BM - 1) / Cfg::BM, tiles_n = (N + Cfg::BN - 1) / Cfg::BN;
  int tm, tn;
  tile_coords(xcd_remap(blockIdx.x, gridDim.x), tiles_m, tiles_n, tm, tn);
  const int m0 = tm * Cfg::BM, n0 = tn * Cfg::BN;
  f32x16 acc[Cfg::FM][Cfg::FN];
  bpk_mainloop<MfmaBf16, Cfg>(reinterpret_cast<const char*>(A), reinterpret_cast<const char*>(Bp), M, N / 32, K * 2, 0, K * 2,
                              m0, n0, smem, acc);
  static_assert(kLdsEpilogue<Cfg>, "the LDS-staged epilogue must fit the main loop's LDS");
  const bool whole = m0 + Cfg::BM <= M && n0 + Cfg::BN <= N && N % 4 == 0;
  if constexpr (BWD != 0 && Cfg::WTN % 64 != 0) {
    bf16_store_tile_bwd<Cfg, BWD>(acc, m0, n0, M, N, C, pre, ctr);
    return;
  } else if constexpr (BWD != 0) {
    if (whole && (!ctr || M % 8 == 0)) {
      bf16_epilogue_bwd_lds<Cfg, bpk_bf16_smem<Cfg, true>(), BWD>(acc, m0, n0, M, N, C, pre, smem, ctr);
      return;
    }
  } else if constexpr (DERIV) {
    if (whole) {
      __syncthreads();  // every wave is past its last read of the main loop's LDS
      bf16_epilogue_tile_lds<Cfg, 2>(acc, m0, n0, N, C, pre, smem);
      return;
    }
  } else {
    const bool v0 = epi == VDSL_EPI_NONE && c_dtype == VDSL_F32 && !pre;
    const bool v1 = epi == VDSL_EPI_GELU && c_dtype == VDSL_BF16 && pre;
    if (whole && (v0 || v1)) {
      __syncthreads();  // every wave is past its last read of the main loop's LDS
      if (v0 && stream) bf16_epilogue_tile_lds<Cfg, 3>(acc, m0, n0, N, C, pre, smem);
      else if (v0) bf16_epilogue_tile_lds<Cfg, 0>(acc, m0, n0, N, C, pre, smem);
      else bf16_epilogue_tile_lds<Cfg, 1>(acc, m0, n0, N, C, pre, smem);
      return;
    }
  }
  bf16_store_tile<Cfg, BWD, DERIV>(acc, m0, n0, M, N, C, pre, epi, c_dtype, ctr);
}

// The packed GEMM fused with the MSE loss of its f32 output (vdsl_op_gemm_bf16_mse_packed): whole
// tiles only; partials[tile * W + wave] receives each wave's sum of squared differences.
template <class Cfg>
__global__ __launch_bounds__(Cfg::NT, 1) void gemm_bf16_bpk_mse(const uint16_t* __restrict__ A, const uint16_t* __restrict__ Bp,
                                                             const float* __restrict__ t, float* __restrict__ y,
                                                             uint16_t* __restrict__ dy, uint16_t* __restrict__ dyt,
                                                             double* __restrict__ partials, int M, int N, int K, float scale) {
  __shared__ __attribute__((aligned(1024))) char smem[bpk_bf16_smem<Cfg, true>()];
  const int tiles_m = M / Cfg::BM, tiles_n = N / Cfg::BN;
  int tm, tn;
  tile_coords(xcd_remap(blockIdx.x, gridDim.x), tiles_m, tiles_n, tm, tn);
  const int m0 = tm * Cfg::BM, n0 = tn * Cfg::BN;
  f32x16 acc[Cfg::FM][Cfg::FN];
  bpk_mainloop<MfmaBf16, Cfg>(reinterpret_cast<const char*>(A), reinterpret_cast<const char*>(Bp), M, N / 32, K * 2, 0, K * 2,
                              m0, n0, smem, acc);
  double* const part = partials + (static_cast<size_t>(tm) * tiles_n + tn) * Cfg::W + (threadIdx.x >> 6);
  bf16_epilogue_mse_lds<Cfg, bpk_bf16_smem<Cfg, true>()>(acc, m0, n0, M, N, t, scale, y, dy, dyt, part, smem);
}

template <class Cfg>
int launch_cfg(const uint16_t* A, const uint16_t* B, void* C, float* pre, int M, int N, int K, int epi, int ct, hipStream_t s,
               uint16_t* ctr) {
  const int64_t tiles = static_cast<int64_t>((M + Cfg::BM - 1) / Cfg::BM) * ((N + Cfg::BN - 1) / Cfg::BN);
  const dim3 g(static_cast<unsigned>(tiles)), b(Cfg::NT);
  const bool edge = gemm_needs_edge<Cfg>(M, N, static_cast<int64_t>(K) * 2);
  if (epi == kEpiGeluBwd) {
    if (edge) hipLaunchKernelGGL((gemm_bf16_nt<Cfg, true, true>), g, b, 0, s, A, B, C, pre, M, N, K, epi, ct, ctr);
    else hipLaunchKernelGGL((gemm_bf16_nt<Cfg, false, true>), g, b, 0, s, A, B, C, pre, M, N, K, epi, ct, ctr);
  } else {
    if (edge) hipLaunchKernelGGL((gemm_bf16_nt<Cfg, true, false>), g, b, 0, s, A, B, C, pre, M, N, K, epi, ct, ctr);
    else hipLaunchKernelGGL((gemm_bf16_nt<Cfg, false, false>), g, b, 0, s, A, B, C, pre, M, N, K, epi, ct, ctr);
  }
  return check_launch("gemm_bf16_nt");
}

template <class Cfg>
int launch_dma(const uint16_t* A, const uint16_t* B, void* C, float* pre, int M, int N, int K, int epi, int ct, hipStream_t s,
               uint16_t* ctr) {
  const int64_t tiles = static_cast<int64_t>((M + Cfg::BM - 1) / Cfg::BM) * ((N + Cfg::BN - 1) / Cfg::BN);
  if (epi == kEpiGeluBwd)
    hipLaunchKernelGGL((gemm_bf16_dma<Cfg, true>), dim3(static_cast<unsigned>(tiles)), dim3(Cfg::NT), 0, s, A, B, C, pre, M, N, K, epi,
                       ct, ctr);
  else
    hipLaunchKernelGGL((gemm_bf16_dma<Cfg, false>), dim3(static_cast<unsigned>(tiles)), dim3(Cfg::NT), 0, s, A, B, C, pre, M, N, K,
                       epi, ct, ctr);
  return check_launch("gemm_bf16_dma");
}

// The "NN" form (B stored [K][N]) without a transpose: the direct-to-LDS configurations with
// 256-wide tiles read B K-major (gemm_dma.h) when every tile is whole along N.  With akm, the "TN"
// form (A stored [K][M] as well, e.g. dW = g^T x with g [batch][out] as stored): the 256 x 256
// configuration reads both operands K-major when M % 256 == 0 too.  Returns 1 (never a status)
// when the shape needs the transpose path instead.
bool dma_kn_runs(int cfg, int64_t M, int64_t N, bool akm) {
  if (N % 256 != 0) return false;
  return akm ? (M % 256 == 0 && cfg == 15) : (cfg == 15 || cfg == 23);
}

int launch_dma_kn(int cfg, const uint16_t* A, const uint16_t* B, void* C, float* pre, int M, int N, int K, int epi, int ct,
                  hipStream_t s, bool akm = false) {
  if (!dma_kn_runs(cfg, M, N, akm)) return 1;
  auto go = [&](auto cfg_tag, auto akm_tag) {
    using Cfg = decltype(cfg_tag);
    constexpr bool kAkm = decltype(akm_tag)::value;
    const int64_t tiles = static_cast<int64_t>((M + Cfg::BM - 1) / Cfg::BM) * (N / Cfg::BN);
    hipLaunchKernelGGL((gemm_bf16_dma<Cfg, false, true, kAkm>), dim3(static_cast<unsigned>(tiles)), dim3(Cfg::NT), 0, s, A, B, C,
                       pre, M, N, K, epi, ct, nullptr);
    return check_launch(kAkm ? "gemm_bf16_dma<K-major A and B>" : "gemm_bf16_dma<K-major B>");
  };
  if (akm) return go(Dm15{}, std::true_type{});
  if (cfg == 15) return go(Dm15{}, std::false_type{});
  if (cfg == 23) return go(Dm23{}, std::false_type{});
  return 1;
}

// Configuration for a shape.  The direct-to-LDS loop (14..) runs whenever K is a whole number of
// its 64-byte stages (K % 32 == 0); measured on MI355X with random operands (bf16, f32 out):
// 128x256 blocks of 8 waves are fastest while they still give every CU a block, with 128-byte
// stages and fragments read two k-steps ahead when K % 64 == 0 (2048x4096x4096: 890-915 TFLOP/s
// against 845-860 with 64-byte stages), 256x256 blocks once those do (4096x4096x2048: 955 against
// 870).  Smaller launches take 128x128 blocks, two per CU.  Other K use the register-staged loop
// (0..13), where 128x128 tiles are fastest below 512 tiles of 256x128 and 256x128 tiles of 8
// waves above.
int choose_config(int64_t M, int64_t N, int64_t K) {
  const bool dma = dma_k_ok(0, K * 2), dma128 = dma_k_ok(0, K * 2, 128);
  const int o = gemm_config_override();
  if (o >= 0 && o < kNumConfigs && (o < kFirstDma || (o < kFirstDma128 ? dma : dma128))) return o;
  if (dma) {
    const int64_t t256 = ((M + 255) / 256) * ((N + 255) / 256);
    const int64_t t128x256 = ((M + 127) / 128) * ((N + 255) / 256);
    if (t256 >= 240) return 15;
    if (t128x256 >= 128) return dma128 ? 23 : 14;
    return 17;
  }
  const int64_t tiles_256x128 = ((M + 255) / 256) * ((N + 127) / 128);
  return tiles_256x128 >= 512 ? 13 : 0;
}

int launch_nt(const uint16_t* A, const uint16_t* B, void* C, float* pre, int M, int N, int K, int epi, int ct, hipStream_t s,
              uint16_t* ctr = nullptr) {
  if (skinny_runs(false, M, N, K))
    return launch_skinny(false, A, B, C, pre, M, N, K, epi == kEpiGeluBwd ? kSkinnyGeluBwd : kSkinnyForward, epi, ct, s, ctr);
  // Row-major operands by gemm_any.h: rows that are not whole 16-byte units (one lane per output
  // before: 300x784x1000 with K = 300, 303 us against 7), outputs of fewer than 512 tiles of 64 x 64
  // (256 x 256 and 128-wide tiles leave CUs idle: 300x4096x4096 44.6 us against 36.3, 512^3 7.4 against
  // 6.4; 2048^3, 1024 tiles, 30.6 against 31.1), 1024 where K has no 64-byte stages (1500x1500x1000 23.4
  // against 19.1, 300x784x1000 20.8 against 11.6; 2000x4000x1000 31.7 against 33.0), and those where that
  // loop takes its 256-wide tiles (4000x4000x2000 126 against 102).
  if (any_runs(M, N, K) &&
      (K % 8 != 0 || tiles64(M, N) < (K % 32 == 0 ? 512 : 1024) || (K % 32 != 0 && choose_config(M, N, K) == 13)))
    return launch_any(false, true, A, B, C, pre, M, N, K, epi, ct, s, ctr);
  if (K % 8 != 0) {
    const int64_t blocks = (static_cast<int64_t>(M) * N + 255) / 256;
    hipLaunchKernelGGL(gemm_bf16_nt_simple, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, s, A, B, C, pre, M, N, K, epi, ct, ctr);
    return check_launch("gemm_bf16_nt_simple");
  }
  switch (choose_config(M, N, K)) {
    case 1: return launch_cfg<Bf1>(A, B, C, pre, M, N, K, epi, ct, s, ctr);
    case 2: return launch_cfg<Bf2>(A, B, C, pre, M, N, K, epi, ct, s, ctr);
    case 3: return launch_cfg<Bf3>(A, B, C, pre, M, N, K, epi, ct, s, ctr);
    case 4: return launch_cfg<Bf4>(A, B, C, pre, M, N, K, epi, ct, s, ctr);
    case 5: return launch_cfg<Bf5>(A, B, C, pre, M, N, K, epi, ct, s, ctr);
    case 6: return launch_cfg<Bf6>(A, B, C, pre, M, N, K, epi, ct, s, ctr);
    case 7: return launch_cfg<Bf7>(A, B, C, pre, M, N, K, epi, ct, s, ctr);
    case 8: return launch_cfg<Bf8>(A, B, C, pre, M, N, K, epi, ct, s, ctr);
    case 9: return launch_cfg<Bf9>(A, B, C, pre, M, N, K, epi, ct, s, ctr);
    case 10: return launch_cfg<Bf10>(A, B, C, pre, M, N, K, epi, ct, s, ctr);
    case 11: return launch_cfg<Bf11>(A, B, C, pre, M, N, K, epi, ct, s, ctr);
    case 12: return launch_cfg<Bf12>(A, B, C, pre, M, N, K, epi, ct, s, ctr);
    case 13: return launch_cfg<Bf13>(A, B, C, pre, M, N, K, epi, ct, s, ctr);
    case 14: return launch_dma<Dm14>(A, B, C, pre, M, N, K, epi, ct, s, ctr);
    case 15: return launch_dma<Dm15>(A, B, C, pre, M, N, K, epi, ct, s, ctr);
    case 16: return launch_dma<Dm16>(A, B, C, pre, M, N, K, epi, ct, s, ctr);
    case 17: return launch_dma<Dm17>(A, B, C, pre, M, N, K, epi, ct, s, ctr);
    case 18: return launch_dma<Dm18>(A, B, C, pre, M, N, K, epi, ct, s, ctr);
    case 19: return launch_dma<Dm19>(A, B, C, pre, M, N, K, epi, ct, s, ctr);
    case 20: return launch_dma<Dm20>(A, B, C, pre, M, N, K, epi, ct, s, ctr);
    case 21: return launch_dma<Dm21>(A, B, C, pre, M, N, K, epi, ct, s, ctr);
    case 22: return launch_dma<Dm22>(A, B, C, pre, M, N, K, epi, ct, s, ctr);
    case 23: return launch_dma<Dm23>(A, B, C, pre, M, N, K, epi, ct, s, ctr);
    case 24: return launch_dma<Dm24>(A, B, C, pre, M, N, K, epi, ct, s, ctr);
    case 25: return launch_dma<Dm25>(A, B, C, pre, M, N, K, epi, ct, s, ctr);
    case 26: return launch_dma<Dm26>(A, B, C, pre, M, N, K, epi, ct, s, ctr);
    default: return launch_cfg<Bf0>(A, B, C, pre, M, N, K, epi, ct, s, ctr);
  }
}

// Whether a GEMM's result leaves through streaming stores: a plain f32 output bound as an output.
bool stream_out(vdsl_buffer C, int epilogue, int c_dtype) {
  return epilogue == VDSL_EPI_NONE && c_dtype == VDSL_F32 && C->binding == VDSL_BIND_OUTPUT;
}

// kSizeOverflow when the re-layout copies' size does not fit size_t.
// Workspace of the transpose path: none when B is stored [K][N] and a configuration that reads the
// operands K-major runs the shape (vdsl_op_gemm_bf16 then transposes nothing).
size_t workspace_bytes(int ta, int tb, int64_t M, int64_t N, int64_t K) {
  if (!tb && K % 8 == 0 && M <= 0x7fffffff && N <= 0x7fffffff && dma_kn_runs(choose_config(M, N, K), M, N, ta)) return 0;
  const size_t a = ta ? nbytes(M, K, 2) : 0, b = tb ? 0 : nbytes(N, K, 2);
  if (a == kSizeOverflow || b == kSizeOverflow || a > kSizeOverflow - 1 - b) return kSizeOverflow;
  return a + b;
}

}  // namespace
}  // namespace vdsl

using namespace vdsl;

extern "C" int vdsl_gemm_bf16_workspace_bytes(int32_t trans_a, int32_t trans_b, int64_t M, int64_t N, int64_t K,
                                              size_t* bytes) {
  if (!bytes) return fail(VDSL_ERR_INVALID_ARG, "bytes is null");
  if (M < 0 || N < 0 || K < 0) return fail(VDSL_ERR_INVALID_ARG, "negative GEMM extent");
  const size_t ws = workspace_bytes(trans_a != 0, trans_b != 0, M, N, K);
  if (ws == kSizeOverflow) return fail(VDSL_ERR_SHAPE, "GEMM workspace size overflows (extents too large)");
  *bytes = ws;
  return VDSL_OK;
}

extern "C" int vdsl_op_gemm_bf16(vdsl_queue q, int32_t trans_a, int32_t trans_b, int64_t M, int64_t N, int64_t K,
                                 vdsl_buffer A, vdsl_buffer B, vdsl_buffer C, int32_t c_dtype, int32_t epilogue,
                                 vdsl_buffer pre_act, vdsl_buffer workspace) {
  VDSL_TRY(enter_queue(q));
  if (M < 0 || N < 0 || K < 0) return fail(VDSL_ERR_INVALID_ARG, "negative GEMM extent");
  if (M > 0x7fffffff || N > 0x7fffffff || K > 0x3fffffff) return fail(VDSL_ERR_UNSUPPORTED, "GEMM extent too large");
  if (c_dtype != VDSL_F32 && c_dtype != VDSL_BF16) return fail(VDSL_ERR_UNSUPPORTED, "C must be f32 or bf16");
  if (epilogue < VDSL_EPI_NONE || epilogue > VDSL_EPI_RELU) return fail(VDSL_ERR_INVALID_ARG, "unknown epilogue");
  const bool ta = trans_a != 0, tb = trans_b != 0;
  VDSL_TRY(check_buffer(q, A, nbytes(M, K, 2), "A", false));
  VDSL_TRY(check_buffer(q, B, nbytes(N, K, 2), "B", false));
  VDSL_TRY(check_buffer(q, C, nbytes(M, N, dtype_size(c_dtype)), "C", true));
  if (pre_act) VDSL_TRY(check_buffer(q, pre_act, nbytes(M, N, 4), "pre_act", true));
  // checked here, for the path this call takes (the K-major configurations need none)
  const size_t ws = workspace_bytes(ta, tb, M, N, K);
  if (ws == kSizeOverflow) return fail(VDSL_ERR_SHAPE, "GEMM workspace size overflows (extents too large)");
  if (ws) VDSL_TRY(check_buffer(q, workspace, ws, "workspace", true));
  if (M == 0 || N == 0) return VDSL_OK;

  const uint16_t* a = static_cast<const uint16_t*>(A->ptr);
  const uint16_t* b = static_cast<const uint16_t*>(B->ptr);
  float* pre = pre_act ? static_cast<float*>(pre_act->ptr) : nullptr;
  const int epi = epilogue | (stream_out(C, epilogue, c_dtype) ? kEpiStreamOut : 0);
  if (ws == 0 && !tb) {  // B stored [K][N] (and A [K][M] if ta): read K-major by a 256-wide configuration
    return launch_dma_kn(choose_config(M, N, K), a, b, C->ptr, pre, static_cast<int>(M), static_cast<int>(N),
                         static_cast<int>(K), epi, c_dtype, q->stream, ta);
  }
  // Transposed operands read as stored (gemm_any.h) instead of transposing them into the workspace
  // first (1000x784x300 TN 24.8 us against 7.2, 2048^3 40.2 against 31.1, 2000x4096x4096 94.2 against 92.7),
  // but for outputs large enough that the direct-to-LDS tiles repay the transposes (4032x4096x2048 TN
  // 87.0 against 97.6, 8000x8192x4096 522 against 657; 3056x4080x1024, 768 tiles, NN 51.6 against 55.1, TN
  // 53.9, 56.1) and, where B alone is transposed, those whose 128 x 128 tiles are a few more than the CUs (NN
  // 3952x1136x4096, 279 tiles, 69.7 against 77.7; 2032x2160x1024, 272, 27.8, 30.0; 2544x2032x1024, 320, 30.8, 30.5).
  const int64_t t128 = ((M + 127) / 128) * ((N + 127) / 128);
  const bool large = K % 32 == 0 && (t128 >= 768 || (!ta && t128 > 256 && t128 <= 304));
  if (any_runs(M, N, K) && (ta || !tb) && !large)
    return launch_any(ta, tb, a, b, C->ptr, pre, static_cast<int>(M), static_cast<int>(N), static_cast<int>(K), epi, c_dtype,
                      q->stream);
  char* w = ws ? static_cast<char*>(workspace->ptr) : nullptr;
  if (ta) {  // A stored [K][M] -> [M][K]
    VDSL_TRY(launch_transpose(a, w, K, M, VDSL_BF16, q->stream));
    a = reinterpret_cast<const uint16_t*>(w);
    w += static_cast<size_t>(M) * K * 2;
  }
  if (!tb) {  // B stored [K][N] -> [N][K]
    VDSL_TRY(launch_transpose(b, w, K, N, VDSL_BF16, q->stream));
    b = reinterpret_cast<const uint16_t*>(w);
  }
  return launch_nt(a, b, C->ptr, pre, static_cast<int>(M), static_cast<int>(N), static_cast<int>(K), epi, c_dtype,
                   q->stream);
}

extern "C" int vdsl_debug_gemm_config(int32_t config) {
  vdsl::gemm_config_override();  // consume the environment value first, so it cannot override this
  vdsl::g_gemm_config.store(config < 0 ? -1 : config, std::memory_order_relaxed);
  return VDSL_OK;
}

extern "C" int vdsl_op_gemm_bf16_gelu_bwd(vdsl_queue q, int64_t M, int64_t N, int64_t K, vdsl_buffer A, vdsl_buffer B,
                                          vdsl_buffer pre, vdsl_buffer da, vdsl_buffer da_t) {
  VDSL_TRY(enter_queue(q));
  if (M < 0 || N < 0 || K < 0) return fail(VDSL_ERR_INVALID_ARG, "negative GEMM extent");
  if (M > 0x7fffffff || N > 0x7fffffff || K > 0x3fffffff) return fail(VDSL_ERR_UNSUPPORTED, "GEMM extent too large");
  VDSL_TRY(check_buffer(q, A, nbytes(M, K, 2), "A", false));
  VDSL_TRY(check_buffer(q, B, nbytes(N, K, 2), "B", false));
  VDSL_TRY(check_buffer(q, pre, nbytes(M, N, 4), "pre", false));
  VDSL_TRY(check_buffer(q, da, nbytes(M, N, 2), "da", true));
  if (da_t) VDSL_TRY(check_buffer(q, da_t, nbytes(M, N, 2), "da_t", true));
  if (M == 0 || N == 0) return VDSL_OK;
  return launch_nt(static_cast<const uint16_t*>(A->ptr), static_cast<const uint16_t*>(B->ptr), da->ptr,
                   static_cast<float*>(pre->ptr), static_cast<int>(M), static_cast<int>(N), static_cast<int>(K), kEpiGeluBwd,
                   VDSL_BF16, q->stream, da_t ? static_cast<uint16_t*>(da_t->ptr) : nullptr);
}

extern "C" int vdsl_op_pack_bf16_weights(vdsl_queue q, int64_t N, int64_t K, vdsl_buffer w, vdsl_buffer wp) {
  VDSL_TRY(enter_queue(q));
  if (N < 0 || K < 0) return fail(VDSL_ERR_INVALID_ARG, "negative weight extent");
  if (N % 32 || K % 16) return fail(VDSL_ERR_UNSUPPORTED, "packed bf16 weights need N % 32 == 0 and K % 16 == 0");
  const size_t n = nbytes(N, K, 2);
  VDSL_TRY(check_buffer(q, w, n, "w", false));
  VDSL_TRY(check_buffer(q, wp, n, "wp", true));
  if (w == wp) return fail(VDSL_ERR_INVALID_ARG, "w and wp must be different buffers");
  if (n == 0) return VDSL_OK;
  int64_t blocks = (static_cast<int64_t>(n / 16) + 255) / 256;
  if (blocks > 16384) blocks = 16384;
  hipLaunchKernelGGL(bpk_pack_kernel, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, q->stream,
                     static_cast<const char*>(w->ptr), static_cast<char*>(wp->ptr), N / 32, 2 * K / 32, 2 * K);
  return check_launch("bpk_pack_kernel");
}

extern "C" int vdsl_op_gemm_bf16_packed(vdsl_queue q, int64_t M, int64_t N, int64_t K, vdsl_buffer A, vdsl_buffer Bp,
                                        vdsl_buffer C, int32_t c_dtype, int32_t epilogue, vdsl_buffer pre_act) {
  VDSL_TRY(enter_queue(q));
  if (M < 0 || N < 0 || K < 0) return fail(VDSL_ERR_INVALID_ARG, "negative GEMM extent");
  if (M > 0x7fffffff || N > 0x7fffffff || K > 0x3fffffff) return fail(VDSL_ERR_UNSUPPORTED, "GEMM extent too large");
  if (N % 32) return fail(VDSL_ERR_UNSUPPORTED, "packed GEMM needs N % 32 == 0");
  if ((2 * K) % (128 * Pb0::NR) || K == 0) return fail(VDSL_ERR_UNSUPPORTED, "packed bf16 GEMM needs K % 256 == 0 and K > 0");
  if (c_dtype != VDSL_F32 && c_dtype != VDSL_BF16) return fail(VDSL_ERR_UNSUPPORTED, "C must be f32 or bf16");
  if (epilogue < VDSL_EPI_NONE || epilogue > VDSL_EPI_GELU_DERIV) return fail(VDSL_ERR_INVALID_ARG, "unknown epilogue");
  if (epilogue == VDSL_EPI_GELU_DERIV && (!pre_act || c_dtype != VDSL_BF16))
    return fail(VDSL_ERR_INVALID_ARG, "VDSL_EPI_GELU_DERIV needs pre_act and a bf16 C");
  VDSL_TRY(check_buffer(q, A, nbytes(M, K, 2), "A", false));
  VDSL_TRY(check_buffer(q, Bp, nbytes(N, K, 2), "Bp", false));
  VDSL_TRY(check_buffer(q, C, nbytes(M, N, dtype_size(c_dtype)), "C", true));
  if (pre_act) VDSL_TRY(check_buffer(q, pre_act, nbytes(M, N, 4), "pre_act", true));
  if (M == 0 || N == 0) return VDSL_OK;
  if (skinny_runs(true, M, N, K))
    return launch_skinny(true, static_cast<const uint16_t*>(A->ptr), static_cast<const uint16_t*>(Bp->ptr), C->ptr,
                         pre_act ? static_cast<float*>(pre_act->ptr) : nullptr, static_cast<int>(M), static_cast<int>(N),
                         static_cast<int>(K), epilogue == VDSL_EPI_GELU_DERIV ? kSkinnyDeriv : kSkinnyForward, epilogue, c_dtype,
                         q->stream, nullptr);
  return bpk_dispatch(M, N, [&](auto cfg, int64_t tiles) {
    using Cfg = decltype(cfg);
    auto* kern = epilogue == VDSL_EPI_GELU_DERIV ? gemm_bf16_bpk<Cfg, 0, true> : gemm_bf16_bpk<Cfg, 0, false>;
    hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>(tiles)), dim3(Cfg::NT), 0, q->stream,
                       static_cast<const uint16_t*>(A->ptr), static_cast<const uint16_t*>(Bp->ptr), C->ptr,
                       pre_act ? static_cast<float*>(pre_act->ptr) : nullptr, static_cast<int>(M), static_cast<int>(N),
                       static_cast<int>(K), epilogue | (stream_out(C, epilogue, c_dtype) ? kEpiStreamOut : 0), c_dtype, nullptr);
    return check_launch("gemm_bf16_bpk");
  });
}

extern "C" int vdsl_op_gemm_bf16_gelu_bwd_packed(vdsl_queue q, int64_t M, int64_t N, int64_t K, vdsl_buffer A,
                                                 vdsl_buffer Bp, vdsl_buffer pre, vdsl_buffer da, vdsl_buffer da_t) {
  VDSL_TRY(enter_queue(q));
  if (M < 0 || N < 0 || K < 0) return fail(VDSL_ERR_INVALID_ARG, "negative GEMM extent");
  if (M > 0x7fffffff || N > 0x7fffffff || K > 0x3fffffff) return fail(VDSL_ERR_UNSUPPORTED, "GEMM extent too large");
  if (N % 32) return fail(VDSL_ERR_UNSUPPORTED, "packed GEMM needs N % 32 == 0");
  if ((2 * K) % (128 * Pb0::NR) || K == 0) return fail(VDSL_ERR_UNSUPPORTED, "packed bf16 GEMM needs K % 256 == 0 and K > 0");
  VDSL_TRY(check_buffer(q, A, nbytes(M, K, 2), "A", false));
  VDSL_TRY(check_buffer(q, Bp, nbytes(N, K, 2), "Bp", false));
  VDSL_TRY(check_buffer(q, pre, nbytes(M, N, 4), "pre", false));
  VDSL_TRY(check_buffer(q, da, nbytes(M, N, 2), "da", true));
  if (da_t) VDSL_TRY(check_buffer(q, da_t, nbytes(M, N, 2), "da_t", true));
  if (M == 0 || N == 0) return VDSL_OK;
  if (skinny_runs(true, M, N, K))
    return launch_skinny(true, static_cast<const uint16_t*>(A->ptr), static_cast<const uint16_t*>(Bp->ptr), da->ptr,
                         static_cast<float*>(pre->ptr), static_cast<int>(M), static_cast<int>(N), static_cast<int>(K), kSkinnyGeluBwd,
                         kEpiGeluBwd, VDSL_BF16, q->stream, da_t ? static_cast<uint16_t*>(da_t->ptr) : nullptr);
  return bpk_dispatch(M, N, [&](auto cfg, int64_t tiles) {
    using Cfg = decltype(cfg);
    hipLaunchKernelGGL((gemm_bf16_bpk<Cfg, 1>), dim3(static_cast<unsigned>(tiles)), dim3(Cfg::NT), 0, q->stream,
                       static_cast<const uint16_t*>(A->ptr), static_cast<const uint16_t*>(Bp->ptr), da->ptr,
                       static_cast<float*>(pre->ptr), static_cast<int>(M), static_cast<int>(N), static_cast<int>(K),
                       kEpiGeluBwd, VDSL_BF16, da_t ? static_cast<uint16_t*>(da_t->ptr) : nullptr);
    return check_launch("gemm_bf16_bpk<gelu_bwd>");
  });
}

extern "C" int vdsl_op_gemm_bf16_mul_packed(vdsl_queue q, int64_t M, int64_t N, int64_t K, vdsl_buffer A, vdsl_buffer Bp,
                                            vdsl_buffer g, vdsl_buffer c, vdsl_buffer c_t) {
  VDSL_TRY(enter_queue(q));
  if (M < 0 || N < 0 || K < 0) return fail(VDSL_ERR_INVALID_ARG, "negative GEMM extent");
  if (M > 0x7fffffff || N > 0x7fffffff || K > 0x3fffffff) return fail(VDSL_ERR_UNSUPPORTED, "GEMM extent too large");
  if (N % 32) return fail(VDSL_ERR_UNSUPPORTED, "packed GEMM needs N % 32 == 0");
  if ((2 * K) % (128 * Pb0::NR) || K == 0) return fail(VDSL_ERR_UNSUPPORTED, "packed bf16 GEMM needs K % 256 == 0 and K > 0");
  VDSL_TRY(check_buffer(q, A, nbytes(M, K, 2), "A", false));
  VDSL_TRY(check_buffer(q, Bp, nbytes(N, K, 2), "Bp", false));
  VDSL_TRY(check_buffer(q, g, nbytes(M, N, 4), "g", false));
  VDSL_TRY(check_buffer(q, c, nbytes(M, N, 2), "c", true));
  if (c_t) VDSL_TRY(check_buffer(q, c_t, nbytes(M, N, 2), "c_t", true));
  if (M == 0 || N == 0) return VDSL_OK;
  if (skinny_runs(true, M, N, K))
    return launch_skinny(true, static_cast<const uint16_t*>(A->ptr), static_cast<const uint16_t*>(Bp->ptr), c->ptr,
                         static_cast<float*>(g->ptr), static_cast<int>(M), static_cast<int>(N), static_cast<int>(K), kSkinnyMul,
                         kEpiGeluBwd, VDSL_BF16, q->stream, c_t ? static_cast<uint16_t*>(c_t->ptr) : nullptr);
  return bpk_dispatch(M, N, [&](auto cfg, int64_t tiles) {
    using Cfg = decltype(cfg);
    hipLaunchKernelGGL((gemm_bf16_bpk<Cfg, 2>), dim3(static_cast<unsigned>(tiles)), dim3(Cfg::NT), 0, q->stream,
                       static_cast<const uint16_t*>(A->ptr), static_cast<const uint16_t*>(Bp->ptr), c->ptr,
                       static_cast<float*>(g->ptr), static_cast<int>(M), static_cast<int>(N), static_cast<int>(K),
                       kEpiGeluBwd, VDSL_BF16, c_t ? static_cast<uint16_t*>(c_t->ptr) : nullptr);
    return check_launch("gemm_bf16_bpk<mul>");
  });
}

extern "C" int vdsl_op_gemm_bf16_mse_packed(vdsl_queue q, int64_t M, int64_t N, int64_t K, vdsl_buffer A, vdsl_buffer Bp,
                                            vdsl_buffer t, vdsl_buffer y, vdsl_buffer loss, vdsl_buffer dy, vdsl_buffer dy_t,
                                            vdsl_buffer partials) {
  VDSL_TRY(enter_queue(q));
  if (M <= 0 || N <= 0 || K <= 0) return fail(VDSL_ERR_INVALID_ARG, "GEMM + MSE needs positive extents");
  if (M > 0x7fffffff || N > 0x7fffffff || K > 0x3fffffff) return fail(VDSL_ERR_UNSUPPORTED, "GEMM extent too large");
  if (M % Pb0::BM || N % Pb0::BN) return fail(VDSL_ERR_UNSUPPORTED, "GEMM + MSE needs M % 128 == 0 and N % 256 == 0");
  if ((2 * K) % (128 * Pb0::NR)) return fail(VDSL_ERR_UNSUPPORTED, "packed bf16 GEMM needs K % 256 == 0");
  VDSL_TRY(check_buffer(q, A, nbytes(M, K, 2), "A", false));
  VDSL_TRY(check_buffer(q, Bp, nbytes(N, K, 2), "Bp", false));
  VDSL_TRY(check_buffer(q, t, nbytes(M, N, 4), "t", false));
  if (y) VDSL_TRY(check_buffer(q, y, nbytes(M, N, 4), "y", true));
  VDSL_TRY(check_buffer(q, loss, 4, "loss", true));
  VDSL_TRY(check_buffer(q, dy, nbytes(M, N, 2), "dy", true));
  if (dy_t) VDSL_TRY(check_buffer(q, dy_t, nbytes(M, N, 2), "dy_t", true));
  const int64_t tiles = (M / Pb0::BM) * (N / Pb0::BN), n_part = tiles * Pb0::W;
  VDSL_TRY(check_buffer(q, partials, nbytes(vdsl_mse_partials_count(M, N), 4), "partials", true));
  if (static_cast<int64_t>(n_part * 2) > vdsl_mse_partials_count(M, N))
    return fail(VDSL_ERR_UNSUPPORTED, "GEMM + MSE: partial sums exceed the MSE scratch size");
  const size_t n = static_cast<size_t>(M) * static_cast<size_t>(N);
  const float scale = 2.0f / static_cast<float>(n);  // as vdsl_op_mse_fwd_bwd
  double* part = static_cast<double*>(partials->ptr);
  hipLaunchKernelGGL((gemm_bf16_bpk_mse<Pb0>), dim3(static_cast<unsigned>(tiles)), dim3(Pb0::NT), 0, q->stream,
                     static_cast<const uint16_t*>(A->ptr), static_cast<const uint16_t*>(Bp->ptr),
                     static_cast<const float*>(t->ptr), y ? static_cast<float*>(y->ptr) : nullptr,
                     static_cast<uint16_t*>(dy->ptr), dy_t ? static_cast<uint16_t*>(dy_t->ptr) : nullptr, part,
                     static_cast<int>(M), static_cast<int>(N), static_cast<int>(K), scale);
  VDSL_TRY(check_launch("gemm_bf16_bpk_mse"));
  return launch_mse_finish(part, n_part, static_cast<float*>(loss->ptr), 1.0 / static_cast<double>(n), q->stream);
}
