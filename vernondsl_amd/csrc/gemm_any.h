// Register-staged bf16 MFMA main loop for gfx950 that takes its operands as they are stored:
// C[m][n] = sum_k A(m, k) B(n, k), each operand row-major ([rows][K], K contiguous) or K-major
// ([K][rows]), with any extents.  It replaces transposes into a workspace, and one lane per output
// where K % 8 != 0, for products that no direct-to-LDS configuration takes.
//
// Loads are 16 bytes per lane at the element's alignment (rows of an odd length start anywhere) and
// unconditional: rows past the operand repeat its last one (their products reach no stored output),
// chunks of a K-major row past its end read on into the next row, and a lane whose 16 bytes would
// pass the tensor's end loads its last 16 bytes.  Only stages within 8 rows of K's end look back at
// that when they go to LDS: they shift such lanes' bytes into place and zero what lies past K.
//
// LDS, per stage of 64 K values: a row-major operand as [rows][128 + 16] bytes, fragments by 16-byte
// reads; a K-major one as [64][2 rows + 64] bytes (the 4 K rows of a transposing read then start 64
// bytes apart modulo the 256 bytes of all banks), a fragment being two ds_read_b64_tr_b16 (the lane
// layout is described in gemm_dma.h).  Two stages; two register sets keep the loads of two more in
// flight.  The same k-steps in the same order as every other main loop, so the same bits.
#pragma once

#include "gemm_dma.h"
#include "gemm_skinny.h"

namespace vdsl {

template <int BM_, int BN_, int WGM_, int WGN_, bool AKM_, bool BKM_>
struct AnyConfig {
  static constexpr int BM = BM_, BN = BN_, WGM = WGM_, WGN = WGN_;
  static constexpr bool AKM = AKM_, BKM = BKM_;
  static constexpr int BK = 64;                      // K values per stage
  static constexpr int NT = 64 * WGM * WGN;
  static constexpr int WTM = BM / WGM, WTN = BN / WGN;
  static constexpr int FM = WTM / 32, FN = WTN / 32;
  static constexpr int CA = BM * BK / 8 / NT, CB = BN * BK / 8 / NT;  // 16-byte chunks per lane and stage
  static constexpr int ROW = 2 * BK + 16;            // LDS row of a row-major operand
  static constexpr int A_ROW = AKM ? 2 * BM + 64 : ROW, B_ROW = BKM ? 2 * BN + 64 : ROW;
  static constexpr int A_BYTES = (AKM ? BK : BM) * A_ROW, B_BYTES = (BKM ? BK : BN) * B_ROW;
  static constexpr int STAGE = A_BYTES + B_BYTES;
  static constexpr int LDS_BYTES = 2 * STAGE;
  static_assert(CA * NT * 8 == BM * BK && CB * NT * 8 == BN * BK, "chunks must split evenly over lanes");
};

// One operand's share of a lane: chunk i of C at LDS byte lds[i] of the stage, read from element
// `at` + kstep * stage * 64 of the tensor.
template <bool KM, int ROWS, int NT, int C, int LDS_ROW>
struct AnyOperand {
  static constexpr int CPR = KM ? ROWS / 8 : 8;  // chunks per LDS row
  const char* base;
  int64_t size, last;  // elements; the start of the last 16 bytes
  int64_t at[C];       // of stage 0
  int64_t kstep;       // elements per K value
  int k_of[C];         // the chunk's first K value within a stage
  int lds[C];

  __device__ __forceinline__ AnyOperand(const uint16_t* p, int rows, int K, int r0) {
    base = reinterpret_cast<const char*>(p);
    size = static_cast<int64_t>(rows) * K;
    last = size - 8;
    kstep = KM ? rows : 1;
#pragma unroll
    for (int i = 0; i < C; ++i) {
      const int c = static_cast<int>(threadIdx.x) + NT * i, row = c / CPR, chunk = c % CPR;
      lds[i] = row * LDS_ROW + chunk * 16;
      if constexpr (KM) {
        k_of[i] = row;
        at[i] = static_cast<int64_t>(row) * rows + (r0 + 8 * chunk < rows ? r0 + 8 * chunk : 0);
      } else {
        k_of[i] = 8 * chunk;
        at[i] = static_cast<int64_t>(r0 + row < rows ? r0 + row : rows - 1) * K + 8 * chunk;
      }
    }
  }
  __device__ __forceinline__ void load(u32x4 (&r)[C], int k0) const {
#pragma unroll
    for (int i = 0; i < C; ++i) {
      const int64_t e = at[i] + k0 * kstep;
      r[i] = load16(base + 2 * (e < last ? e : last));
    }
  }
  __device__ __forceinline__ void store(const u32x4 (&r)[C], int k0, int K, char* stage) const {
    if (k0 + 64 + 8 > K) {  // block-uniform: lanes of this stage may have met the tensor's or K's end
#pragma unroll
      for (int i = 0; i < C; ++i) {
        const int64_t over = at[i] + k0 * kstep - last;
        u32x4 v = over > 0 ? shift_down(r[i], over > 8 ? 16 : static_cast<int>(2 * over)) : r[i];
        const int left = K - k0 - k_of[i];  // K values from the chunk's first on
        v = KM ? first_bytes(v, left > 0 ? 16 : 0) : first_bytes(v, 2 * left);
        *reinterpret_cast<u32x4*>(stage + lds[i]) = v;
      }
    } else {
#pragma unroll
      for (int i = 0; i < C; ++i) *reinterpret_cast<u32x4*>(stage + lds[i]) = r[i];
    }
  }
};

// Fragment f (of FR) of k-step kk for this lane: rows row0 + 32 f + l % 32, K values 8 (l / 32) .. + 7.
template <bool KM, int LDS_ROW>
__device__ __forceinline__ bf16x8 any_fragment(const char* area, int row0, int f, int kk) {
  const int lane = threadIdx.x & 63;
  if constexpr (KM) {
    const int g = lane >> 4, i = lane & 15;
    const int k = 16 * kk + 8 * (g >> 1) + (i >> 2), col = row0 + 32 * f + 16 * (g & 1) + 4 * (i & 3);
    const char* p = area + k * LDS_ROW + 2 * col;
    const i16x4_t lo = lds_read_tr16(p), hi = lds_read_tr16(p + 4 * LDS_ROW);
    typedef short i16x8_t __attribute__((ext_vector_type(8)));
    const i16x8_t v = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    return __builtin_bit_cast(bf16x8, v);
  } else {
    return *reinterpret_cast<const bf16x8*>(area + (row0 + 32 * f + (lane & 31)) * LDS_ROW + 32 * kk + 16 * (lane >> 5));
  }
}

template <class Cfg>
__device__ __forceinline__ void any_mainloop(const uint16_t* __restrict__ A, const uint16_t* __restrict__ B, int M, int N, int K,
                                             int m0, int n0, char* smem, f32x16 (&acc)[Cfg::FM][Cfg::FN]) {
  constexpr int FM = Cfg::FM, FN = Cfg::FN;
  const int wave = threadIdx.x >> 6;
  const int wr = (wave / Cfg::WGN) * Cfg::WTM, wc = (wave % Cfg::WGN) * Cfg::WTN;
  const AnyOperand<Cfg::AKM, Cfg::BM, Cfg::NT, Cfg::CA, Cfg::A_ROW> a(A, M, K, m0);
  const AnyOperand<Cfg::BKM, Cfg::BN, Cfg::NT, Cfg::CB, Cfg::B_ROW> b(B, N, K, n0);
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = MfmaBf16::zero();
  u32x4 ra0[Cfg::CA], rb0[Cfg::CB], ra1[Cfg::CA], rb1[Cfg::CB];
  const int nk = (K + Cfg::BK - 1) / Cfg::BK, k_last = (nk - 1) * Cfg::BK;

  const auto compute = [&](const char* stage) {
#pragma unroll
    for (int kk = 0; kk < Cfg::BK / 16; ++kk) {
      bf16x8 fa[FM], fb[FN];
#pragma unroll
      for (int i = 0; i < FM; ++i) fa[i] = any_fragment<Cfg::AKM, Cfg::A_ROW>(stage, wr, i, kk);
#pragma unroll
      for (int j = 0; j < FN; ++j) fb[j] = any_fragment<Cfg::BKM, Cfg::B_ROW>(stage + Cfg::A_BYTES, wc, j, kk);
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = MfmaBf16::mma(fa[i], fb[j], acc[i][j]);
    }
  };
// Stage KT computed from LDS stage CUR while set L receives stage KT + 2 and set S (stage KT + 1) goes
// to the other LDS stage.  Past the last stage loads and stores repeat it, unused.
#define VDSL_ANY_STEP(KT, CUR, RA_L, RB_L, RA_S, RB_S)                                        \
  do {                                                                                        \
    const int kl_ = min(((KT) + 2) * Cfg::BK, k_last), ks_ = min(((KT) + 1) * Cfg::BK, k_last); \
    a.load(RA_L, kl_);                                                                        \
    b.load(RB_L, kl_);                                                                        \
    __builtin_amdgcn_sched_barrier(0);                                                        \
    compute(smem + (CUR) * Cfg::STAGE);                                                       \
    a.store(RA_S, ks_, K, smem + ((CUR) ^ 1) * Cfg::STAGE);                                   \
    b.store(RB_S, ks_, K, smem + ((CUR) ^ 1) * Cfg::STAGE + Cfg::A_BYTES);                    \
    __syncthreads();                                                                          \
    __builtin_amdgcn_sched_barrier(0);                                                        \
  } while (0)
  a.load(ra0, 0);
  b.load(rb0, 0);
  a.load(ra1, min(Cfg::BK, k_last));
  b.load(rb1, min(Cfg::BK, k_last));
  a.store(ra0, 0, K, smem);
  b.store(rb0, 0, K, smem + Cfg::A_BYTES);
  __syncthreads();
  int kt = 0;
  for (; kt + 2 <= nk; kt += 2) {
    VDSL_ANY_STEP(kt, 0, ra0, rb0, ra1, rb1);
    VDSL_ANY_STEP(kt + 1, 1, ra1, rb1, ra0, rb0);
  }
  if (kt < nk) VDSL_ANY_STEP(kt, 0, ra0, rb0, ra1, rb1);
#undef VDSL_ANY_STEP
}

}  // namespace vdsl
