// GEMMs with one short side on gfx950 (bf16 and int8): C[m][n] = sum_k A[m][k] B[n][k] where fewer
// than 128 rows (or columns) leave the tile kernels a handful of blocks: bound by reading the long
// operand once, so by bytes in flight on every CU, not by MFMA.
//
// A block owns 16 MT x 16 NT outputs over all of K: its NW waves split K, each loads its fragments
// of v_mfma_f32_16x16x32_bf16 / v_mfma_i32_16x16x64_i8 straight into registers (lane l: row or
// column l % 16, bytes 16 (l / 16) .. + 15 of a 64-byte K step, U steps' loads issued before the
// first MFMA), and the waves' accumulators meet in LDS, added in wave order.  So one launch without
// scratch memory, deterministic, and N / 16 blocks of 8 or 16 waves: an [8][4096] x [4096][4096]
// product has 128 KiB of weights in flight on each of 256 CUs and takes 8.2 us (4.1 TB/s of weights;
// 43 us in 16 tiles of 128 x 256).  Nothing goes through LDS in the loop: no two waves share a
// fragment.  Measured without effect: waves on contiguous K ranges instead of every NW-th pair.
//
// Operand forms: row-major with any row length (rows of an odd number of elements start anywhere; the
// 16-byte loads need no more than the element's alignment), or, for B, packed in fragment order
// (gemm_bpk.h).  K is split by whole steps the same way for every form, so packed and row-major
// weights give the same bits.
#pragma once

#include "gemm_mfma.h"

namespace vdsl {

typedef float f32x4_acc __attribute__((ext_vector_type(4)));

struct Mfma16Bf16 {
  using Frag = bf16x8;
  using Acc = f32x4_acc;
  static constexpr int kElemBytes = 2;
  __device__ static __forceinline__ Acc mma(const Frag& a, const Frag& b, const Acc& c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
};
struct Mfma16I8 {
  using Frag = i32x4;
  using Acc = i32x4;
  static constexpr int kElemBytes = 1;
  __device__ static __forceinline__ Acc mma(const Frag& a, const Frag& b, const Acc& c) {
    return __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, c, 0, 0, 0);
  }
};

// 16 bytes from an address aligned to the element only.
struct __attribute__((packed, aligned(2))) Bytes16 {
  u32x4 v;
};

__device__ __forceinline__ u32x4 load16(const char* p) { return reinterpret_cast<const Bytes16*>(p)->v; }

// v shifted down by w (0..16) bytes, zeros entering at the top.
__device__ __forceinline__ u32x4 shift_down(u32x4 v, int w) {
  const int sh = 8 * (w & 3);
  uint32_t t[5] = {v[0], v[1], v[2], v[3], 0u};
#pragma unroll
  for (int s = 1; s <= 4; ++s) {
    if (s <= (w >> 2)) {
#pragma unroll
      for (int e = 0; e < 4; ++e) t[e] = t[e + 1];
    }
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = static_cast<uint32_t>((static_cast<uint64_t>(t[e + 1]) << 32 | t[e]) >> sh);
  return v;
}

// The 16 bytes at byte offset `at` of a tensor of `size` >= 16 bytes, those past its end as 0 and
// never read: lanes near the end load the tensor's last 16 bytes and shift them down.
__device__ __forceinline__ u32x4 load16_to_end(const char* __restrict__ base, int64_t at, int64_t size) {
  const int64_t last = size - 16, from = at < last ? at : last;
  return shift_down(load16(base + from), at - from > 16 ? 16 : static_cast<int>(at - from));
}

// Bytes of v from `keep` on set to 0 (keep may be negative or past 16).
__device__ __forceinline__ u32x4 first_bytes(u32x4 v, int keep) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int k = keep - 4 * e;
    v[e] = k <= 0 ? 0u : k >= 4 ? v[e] : v[e] & ((1u << (8 * k)) - 1u);
  }
  return v;
}

// How B is stored: packed in fragment order (K a whole number of 64-byte steps), or in rows like A.
enum SkinnyForm { kSkinnyPacked, kSkinnyRows };

template <class T, SkinnyForm FORM, int MT_, int NT_, int NW_>
struct SkinnyConfig {
  using Mma = T;
  static constexpr bool kPacked = FORM == kSkinnyPacked;
  static constexpr int MT = MT_, NT = NT_, NW = NW_;
  static constexpr int BM = 16 * MT, BN = 16 * NT, THREADS = 64 * NW;
  static constexpr int U = MT * NT == 1 ? 8 : 4;  // K steps loaded together
  static constexpr int LDS_BYTES = NW * MT * NT * 1024;
  static_assert(LDS_BYTES <= 160 * 1024, "gfx950 workgroup LDS limit");
};

// Runs the block's product at (m0, n0) and calls out(row, col, value) for each of its elements
// inside M x N once, on some thread.  Kb: bytes of K per row; a row-major operand has rows of Kb
// bytes and at least 16 bytes in all.
template <class Cfg, class Out>
__device__ __forceinline__ void skinny_gemm(const char* __restrict__ A, const char* __restrict__ B, int M, int N, int Kb, int m0,
                                            int n0, char* smem, Out&& out) {
  using T = typename Cfg::Mma;
  using Frag = typename T::Frag;
  using Acc = typename T::Acc;
  constexpr int MT = Cfg::MT, NT = Cfg::NT, U = Cfg::U;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r16 = lane & 15, g = lane >> 4;
  // Wave w takes every NW-th pair of steps from pair w on (both halves of a row's 128-byte lines).
  const int steps = (Kb + 63) / 64, pairs = (steps + 1) / 2;
  // The last step, when K ends inside it, is left for after the loop: all others lie inside their rows.
  const int whole = Cfg::kPacked ? steps : Kb / 64;
  const bool partial = whole < steps && (pairs - 1) % Cfg::NW == wave;

  int64_t arow[MT], brow[NT];
#pragma unroll
  for (int i = 0; i < MT; ++i) arow[i] = static_cast<int64_t>(m0 + 16 * i + r16 < M ? m0 + 16 * i + r16 : M - 1) * Kb + 16 * g;
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    if constexpr (Cfg::kPacked) {
      // unit (nb, kb): 32 columns x 32 bytes, column c's half h at 16 (c + 32 h); N % 32 == 0
      const int c = n0 + 16 * j + r16;
      brow[j] = (static_cast<int64_t>((n0 + 16 * j) >> 5) * (Kb / 32) + (g >> 1)) * 1024 + ((c & 31) + 32 * (g & 1)) * 16;
    } else {
      brow[j] = static_cast<int64_t>(n0 + 16 * j + r16 < N ? n0 + 16 * j + r16 : N - 1) * Kb + 16 * g;
    }
  }

  Acc acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = Acc{0, 0, 0, 0};

  for (int p0 = wave; p0 < pairs; p0 += U / 2 * Cfg::NW) {
    u32x4 a[U][MT], b[U][NT];
#pragma unroll
    for (int u = 0; u < U; u += 2) {
      // past the end: any step that is there
      const int st = 2 * (p0 + u / 2 * Cfg::NW), x0 = st < whole ? st : 0, x1 = st + 1 < whole ? st + 1 : 0;
      if (whole == 0) continue;  // K inside the first step
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        if constexpr (Cfg::kPacked) {
          b[u][j] = *reinterpret_cast<const u32x4*>(B + brow[j] + static_cast<int64_t>(x0) * 2048);
          b[u + 1][j] = *reinterpret_cast<const u32x4*>(B + brow[j] + static_cast<int64_t>(x1) * 2048);
        } else {
          b[u][j] = load16(B + brow[j] + static_cast<int64_t>(x0) * 64);
          b[u + 1][j] = load16(B + brow[j] + static_cast<int64_t>(x1) * 64);
        }
      }
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        a[u][i] = load16(A + arow[i] + static_cast<int64_t>(x0) * 64);
        a[u + 1][i] = load16(A + arow[i] + static_cast<int64_t>(x1) * 64);
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (2 * (p0 + u / 2 * Cfg::NW) + u % 2 < whole) {  // wave-uniform
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
          for (int j = 0; j < NT; ++j)
            acc[i][j] = T::mma(__builtin_bit_cast(Frag, a[u][i]), __builtin_bit_cast(Frag, b[u][j]), acc[i][j]);
      }
    }
  }

  if (partial) {  // wave-uniform; both sides' bytes past K are made 0, whatever lies there
    const int64_t at = static_cast<int64_t>(whole) * 64;
    const int keep = Kb - 64 * whole - 16 * g;
    u32x4 b[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) b[j] = first_bytes(load16_to_end(B, brow[j] + at, static_cast<int64_t>(N) * Kb), keep);
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const u32x4 a = first_bytes(load16_to_end(A, arow[i] + at, static_cast<int64_t>(M) * Kb), keep);
#pragma unroll
      for (int j = 0; j < NT; ++j) acc[i][j] = T::mma(__builtin_bit_cast(Frag, a), __builtin_bit_cast(Frag, b[j]), acc[i][j]);
    }
  }

  // Element r of lane l: row 4 (l / 16) + r, column l % 16 of its 16 x 16 tile.
  Acc* const area = reinterpret_cast<Acc*>(smem);
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) area[(wave * MT * NT + i * NT + j) * 64 + lane] = acc[i][j];
  __syncthreads();
  for (int u = threadIdx.x; u < MT * NT * 64; u += Cfg::THREADS) {
    Acc v = area[u];
#pragma unroll
    for (int w = 1; w < Cfg::NW; ++w) v += area[w * MT * NT * 64 + u];
    const int l = u & 63, t = u >> 6;
    const int col = n0 + 16 * (t % NT) + (l & 15), row = m0 + 16 * (t / NT) + 4 * (l >> 4);
    if (col < N) {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (row + r < M) out(row + r, col, v[r]);
    }
  }
}

// Waves per block, by the short side and K alone, so that every form of one product splits K alike.
inline int skinny_waves(int64_t M, int64_t N, int64_t Kb) { return (M < N ? M : N) <= 32 && Kb >= 4096 ? 16 : 8; }

// Calls go(Cfg{}) with the configuration of an M x N x Kb product whose A side is the one tiled by
// MT: up to 64 rows (32 with 16 waves) per block; two column tiles per block once 32-wide strips
// alone cover the CUs.
template <class T, SkinnyForm FORM, class Go>
int skinny_dispatch(int64_t M, int64_t N, int64_t Kb, Go&& go) {
  const bool wide = (N + 31) / 32 * ((M + 63) / 64) >= 256;
  if (skinny_waves(M, N, Kb) == 16) {
    if (M <= 16) return wide ? go(SkinnyConfig<T, FORM, 1, 2, 16>{}) : go(SkinnyConfig<T, FORM, 1, 1, 16>{});
    return wide ? go(SkinnyConfig<T, FORM, 2, 2, 16>{}) : go(SkinnyConfig<T, FORM, 2, 1, 16>{});
  }
  if (M <= 16) return wide ? go(SkinnyConfig<T, FORM, 1, 2, 8>{}) : go(SkinnyConfig<T, FORM, 1, 1, 8>{});
  if (M <= 32) return wide ? go(SkinnyConfig<T, FORM, 2, 2, 8>{}) : go(SkinnyConfig<T, FORM, 2, 1, 8>{});
  return wide ? go(SkinnyConfig<T, FORM, 4, 2, 8>{}) : go(SkinnyConfig<T, FORM, 4, 1, 8>{});
}

}  // namespace vdsl
