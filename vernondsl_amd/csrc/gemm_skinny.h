// GEMMs with one short side on gfx950: C[m][n] = sum_k A[m][k] B[n][k] where fewer than 128 rows (or
// columns) leave the tile kernels a handful of blocks: bound by reading the long operand once, so by
// bytes in flight on every CU, not by MFMA.  A block owns 16 MT x 16 NT outputs over all of K, so N / 16
// blocks, one launch, no scratch memory, deterministic.  Fragments are those of v_mfma_f32_16x16x32_bf16
// / v_mfma_i32_16x16x64_i8 (lane l: row or column l % 16, bytes 16 (l / 16) .. + 15 of a 64-byte K step).
//
// int8 (skinny_gemm): the block's NW waves split K, each loads its fragments straight into registers
// (U steps' loads issued before the first MFMA), and the waves' accumulators meet in LDS: integer sums
// are the same in any order.  Nothing goes through LDS in the loop: no two waves share a fragment.
// Measured without effect: waves on contiguous K ranges instead of every NW-th pair.
//
// bf16 (skinny_chain): every output is one chain of MFMAs over K, the k-steps in the order of every other
// main loop (a 16x16x32 MFMA rounds as the two 32x32x16 ones of its halves), so a product gives the same
// bits whatever its layout, its batch and the kernel that its sizes select.  Eight waves load fragments
// and pass them through LDS in stages of S steps; one wave per 16 x 16 tile runs its chain on the stage
// before, while the next stage's loads are in flight.  [8][4096] x [4096][4096] packed, operands rotating:
// 11.0 us (48.5 in 128 x 256 tiles, 9.9 with K split over the waves, which adds in another order); [20]
// 14.6 (50.6, 13.3); [8][4096] x [16384] 26.4 (51, 27.5); [64][4000] x [4000], row-major 22.4 (56, 20.7).
// Loads of two to eight stages in registers instead of one: 11.1 to 13.7 us for the first; the loading
// waves also running the chains 11.3; 16 loading waves 11.2, stages of 32 steps 11.5.
//
// Operand forms: row-major with any row length (rows of an odd number of elements start anywhere; the
// 16-byte loads need no more than the element's alignment), or, for B, packed in fragment order
// (gemm_bpk.h).
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

// ---- int8: K split over the waves -------------------------------------------------------------------
template <SkinnyForm FORM, int MT_, int NT_, int NW_>
struct SkinnyConfig {
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
  using T = Mfma16I8;
  using Frag = T::Frag;
  using Acc = T::Acc;
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

// Waves per block.
inline int skinny_waves(int64_t M, int64_t N, int64_t Kb) { return (M < N ? M : N) <= 32 && Kb >= 4096 ? 16 : 8; }

// Calls go(Cfg{}) with the configuration of an M x N x Kb product whose A side is the one tiled by
// MT: up to 64 rows (32 with 16 waves) per block; two column tiles per block once 32-wide strips
// alone cover the CUs.
template <SkinnyForm FORM, class Go>
int skinny_dispatch(int64_t M, int64_t N, int64_t Kb, Go&& go) {
  const bool wide = (N + 31) / 32 * ((M + 63) / 64) >= 256;
  if (skinny_waves(M, N, Kb) == 16) {
    if (M <= 16) return wide ? go(SkinnyConfig<FORM, 1, 2, 16>{}) : go(SkinnyConfig<FORM, 1, 1, 16>{});
    return wide ? go(SkinnyConfig<FORM, 2, 2, 16>{}) : go(SkinnyConfig<FORM, 2, 1, 16>{});
  }
  if (M <= 16) return wide ? go(SkinnyConfig<FORM, 1, 2, 8>{}) : go(SkinnyConfig<FORM, 1, 1, 8>{});
  if (M <= 32) return wide ? go(SkinnyConfig<FORM, 2, 2, 8>{}) : go(SkinnyConfig<FORM, 2, 1, 8>{});
  return wide ? go(SkinnyConfig<FORM, 4, 2, 8>{}) : go(SkinnyConfig<FORM, 4, 1, 8>{});
}

// ---- bf16: chains over K ----------------------------------------------------------------------------
// A lane's 16 bytes of the first K step of the 16 rows of a row-major operand from row r0 on (rows past
// the end repeat the last), and of 16 columns of B (packed: unit (nb, kb) is 32 columns x 32 bytes, column
// c's half h at 16 (c + 32 h); N % 32 == 0).
__device__ __forceinline__ const char* row_source(const char* p, int r0, int rows, int Kb) {
  const int lane = threadIdx.x & 63, r = r0 + (lane & 15);
  return p + static_cast<int64_t>(r < rows ? r : rows - 1) * Kb + 16 * (lane >> 4);
}
template <bool PACKED>
__device__ __forceinline__ const char* column_source(const char* B, int n0, int N, int Kb) {
  if constexpr (!PACKED) return row_source(B, n0, N, Kb);
  const int lane = threadIdx.x & 63, c = n0 + (lane & 15), g = lane >> 4;
  return B + (static_cast<int64_t>(c >> 5) * (Kb / 32) + (g >> 1)) * 1024 + ((c & 31) + 32 * (g & 1)) * 16;
}

// The step K ends in, of the rows whose first step is at `src`: bytes past K are 0, whatever lies there.
__device__ __forceinline__ bf16x8 last_step(const char* p, const char* src, int rows, int Kb) {
  const int at = Kb / 64 * 64, keep = Kb - at - 16 * (static_cast<int>(threadIdx.x & 63) >> 4);
  return __builtin_bit_cast(bf16x8, first_bytes(load16_to_end(p, src - p + at, static_cast<int64_t>(rows) * Kb), keep));
}

// A wave's 16 x 16 tile at (m0, n0): element r of lane l is row 4 (l / 16) + r, column l % 16.
template <class Out>
__device__ __forceinline__ void tile_out(const f32x4_acc& acc, int m0, int n0, int M, int N, Out&& out) {
  const int lane = threadIdx.x & 63, col = n0 + (lane & 15), row = m0 + 4 * (lane >> 4);
  if (col >= N) return;
#pragma unroll
  for (int r = 0; r < 4; ++r)
    if (row + r < M) out(row + r, col, acc[r]);
}

template <SkinnyForm FORM, int MT_, int NT_>
struct ChainConfig {
  static constexpr bool kPacked = FORM == kSkinnyPacked;
  static constexpr int MT = MT_, NT = NT_, TILES = MT * NT;
  static constexpr int BM = 16 * MT, BN = 16 * NT;
  static constexpr int NW = 8, THREADS = 64 * (TILES + NW);  // waves 0 .. TILES - 1 run the chains, the others load
  static constexpr int PARTS = MT + NT;                      // fragments of a K step, 1 KiB each
  static constexpr int S = TILES == 1 ? 16 : 8;              // K steps per stage
  static constexpr int L = S * PARTS / NW;                   // fragments a wave loads per stage
  static constexpr int STAGE = S * PARTS * 1024, LDS_BYTES = 2 * STAGE;
  static_assert(L * NW == S * PARTS, "a stage's fragments must split evenly over the loading waves");
  static_assert(THREADS <= 1024 && LDS_BYTES <= 160 * 1024, "gfx950 workgroup limits");
};

// As skinny_gemm.
template <class Cfg, class Out>
__device__ __forceinline__ void skinny_chain(const char* __restrict__ A, const char* __restrict__ B, int M, int N, int Kb, int m0,
                                             int n0, char* smem, Out&& out) {
  using Mma = Mfma16Bf16;
  constexpr int MT = Cfg::MT, NT = Cfg::NT, NW = Cfg::NW, S = Cfg::S, L = Cfg::L, PARTS = Cfg::PARTS;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int whole = Kb / 64;  // the last step, when K ends inside it, is taken after the loop
  const int stages = whole / S + (whole % S != 0);

  // This lane's 16 bytes of part p (A's row tiles, then B's column tiles) of step 0.
  const auto source = [&](int p) {
    return p < MT ? row_source(A, m0 + 16 * p, M, Kb) : column_source<Cfg::kPacked>(B, n0 + 16 * (p - MT), N, Kb);
  };

  // Loading wave w takes fragments w, w + NW, ... of a stage, numbered step by step.
  const int w = wave - Cfg::TILES;
  const bool loads = w >= 0;
  const char* src[L];
  int pitch[L], step[L];
  u32x4 v[L];
  const auto load = [&](int stage) {
#pragma unroll
    for (int i = 0; i < L; ++i) {
      const int st = stage * S + step[i];  // past the end: one line for all lanes, its bytes unused
      v[i] = load16(st < whole ? src[i] + static_cast<int64_t>(st) * pitch[i] : A);
    }
  };
  const int ti = wave / NT, tj = wave % NT;  // a chain's tile
  const bool partial = !Cfg::kPacked && Kb % 64 != 0;
  f32x4_acc acc{0, 0, 0, 0};
  bf16x8 ka{}, kb{};
  if (loads) {
#pragma unroll
    for (int i = 0; i < L; ++i) {
      const int u = w + NW * i, p = u % PARTS;
      src[i] = source(p);
      pitch[i] = Cfg::kPacked && p >= MT ? 2048 : 64;
      step[i] = u / PARTS;
    }
    load(0);
  } else if (partial) {
    ka = last_step(A, source(ti), M, Kb);
    kb = last_step(B, source(MT + tj), N, Kb);
  }

  for (int st = 0; st < stages; ++st) {
    char* const area = smem + (st & 1) * Cfg::STAGE + lane * 16;  // read in stage st - 2, before the last barrier
    if (loads) {
#pragma unroll
      for (int i = 0; i < L; ++i) *reinterpret_cast<u32x4*>(area + (w + NW * i) * 1024) = v[i];
      load(st + 1);
    }
    __syncthreads();
    if (!loads) {
      const auto mma = [&](int k) {
        const char* const f = area + k * PARTS * 1024;
        acc = Mma::mma(*reinterpret_cast<const bf16x8*>(f + ti * 1024), *reinterpret_cast<const bf16x8*>(f + (MT + tj) * 1024), acc);
      };
      const int n = whole - st * S;
      if (n >= S) {
#pragma unroll
        for (int k = 0; k < S; ++k) mma(k);
      } else {
        for (int k = 0; k < n; ++k) mma(k);
      }
    }
  }
  if (loads) return;
  if (partial) acc = Mma::mma(ka, kb, acc);
  tile_out(acc, m0 + 16 * ti, n0 + 16 * tj, M, N, out);
}

// K of a few steps: nothing to stage, each wave loads the fragments of its own column tile straight
// into registers.
template <SkinnyForm FORM, int MT_>
struct DirectConfig {
  static constexpr bool kPacked = FORM == kSkinnyPacked;
  static constexpr int MT = MT_, NW = 4;
  static constexpr int BM = 16 * MT, BN = 16 * NW, THREADS = 64 * NW, LDS_BYTES = 0;
};

// As skinny_gemm.
template <class Cfg, class Out>
__device__ __forceinline__ void skinny_direct(const char* __restrict__ A, const char* __restrict__ B, int M, int N, int Kb, int m0,
                                              int n0, Out&& out) {
  constexpr int MT = Cfg::MT;
  n0 += 16 * static_cast<int>(threadIdx.x >> 6);
  if (n0 >= N) return;
  const char *a[MT], *b = column_source<Cfg::kPacked>(B, n0, N, Kb);
  f32x4_acc acc[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    a[i] = row_source(A, m0 + 16 * i, M, Kb);
    acc[i] = f32x4_acc{0, 0, 0, 0};
  }
  for (int st = 0; st < Kb / 64; ++st) {
    const bf16x8 fb = __builtin_bit_cast(bf16x8, load16(b + static_cast<int64_t>(st) * (Cfg::kPacked ? 2048 : 64)));
#pragma unroll
    for (int i = 0; i < MT; ++i) acc[i] = Mfma16Bf16::mma(__builtin_bit_cast(bf16x8, load16(a[i] + static_cast<int64_t>(st) * 64)), fb, acc[i]);
  }
  if (!Cfg::kPacked && Kb % 64 != 0) {
    const bf16x8 fb = last_step(B, b, N, Kb);
#pragma unroll
    for (int i = 0; i < MT; ++i) acc[i] = Mfma16Bf16::mma(last_step(A, a[i], M, Kb), fb, acc[i]);
  }
#pragma unroll
  for (int i = 0; i < MT; ++i) tile_out(acc[i], m0 + 16 * i, n0, M, N, out);
}

// Whether each wave loads for itself: K of up to 128, of 256 from 65536 columns on; above 16 rows, where
// the column fragments are used by two tiles of one wave, from 8192 columns on.  us through LDS stages
// (with K split over the waves) and here: [8][64] x [1000000] 123 (109), 36; [20] 164 (161), 49; [20][64] x
// [10000] 3.8 (3.7), 3.7 but x [1000] 3.0 (3.1), 3.6; [8][256] x [100000] 19.6 (22.5), 16.3 but x [10000] 4.6
// (5.6), 5.0; [1][33] x [100000] 13.5 (15.2), 6.5 (6.9 with a lane per output).
inline bool direct_runs(int64_t M, int64_t N, int64_t K) {
  return M <= 32 && K <= (N >= 65536 ? 256 : 128) && (M <= 16 || N >= 8192);
}

// Calls go(Cfg{}) with the configuration of an M x N x K product whose A side is the one tiled by MT: up
// to 64 rows per block; two column tiles per block where one makes more blocks than CUs (us for one and
// two: [127][4096] x [4000] 41.2, 28.7; [64][1000] x [4200] 10.6, 8.5; [32][4096] x [6000] 27.8, 21.3; [8] 17.4, 16.3).
template <SkinnyForm FORM, class Go>
int chain_dispatch(int64_t M, int64_t N, int64_t K, Go&& go) {
  if (direct_runs(M, N, K)) return M <= 16 ? go(DirectConfig<FORM, 1>{}) : go(DirectConfig<FORM, 2>{});
  const bool wide = (N + 15) / 16 * ((M + 63) / 64) > 256;
  if (M <= 16) return wide ? go(ChainConfig<FORM, 1, 2>{}) : go(ChainConfig<FORM, 1, 1>{});
  if (FORM == kSkinnyPacked || M <= 32) return wide ? go(ChainConfig<FORM, 2, 2>{}) : go(ChainConfig<FORM, 2, 1>{});
  if constexpr (FORM != kSkinnyPacked) return wide ? go(ChainConfig<FORM, 4, 2>{}) : go(ChainConfig<FORM, 4, 1>{});
}

}  // namespace vdsl
