// A block's tile of C = A W^T for many rows: bfloat16 operands through LDS, 32x32x16 matrix instructions (they run at twice
// the rate of 16x16x32 on this GPU).  Like tile_product.h, the rows are found through functions, so that they may be
// gathered (tokens sorted by expert), strided or plain; K a multiple of 8 and rows aligned to 16 bytes.
//
// WM x WN waves, each with TM x TN tiles of 32 x 32.  A step is 64 k-values, cut into four products of 16.
//   * The rows' pieces of 16 bytes go from memory straight into LDS (no registers hold them), STAGES steps ahead.  A load
//     instruction fills 1 KB of LDS in the order of its lanes, 8 rows of 128 bytes; which piece of its row a lane asks for
//     is XOR-swizzled with the row, so that the operand reads of eight neighbouring rows cover all banks.
//   * Operands are read one product ahead into a second set of registers.  A wave waits at a step's one barrier only when it
//     has read all of the step and its last product but one is on its way; the loads into the step's buffer are then asked for
//     between the matrix instructions of the last product.
// Measured as a plain product of 2048 rows with STAGES = 2 (the vendor's product beside it): N 4096, K 14336 212 us with
// 2 x 4 waves of 2 x 2 tiles (193), N 28672, K 4096 448 us with 2 x 4 waves of 4 x 2 tiles (376).  With operands read where they
// are used 252 and 487, with the loads before the last product's matrix instructions 222 and 457, with steps of 32 k-values
// 240 and 489.
#pragma once

#include "common.h"

#define TL_BK 64

template <int WM, int WN, int TM, int TN, int STAGES>
struct TileLds {
  static constexpr int WAVES = WM * WN, THREADS = WAVES * WAVE, BM = WM * TM * 32, BN = WN * TN * 32;
  static constexpr int LDS_ELEMENTS = STAGES * (BM + BN) * TL_BK;
};

__device__ __attribute__((aligned(16))) const unsigned int tile_zeros[4] = {0, 0, 0, 0};

// 64 lanes' 16 bytes each, from memory to LDS at `lds_at` + 16 * lane (lds_at: the same in all lanes).  The compiler does not
// know that this is a load: whoever reads the bytes waits for vmcnt and for the block's barrier first (tile_wait).
__device__ __forceinline__ void load_to_lds(const void* from, unsigned lds_at) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(from), "s"(lds_at) : "memory", "m0");
}

// The same for bytes that nobody else reads soon: they pass the caches by.
__device__ __forceinline__ void load_once_to_lds(const void* from, unsigned lds_at) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off nt" ::"v"(from), "s"(lds_at) : "memory", "m0");
}

// The same as load_to_lds from `offset` bytes behind an address that all lanes share.
__device__ __forceinline__ void load_to_lds(const void* base, unsigned offset, unsigned lds_at) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(offset), "s"(base), "s"(lds_at) : "memory", "m0");
}

// All but the last OUTSTANDING loads of this wave have arrived and its reads from LDS are done; then the block's barrier.
template <int OUTSTANDING>
__device__ __forceinline__ void tile_wait() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(OUTSTANDING) : "memory");
}

// a_row(m), m < BM, and w_row(n), n < BN, return the first element of a row that can be read; a row that is not there is any
// row that is (its results are not stored).  After the call, lane l of wave w holds
//   acc[i][j][e] = C[row ((w / WN) * TM + i) * 32 + 8 (e / 4) + 4 (l / 32) + e % 4][column ((w % WN) * TN + j) * 32 + l % 32].
// W_ONCE: nobody else reads these rows of W soon.
template <int WM, int WN, int TM, int TN, int STAGES, bool W_ONCE = false, typename ARow, typename WRow>
__device__ __forceinline__ void tile_product_lds(ARow a_row, WRow w_row, int K, bf16* lds, f32x16 (&acc)[TM][TN]) {
  typedef TileLds<WM, WN, TM, TN, STAGES> S;
  // load instructions of a step, 8 rows each: RA for rows of A and RB for rows of W a wave (where there are fewer rows of A
  // than waves can load, some waves load the same ones)
  constexpr int PIECES = TL_BK / 8, ROWS = WAVE / PIECES, PRODUCTS = TL_BK / 16;
  constexpr int GA = S::BM / ROWS, RA = GA >= S::WAVES ? GA / S::WAVES : 1, RB = S::BN / ROWS / S::WAVES, R = RA + RB;
  static_assert((GA % S::WAVES == 0 || S::WAVES % GA == 0) && S::BN % (ROWS * S::WAVES) == 0, "whole rounds of loads");
  constexpr int STAGE = (S::BM + S::BN) * TL_BK;  // elements
  const int lane = threadIdx.x & (WAVE - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int wm = wave / WN, wn = wave % WN, r = lane & 31, h = lane >> 5;
  const int lrow = lane / PIECES, piece = (lane % PIECES) ^ (lrow & (PIECES - 1));
  const bf16* src[R];
  unsigned put[R];
  const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) bf16*)lds;
#pragma unroll
  for (int i = 0; i < RA; ++i) {
    const int g = (wave + i * S::WAVES) % GA;
    src[i] = a_row(g * ROWS + lrow) + piece * 8;
    put[i] = lds0 + g * ROWS * TL_BK * 2;
  }
#pragma unroll
  for (int i = 0; i < RB; ++i) {
    const int g = wave + i * S::WAVES;
    src[RA + i] = w_row(g * ROWS + lrow) + piece * 8;
    put[RA + i] = lds0 + (S::BM + g * ROWS) * TL_BK * 2;
  }
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  auto load = [&](int i, const void* from, unsigned to) {
    if (W_ONCE && i >= RA)
      load_once_to_lds(from, to);
    else
      load_to_lds(from, to);
  };
  const int steps = (K + TL_BK - 1) / TL_BK;
  const void* from[R];
  // where step s comes from; past the end: zeros, so that every step has the same number of loads under way
  auto find = [&](int s) {
    const int k0 = s * TL_BK;
#pragma unroll
    for (int i = 0; i < R; ++i) from[i] = src[i] + k0;
    if (k0 + TL_BK > K) {  // uniform
      const bool in = k0 + piece * 8 < K;
#pragma unroll
      for (int i = 0; i < R; ++i) from[i] = in ? from[i] : (const void*)tile_zeros;
    }
  };
  bf16x8 av[2][TM], wv[2][TN];
  auto read = [&](int set, const bf16* base, int ks) {
    const int at = r * TL_BK + ((ks * 2 + h) ^ (r & (PIECES - 1))) * 8;
#pragma unroll
    for (int i = 0; i < TM; ++i) av[set][i] = *reinterpret_cast<const bf16x8*>(base + (wm * TM + i) * 32 * TL_BK + at);
#pragma unroll
    for (int j = 0; j < TN; ++j) wv[set][j] = *reinterpret_cast<const bf16x8*>(base + (S::BM + (wn * TN + j) * 32) * TL_BK + at);
  };

#pragma unroll
  for (int s = 0; s < STAGES; ++s) {
    find(s);
#pragma unroll
    for (int i = 0; i < R; ++i) load(i, from[i], put[i] + s * (STAGE * 2));
  }
  tile_wait<(STAGES - 1) * R>();
  read(0, lds, 0);
  int stage = 0;
  for (int s = 0; s < steps; ++s) {
    const bf16* base = lds + stage * STAGE;
    const int next = stage == STAGES - 1 ? 0 : stage + 1;
#pragma unroll
    for (int ks = 0; ks < PRODUCTS; ++ks) {
      const int set = ks & 1;
      if (ks + 1 < PRODUCTS) {
        read(set ^ 1, base, ks + 1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av[set][i], wv[set][j], acc[i][j], 0, 0, 0);
      } else {
        tile_wait<(STAGES - 2) * R>();  // everybody has read step s, and step s + 1 is there
        read(set ^ 1, lds + next * STAGE, 0);
        find(s + STAGES);
        __builtin_amdgcn_sched_barrier(0);
        constexpr int PER = (R + TM * TN - 1) / (TM * TN);  // loads behind a matrix instruction
#pragma unroll
        for (int q = 0; q < TM * TN; ++q) {
          const int i = q / TN, j = q % TN;
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av[set][i], wv[set][j], acc[i][j], 0, 0, 0);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int l = q * PER; l < (q + 1) * PER && l < R; ++l) load(l, from[l], put[l] + stage * (STAGE * 2));
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    stage = next;
  }
  tile_wait<0>();  // nothing is on its way to LDS when the block ends or uses it again
}
