// A block's tile of C = A W^T for many rows: bfloat16 operands through LDS, 32x32x16 matrix instructions (half the
// instructions and operand reads a product of 16x16x32).  Like tile_product.h, the rows are found through functions, so that they may be
// gathered (tokens sorted by expert), strided or plain; K a multiple of 8 and rows aligned to 16 bytes.
//
// WM x WN waves, each with TM x TN tiles of 32 x 32.  A step is 64 k-values, cut into four products of 16.
//   * The rows' pieces of 16 bytes go from memory straight into LDS (no registers hold them), STAGES steps ahead.  A load
//     instruction fills 1 KB of LDS in the order of its lanes, 8 rows of 128 bytes; which piece of its row a lane asks for
//     is XOR-swizzled with half the row's number, so that the operand reads of sixteen neighbouring rows cover all 64 banks
//     (4.5 cycles a read of 1 KB; swizzled with the row's number, two rows 8 apart meet: 8.5).
//   * Operands are read one product ahead into a second set of registers.  A wave waits at a step's one barrier only when it
//     has read all of the step and its last product but one is on its way.
//   * The loads into a step's buffer follow that barrier: SPREAD, a quarter behind each of the next four products (a compute
//     unit takes in 64 bytes a clock, so that the loads of a step take longer than one product's matrix instructions and
//     hold them up when they come together), or all of them between the matrix instructions of the last product, which has them under
//     way a step earlier: for two stages, and where the weights' way from memory is what a block waits for.
// Measured as a plain product of 2048 rows (the vendor's product beside it): N 4096, K 14336 208 us with 2 x 4 waves of 2 x 2 tiles, three
// stages, SPREAD (228 with all loads at once and the other swizzle; vendor 203), N 4096, K 4096 66 (71; 75), N 28672, K 4096 458 (492; 366),
// 8192 rows, N 2048, K 2048 73 (79; 66).
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
// W_ONCE: nobody else reads these rows of W soon.  works (the same in all lanes of a wave): false for a wave whose tiles nobody wants;
// it loads what the others need and multiplies nothing.  first (the same in the block): the step of 64 k-values that the walk over K starts
// with, and wraps round to: blocks whose rows lie a multiple of kilobytes apart and that walk in step crowd into few memory channels.
template <int WM, int WN, int TM, int TN, int STAGES, bool W_ONCE = false, bool SPREAD = false, typename ARow, typename WRow>
__device__ __forceinline__ void tile_product_lds(ARow a_row, WRow w_row, int K, bf16* lds, f32x16 (&acc)[TM][TN], bool works = true,
                                                 int first = 0) {
  typedef TileLds<WM, WN, TM, TN, STAGES> S;
  // load instructions of a step, 8 rows each: RA for rows of A and RB for rows of W a wave (where there are fewer rows of A
  // than waves can load, some waves load the same ones)
  constexpr int PIECES = TL_BK / 8, ROWS = WAVE / PIECES, PRODUCTS = TL_BK / 16;
  constexpr int GA = S::BM / ROWS, RA = GA >= S::WAVES ? GA / S::WAVES : 1, RB = S::BN / ROWS / S::WAVES, R = RA + RB;
  static_assert((GA % S::WAVES == 0 || S::WAVES % GA == 0) && S::BN % (ROWS * S::WAVES) == 0, "whole rounds of loads");
  constexpr int STAGE = (S::BM + S::BN) * TL_BK;  // elements
  const int lane = threadIdx.x & (WAVE - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int wm = wave / WN, wn = wave % WN, r = lane & 31, h = lane >> 5;
  static_assert(!SPREAD || STAGES >= 3, "a buffer to fill beside the step's and the next one's");
  const int lrow = lane / PIECES;
  auto piece_of = [&](int g) { return (lane % PIECES) ^ (((g * ROWS + lrow) >> 1) & (PIECES - 1)); };
  const bf16* src[R];
  unsigned put[R];
  int piece[R];  // (two values: with an even and an odd group of 8 rows)
  const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) bf16*)lds;
#pragma unroll
  for (int i = 0; i < RA; ++i) {
    const int g = (wave + i * S::WAVES) % GA;
    piece[i] = piece_of(g) * 8;
    src[i] = a_row(g * ROWS + lrow) + piece[i];
    put[i] = lds0 + g * ROWS * TL_BK * 2;
  }
#pragma unroll
  for (int i = 0; i < RB; ++i) {
    const int g = wave + i * S::WAVES;
    piece[RA + i] = piece_of(g) * 8;
    src[RA + i] = w_row(g * ROWS + lrow) + piece[RA + i];
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
    const int u = s + first;
    const int k0 = (s >= steps || u < steps ? u : u - steps) * TL_BK;
#pragma unroll
    for (int i = 0; i < R; ++i) from[i] = src[i] + k0;
    if (k0 + TL_BK > K) {  // uniform
#pragma unroll
      for (int i = 0; i < R; ++i) from[i] = k0 + piece[i] < K ? from[i] : (const void*)tile_zeros;
    }
  };
  bf16x8 av[2][TM], wv[2][TN];
  auto read = [&](int set, const bf16* base, int ks) {
    const int at = r * TL_BK + ((ks * 2 + h) ^ ((r >> 1) & (PIECES - 1))) * 8;
#pragma unroll
    for (int i = 0; i < TM; ++i) av[set][i] = *reinterpret_cast<const bf16x8*>(base + (wm * TM + i) * 32 * TL_BK + at);
#pragma unroll
    for (int j = 0; j < TN; ++j) wv[set][j] = *reinterpret_cast<const bf16x8*>(base + (S::BM + (wn * TN + j) * 32) * TL_BK + at);
  };

  constexpr int AHEAD = SPREAD ? STAGES - 1 : STAGES;  // steps that are asked for before the first product
#pragma unroll
  for (int s = 0; s < AHEAD; ++s) {
    find(s);
#pragma unroll
    for (int i = 0; i < R; ++i) load(i, from[i], put[i] + s * (STAGE * 2));
  }
  tile_wait<(AHEAD - 1) * R>();
  int stage = 0;
  if (!works) {
    for (int s = 0; s < steps; ++s) {
      if (!SPREAD) tile_wait<(STAGES - 2) * R>();
      find(s + AHEAD);
      const unsigned into = (SPREAD ? (stage == 0 ? STAGES - 1 : stage - 1) : stage) * (STAGE * 2);
#pragma unroll
      for (int l = 0; l < R; ++l) load(l, from[l], put[l] + into);
      if (SPREAD) tile_wait<(STAGES - 2) * R>();
      stage = stage == STAGES - 1 ? 0 : stage + 1;
    }
    tile_wait<0>();
    return;
  }
  read(0, lds, 0);
  if (SPREAD) find(STAGES - 1);
  // Loads of a product: all behind the last product's matrix instructions, or a part behind every product's.  At the last product's
  // barrier everybody has read the step, and the next one has to be there.
  constexpr int PER = SPREAD ? (R + PRODUCTS - 1) / PRODUCTS : R;
  constexpr int BEFORE = SPREAD ? ((PRODUCTS - 1) * PER < R ? (PRODUCTS - 1) * PER : R) : 0;  // of a step's loads, in front of its barrier
  for (int s = 0; s < steps; ++s) {
    const bf16* base = lds + stage * STAGE;
    const int next = stage == STAGES - 1 ? 0 : stage + 1;
    const unsigned into = (SPREAD ? (stage == 0 ? STAGES - 1 : stage - 1) : stage) * (STAGE * 2);
#pragma unroll
    for (int ks = 0; ks < PRODUCTS; ++ks) {
      const int set = ks & 1;
      const bool last = ks + 1 == PRODUCTS;
      if (!last) {
        read(set ^ 1, base, ks + 1);
      } else {
        tile_wait<(STAGES - (SPREAD ? 3 : 2)) * R + BEFORE>();
        read(set ^ 1, lds + next * STAGE, 0);
        if (!SPREAD) find(s + STAGES);
      }
      __builtin_amdgcn_sched_barrier(0);
      constexpr int EACH = (PER + TM * TN - 1) / (TM * TN);  // loads behind a matrix instruction
#pragma unroll
      for (int q = 0; q < TM * TN; ++q) {
        const int i = q / TN, j = q % TN;
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av[set][i], wv[set][j], acc[i][j], 0, 0, 0);
        if (!SPREAD && !last) continue;
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int n = q * EACH; n < (q + 1) * EACH && n < PER; ++n) {
          const int l = (SPREAD ? ks * PER : 0) + n;
          if (l < R) load(l, from[l], put[l] + into);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if (SPREAD) find(s + STAGES);
    stage = next;
  }
  tile_wait<0>();  // nothing is on its way to LDS when the block ends or uses it again
}
