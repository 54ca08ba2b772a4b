// Tiles of C = A W^T for many rows, one after the other in a block that never lets the loads run dry: bfloat16 operands through a
// ring in LDS, 16x16x32 matrix instructions.
//
//   * The tile is as large as the registers hold (256 x 256 results a block): every byte from the caches and from LDS then feeds the
//     most products.  With random data it is the power of the chip that ends the rate, and bytes moved are power; so are sums, of which
//     a 16x16x32 instruction reads and writes half as many a product as a 32x32x16 one (8192 x 8192 x 8192: 795 us with 32x32x16
//     products, 720 with 16x16x32 in the same form; as it is now 725, with zeros for data, which take less power, 552, the vendor
//     library 687 and 487).
//   * A wave's tile is four quadrants, two halves of the block's rows of A by two halves of its rows of W.  A step is 64
//     k-values of them in the order (A0 W0) (A0 W1) (A1 W1) (A1 W0): each quadrant needs one new half, which is read from LDS
//     between the matrix instructions of the quadrant before it.
//   * A half is read as a whole, so its bytes in LDS are free long before the step ends: the ring is four pairs of halves,
//     (A0 W0) and (A1 W1) of two steps, and a pair is asked for one and a half steps before it is read.  Two barriers a step.  (Five and
//     six pairs are slower, 5 to 12 %: their places are no constants any more, and every address an addition.)
//   * The walk goes on over the tiles of a block: the first steps of the next tile are asked for in the last two of this one.
//   * Eight waves, two a SIMD, for the largest tile, whose sums then fit the ordinary registers; four waves with larger tiles of their own
//     and fewer reads from LDS where the sums leave room among the accumulation registers (256 x 192 8 % faster than with eight,
//     256 x 128 3 %).  With 256 x 256 and four waves the compiler moves sums about and spills.
//   * What a load instruction needs in m0 is set in front of a matrix instruction and used behind it: a wave alone on its SIMD
//     has 16 cycles between two matrix instructions, which are 3 other instructions (2 to 3 % with four waves).
#pragma once

#include <type_traits>
#include <utility>

#include "common.h"

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) const bf16x8 RingLds8;

template <typename F, int... I>
__device__ __forceinline__ void ring_each(F f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void ring_for(F f) {
  ring_each(f, std::make_integer_sequence<int, N>{});
}

// A descriptor for loads and stores of `bytes` bytes from p on; what lies outside reads as zero and is not written.
__device__ __forceinline__ i32x4 ring_buffer(const void* p, unsigned bytes) {
  const unsigned long at = (unsigned long)(uintptr_t)p;
  i32x4 d;
  d[0] = __builtin_amdgcn_readfirstlane((int)(unsigned)at);
  d[1] = __builtin_amdgcn_readfirstlane((int)(unsigned)(at >> 32) & 0xffff);
  d[2] = __builtin_amdgcn_readfirstlane((int)bytes);
  d[3] = 0x00020000;
  return d;
}

// WM x WN waves, each with 2 x 2 quadrants of 16 QM x 32 QN results.
template <int WM_, int WN_, int QM_, int QN_>
struct Ring {
  static constexpr int WM = WM_, WN = WN_, QM = QM_, QN = QN_, WAVES = WM * WN, THREADS = WAVES * WAVE;
  static constexpr int HM = WM * QM * 16, HN = WN * QN * 32, BM = 2 * HM, BN = 2 * HN;  // rows of a half, of the block
  // load instructions of a half, 8 rows each, and how many of them a wave has (some are loaded by two waves where they do not divide)
  static constexpr int GA = HM / 8, GW = HN / 8, RA = (GA + WAVES - 1) / WAVES, RW = (GW + WAVES - 1) / WAVES, PAIR = RA + RW;
  static constexpr int PAIR_BYTES = (HM + HN) * 128, LDS_BYTES = 4 * PAIR_BYTES;
  // the sums of rows 16 i.. and columns' group j of quadrant (a, b)
  static constexpr int at(int a, int b, int i, int j) { return ((a * 2 + b) * QM + i) * 2 * QN + j; }
  static constexpr int SUMS = 8 * QM * QN;
};

// A tile's operands: for each half the first byte and the number of bytes of its rows that exist.
struct RingTile {
  const void *a[2], *w[2];
  unsigned a_bytes[2], w_bytes[2];
};

// 64 lanes' 16 bytes each to LDS, ring_put says where (`at` + 16 * lane), ring_get what: no other instruction that uses m0 stands
// between the two (a test looks).
__device__ __forceinline__ void ring_put(unsigned at) { asm volatile("s_mov_b32 m0, %0" ::"s"(at) : "memory", "m0"); }
__device__ __forceinline__ void ring_get(unsigned offset, i32x4 from, unsigned k) {
  asm volatile("buffer_load_dwordx4 %0, %1, %2 offen lds" ::"v"(offset), "s"(from), "s"(k) : "memory");
}

// place(n, tile): the n-th tile of this block; false behind the last one.  finish(n, sums): its results; the lane's
// sums[at(a, b, i, j)] are of row a HM + (wave / WN) QM 16 + 16 i + lane % 16 and of columns
//   b HN + ((wave % WN) QN + j / 2) 32 + 8 (lane / 16) + 4 (j % 2) + 0..3
// of the tile (columns: rows of W), so that those of j and j + 1 are eight columns in a row.
// lda, ldw: bytes from row to row.  K: a multiple of 128, at least 256.  lds: LDS_BYTES.
template <typename R, typename Place, typename Finish>
__device__ __forceinline__ void ring_product(unsigned lda, unsigned ldw, int K, char* lds, Place place, Finish finish) {
  constexpr int WN = R::WN, QM = R::QM, QN = R::QN;
  // (as a value that the compiler does not know before: what it could work out ahead for several calls would be kept in registers)
  int thread = threadIdx.x;
  asm volatile("" : "+v"(thread));
  const int lane = thread & 63, wave = __builtin_amdgcn_readfirstlane(thread / 64);
  const int wm = wave / WN, wn = wave % WN, r = lane & 15, h = lane >> 4;
  const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) char*)lds;
  // A load instruction brings 8 rows of 128 bytes.  Which 16 bytes of its row a lane asks for is swizzled, so that the reads of
  // the 16 rows of an operand cover all banks: those of A are neighbours, those of W lie as the columns above say.
  unsigned oa[R::RA], ow[R::RW], pa[R::RA], pw[R::RW];
#pragma unroll
  for (int i = 0; i < R::RA; ++i) {
    const int group = (wave + i * R::WAVES) % R::GA, row = group * 8 + lane / 8;
    oa[i] = row * lda + ((lane % 8) ^ ((row >> 1) & 7)) * 16;
    pa[i] = lds0 + group * 1024;
  }
#pragma unroll
  for (int i = 0; i < R::RW; ++i) {
    const int group = (wave + i * R::WAVES) % R::GW, row = group * 8 + lane / 8;
    ow[i] = row * ldw + ((lane % 8) ^ (((row >> 1) & 1) | (((row >> 3) & 3) << 1))) * 16;
    pw[i] = lds0 + R::HM * 128 + group * 1024;
  }
  unsigned ra[2], rw[2];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
    const int piece = (ks * 4 + h) ^ (r >> 1);
    ra[ks] = lds0 + (wm * QM * 16 + r) * 128 + piece * 16;
    rw[ks] = lds0 + R::HM * 128 + (wn * QN * 32 + 8 * (r >> 2) + (r & 3)) * 128 + piece * 16;
  }
  bf16x8 av[2][2][QM], wv[2][2][2 * QN];
  f32x4 sums[R::SUMS];
  i32x4 sa[2], sw[2];
  int opened = 0;
  auto open = [&]() __attribute__((always_inline)) {  // the loads go on to the next tile
    RingTile t;
    const bool there = place(opened++, t);
    if (there) {
#pragma unroll
      for (int i = 0; i < 2; ++i) sa[i] = ring_buffer(t.a[i], t.a_bytes[i]), sw[i] = ring_buffer(t.w[i], t.w_bytes[i]);
    } else {  // nothing is read
#pragma unroll
      for (int i = 0; i < 2; ++i) sa[i][2] = 0, sw[i][2] = 0;
    }
    return there;
  };
  // pairs 0 and 2: A0 and W0 of the even and the odd step; 1 and 3: A1 and W1
  auto read_a = [&](int half, int n, int pair) __attribute__((always_inline)) {
    const int ks = n / QM, i = n % QM;
    av[half][ks][i] = *(RingLds8*)(uintptr_t)(ra[ks] + pair * R::PAIR_BYTES + i * 16 * 128);
  };
  auto read_w = [&](int set, int n, int pair) __attribute__((always_inline)) {
    const int ks = n / (2 * QN), j = n % (2 * QN);
    wv[set][ks][j] = *(RingLds8*)(uintptr_t)(rw[ks] + pair * R::PAIR_BYTES + (j / 2) * 32 * 128 + (j % 2) * 4 * 128);
  };
  unsigned k = 0;  // bytes along the rows: the step that is asked for
  bool here = open();
  if (!here) return;
#pragma unroll
  for (int p = 0; p < 4; ++p) {
#pragma unroll
    for (int i = 0; i < R::RA; ++i) {
      ring_put(pa[i] + p * R::PAIR_BYTES);
      asm volatile("s_nop 0");
      ring_get(oa[i], sa[p & 1], (p / 2) * 128);
    }
#pragma unroll
    for (int i = 0; i < R::RW; ++i) {
      ring_put(pw[i] + p * R::PAIR_BYTES);
      asm volatile("s_nop 0");
      ring_get(ow[i], sw[p & 1], (p / 2) * 128);
    }
  }
  // All but the last `n` loads of this wave have arrived and its reads from LDS are done; then the block's barrier.
  auto wait = [&](auto outstanding) __attribute__((always_inline)) {
    constexpr int n = decltype(outstanding)::value < 63 ? decltype(outstanding)::value : 63;
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt((n & 15) | 0x70 | (n >> 4) << 14);
    asm volatile("s_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  wait(std::integral_constant<int, 0>{});
#pragma unroll
  for (int n = 0; n < 2 * QM; ++n) read_a(0, n, 0);
#pragma unroll
  for (int n = 0; n < 4 * QN; ++n) read_w(0, n, 0);

  // Quadrant q of a step of parity p.  Read meanwhile: W1, A1, the next step's A0, its W0; asked for: A0, W0, W1, A1 of the step
  // after the next, into the places of the pair that all waves have read.
  auto quadrant = [&](auto qc, auto pc) __attribute__((always_inline)) {
    constexpr int q = decltype(qc)::value, p = decltype(pc)::value;
    constexpr int a = q >= 2, b = q == 1 || q == 2, set = b ^ p;
    constexpr int READS = q == 0 || q == 3 ? 4 * QN : 2 * QM, LOADS = q == 0 || q == 3 ? R::RA : R::RW, MFMAS = 4 * QM * QN;
    constexpr int OTHERS = READS + 2 * LOADS;  // a load is two instructions, with a matrix instruction between them
    constexpr int into = 2 * p + (q >= 2), next = (2 * p + 2) & 3;
    ring_for<MFMAS>([&](auto mc) __attribute__((always_inline)) {
      constexpr int m = decltype(mc)::value;
      // neighbours share an operand
      constexpr int ks = m / (2 * QM * QN), i = (m / (2 * QN)) % QM, j = i % 2 ? 2 * QN - 1 - m % (2 * QN) : m % (2 * QN);
      f32x4& c = sums[R::at(a, b, i, j)];
      c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv[set][ks][j], av[a][ks][i], c, 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      constexpr int from = m * OTHERS / MFMAS, to = (m + 1) * OTHERS / MFMAS;
      ring_for<to - from>([&](auto oc) __attribute__((always_inline)) {
        constexpr int o = from + decltype(oc)::value;
        if constexpr (o < READS) {
          if constexpr (q == 0) read_w(1 ^ p, o, 2 * p + 1);
          if constexpr (q == 1) read_a(1, o, 2 * p + 1);
          if constexpr (q == 2) read_a(0, o, next);
          if constexpr (q == 3) read_w(p ^ 1, o, next);
        } else {
          constexpr int l = (o - READS) / 2;
          if constexpr ((o - READS) % 2 == 0) {
            ring_put((q == 0 || q == 3 ? pa[l] : pw[l]) + into * R::PAIR_BYTES);
            if constexpr (o + 1 < to) asm volatile("s_nop 0");
          } else if constexpr (q == 0 || q == 3) {
            ring_get(oa[l], sa[q == 3], k);
          } else {
            ring_get(ow[l], sw[q == 2], k);
          }
        }
      });
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  typedef std::integral_constant<int, 0> C0;
  typedef std::integral_constant<int, 1> C1;
  typedef std::integral_constant<int, 2> C2;
  typedef std::integral_constant<int, 3> C3;
  // At a step's first barrier its pair (A1 W1) has arrived, at its second the next step's (A0 W0): all but the last two pairs that
  // were asked for.
  typedef std::integral_constant<int, 2 * R::PAIR> LastTwo;
  auto two_steps = [&]() __attribute__((always_inline)) {
    wait(LastTwo{});
    quadrant(C0{}, C0{});
    quadrant(C1{}, C0{});
    wait(LastTwo{});
    quadrant(C2{}, C0{});
    quadrant(C3{}, C0{});
    k += 128;
    wait(LastTwo{});
    quadrant(C0{}, C1{});
    quadrant(C1{}, C1{});
    wait(LastTwo{});
    quadrant(C2{}, C1{});
    quadrant(C3{}, C1{});
    k += 128;
  };
  const unsigned end = 2 * K;
  for (int n = 0; here; ++n) {
#pragma unroll
    for (int i = 0; i < R::SUMS; ++i) sums[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    bool last;
    k = 256;
    do {
      last = k == end;
      if (__builtin_expect(last, 0)) {
        here = open();
        k = 0;
      }
      two_steps();
    } while (!last);
    __builtin_amdgcn_sched_barrier(0);
    finish(n, sums);
    __builtin_amdgcn_sched_barrier(0);
  }
  wait(C0{});
}
