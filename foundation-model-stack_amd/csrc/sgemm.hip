// The true 32-bit product y = x W^T (+ bias): float32 rows of x and W (K contiguous), float32 result.
//
// A float32 number is the sum of three bfloat16 numbers, each the rounded rest of the one before: 24 bits are 8 + 8 + 8, so the sum
// is exact.  Of the nine products of two such sums the six largest are multiplied, each exactly, on the matrix unit; what
// the other three would add is less than 2^-24 of a product, which is what its rounding to float32 may take (2^-28 in the mean, of either sign).
// Numbers that all have the largest second and third parts, and those of one sign, lose it every time: rows and weights of 1 to 2 with such parts
// lie 3.5e-8 to 5.2e-8 from 64 bits, where float32 instructions have 2.6e-8 to 4.1e-8 (of either sign 4.9e-8 and 7.9e-8).  Six bfloat16
// products take 96 clocks for 16 x 16 results and 32 k-values where float32 ones take 256, and vector instructions run beside them.
//
// Sums of 32 products each in float32, small terms first, added up in float64.  The matrix unit's sums round down, not to nearest, which
// would add up over many of them (relative error 8.2e-8 at K = 4096, 1.2e-7 at 11008): every other run's x is negated and its sum subtracted,
// so that what rounds down in one rounds up in the next (4.5e-8 at both; float32 products in sums of 16 had 7.8e-8).  The runs' signs are
// + - - + over and over, so that the same holds where every other run is zero (9.2e-8 at 11008 with + -).
//
// Every kernel here adds in one order, so that a row's bits do not depend on how many rows there are, on the columns beside an
// element or on alignment:
//   * a run of 32 k-values: (x3, w1), (x1, w3), (x2, w2), (x2, w1), (x1, w2), (x1, w1), one 16x16x32 instruction each;
//   * the even runs in their order, the odd runs in theirs, every other one negated, then the first sum less the second.
// Short rows (sgemm_is_short: by K alone) are summed in float64.
//
// A sum that is no finite number (an infinity among the factors, whose second part would be a NaN, or a number that rounds to one)
// is formed again, the element by itself, from products and sums in float64 (sgemm_tile_f64).
// Below 2^-109 a number's third part begins to leave bfloat16's range (the unit keeps subnormal numbers).  Results of a row with a number
// that its parts do not hold exactly are formed again like those that are not finite.
#include "common.h"
#include "fmsamd.h"
#include "tile_product_lds.h"

#define SG_RUN 32  // products of a float32 sum

typedef float f32x8 __attribute__((ext_vector_type(8)));
typedef float f32x4_at4 __attribute__((ext_vector_type(4), aligned(4)));  // the unit asks for no more
typedef unsigned u32x4_parts __attribute__((ext_vector_type(4)));
typedef float f32x2_parts __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2_parts __attribute__((ext_vector_type(2)));
struct SgemmParts {
  bf16x8 p[3];
};

// Two numbers at a time: 11 instructions where conversions by element take 15.  (The compiler forms the conversion: it does not look
// into inline assembly for registers that a matrix instruction in flight still reads or writes, and so puts no wait in front of it.)
// lost: its lower half becomes other than zero if the third rest of a number has bits that bfloat16 has not.
__device__ __forceinline__ SgemmParts sgemm_split(f32x8 v, unsigned& lost) {
  u32x4_parts w[3];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float a = v[2 * i], b = v[2 * i + 1];
#pragma unroll
    for (int p = 0; p < 3; ++p) {
      const unsigned pair = __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2_parts{a, b}), bf16x2_parts));
      w[p][i] = pair;
      if (p < 2) a -= __uint_as_float(pair << 16), b -= __uint_as_float(pair & 0xffff0000u);
    }
    lost |= __float_as_uint(a) | __float_as_uint(b);
  }
  SgemmParts parts;
#pragma unroll
  for (int p = 0; p < 3; ++p) parts.p[p] = __builtin_bit_cast(bf16x8, w[p]);
  return parts;
}

// Which of the 16 rows that a wave's lanes have split (lane l: row l % 16) have lost bits.
__device__ __forceinline__ unsigned sgemm_lost_rows(unsigned lost) {
  const unsigned long long lanes = __ballot((lost & 0xffffu) != 0);
  const unsigned half = (unsigned)lanes | (unsigned)(lanes >> 32);
  return (half | half >> 16) & 0xffffu;
}

// A run of 16 rows of x by TN tiles of 16 rows of W; lane l of a result has column l % 16 and rows 4 (l / 16) + e.
template <int TN>
__device__ __forceinline__ void sgemm_run(const bf16x8 (&x)[3], const SgemmParts (&w)[TN], f32x4 (&sum)[TN]) {
  constexpr int ORDER[6][2] = {{2, 0}, {0, 2}, {1, 1}, {1, 0}, {0, 1}, {0, 0}};
#pragma unroll
  for (int j = 0; j < TN; ++j) sum[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < 6; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
      sum[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x[ORDER[i][0]], w[j].p[ORDER[i][1]], sum[j], 0, 0, 0);
}

// 16 x 16 results of rows m0 .. of x and n0 .. of W from products and sums in float64, by a wave: lane l has column l % 16 and rows
// l / 16 + 4 e.  For results that the bfloat16 parts cannot give.  Bound by the matrix unit in float64 and the round trips in front of it; a
// product of nothing but such results takes some six times as long as another: 301 rows by 4096 of K = 4096 770 us instead of 120
// (by a thread for each result, K in series: 15800), 8 rows 99 instead of 15 (406); with one infinity in x 274 (960), in W 424 (5860).
typedef double f64x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ f64x4 sgemm_tile_f64(const float* a, long lda, const float* w, int m0, int n0, int M, int N, int K) {
  const int lane = threadIdx.x & (WAVE - 1), r = lane % 16, o = lane / 16;
  const float* const x = a + (size_t)min(m0 + r, M - 1) * lda + o * 4;  // a row that is not there is the last one
  const float* const y = w + (size_t)min(n0 + r, N - 1) * K + o * 4;
  f64x4 sum = {0.0, 0.0, 0.0, 0.0};
  int k = 0;
#pragma unroll 2
  for (; k + 16 <= K; k += 16) {
    const f32x4_at4 u = *reinterpret_cast<const f32x4_at4*>(x + k), v = *reinterpret_cast<const f32x4_at4*>(y + k);
#pragma unroll
    for (int e = 0; e < 4; ++e) sum = __builtin_amdgcn_mfma_f64_16x16x4f64((double)u[e], (double)v[e], sum, 0, 0, 0);
  }
  if (k < K) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const bool in = k + o * 4 + e < K;
      sum = __builtin_amdgcn_mfma_f64_16x16x4f64(in ? (double)x[k + e] : 0.0, in ? (double)y[k + e] : 0.0, sum, 0, 0, 0);
    }
  }
  return sum;
}

// Few rows, and rows that are not 16-byte aligned or very far apart.  A block's tile is 16 TM rows of x by 16 TN rows of W; its
// waves share K, wave i has the runs i, i + WAVES, ...  A lane asks for its eight k-values of each row itself, a run ahead, and splits
// them.  The waves hand their short sums over through LDS, and a thread adds up the even or the odd runs of an element.  Eight waves where K is
// long; with four of them few runs leave no wave idle and a compute unit has room for twice the blocks: one row by 32000 of K = 128 9.6 us
// and 6.5, of K = 320 18.3 and 12.6; 2048 rows by 4096 of K = 321 123 and 101.
template <int TM, int TN, int WAVES>
__global__ void __launch_bounds__(WAVES * WAVE)
    sgemm_few_kernel(const float* __restrict__ a, long lda, const float* __restrict__ w, const float* __restrict__ bias,
                     float* __restrict__ c, long ldc, int M, int N, int K, int m_tiles, int tiles) {
  static_assert(WAVES % 4 == 0, "a wave's runs have one sign");
  constexpr int THREADS = WAVES * WAVE, TILES = TM * TN, ELEMENTS = TILES * 256;
  // A thread adds up the even and the odd runs of its elements threadIdx.x, + THREADS, ...; with one tile the even or the odd ones.
  constexpr bool BOTH = ELEMENTS >= THREADS;
  constexpr int RESULTS = (ELEMENTS + THREADS - 1) / THREADS;
  __shared__ __attribute__((aligned(16))) float lds[2][WAVES][ELEMENTS];
  static_assert(TM <= 4 && TN <= 4, "a bit of 64 for every row");
  __shared__ unsigned long long lost_rows[WAVES][2];  // of x, of W

  // The tiles of x that share a tile of W follow one another on one of the eight dies (blocks are dealt to the dies in
  // turn), so that W comes from memory once.
  const int per_die = (tiles + 7) / 8;
  const int tile = (blockIdx.x & 7) * per_die + (blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per_die || tile >= tiles) return;
  const int m0 = (tile % m_tiles) * 16 * TM, n0 = (tile / m_tiles) * 16 * TN;
  const int lane = threadIdx.x & (WAVE - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int r = lane % 16, o = lane / 16;

  const float* src[TM + TN];  // a row that is not there is the last one
#pragma unroll
  for (int u = 0; u < TM; ++u) src[u] = a + (size_t)min(m0 + u * 16 + r, M - 1) * lda + o * 8;
#pragma unroll
  for (int u = 0; u < TN; ++u) src[TM + u] = w + (size_t)min(n0 + u * 16 + r, N - 1) * K + o * 8;
  f32x8 ahead[TM + TN];
  auto fetch = [&](int run) {
    const int k0 = run * SG_RUN;
    const bool whole = k0 + SG_RUN <= K;  // uniform
#pragma unroll
    for (int u = 0; u < TM + TN; ++u) {
      f32x8 v = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      if (whole) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const f32x4_at4 q = *reinterpret_cast<const f32x4_at4*>(src[u] + k0 + h * 4);
#pragma unroll
          for (int e = 0; e < 4; ++e) v[h * 4 + e] = q[e];
        }
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (k0 + o * 8 + e < K) v[e] = src[u][k0 + e];
      }
      ahead[u] = v;
    }
  };

  double total[RESULTS], odd[RESULTS];
#pragma unroll
  for (int i = 0; i < RESULTS; ++i) total[i] = odd[i] = 0.0;
  unsigned long long lost[2] = {};  // rows of x, of W (in scalar registers: vector ones would cost the block beside this one its place)
  const int rounds = (K + WAVES * SG_RUN - 1) / (WAVES * SG_RUN);
  fetch(wave);
  for (int t = 0; t < rounds; ++t) {
    SgemmParts x[TM], y[TN];
#pragma unroll
    for (int u = 0; u < TM; ++u) {
      unsigned bits = 0;
      x[u] = sgemm_split((wave ^ wave >> 1) & 1 ? -ahead[u] : ahead[u], bits);
      lost[0] |= (unsigned long long)sgemm_lost_rows(bits) << (u * 16);
    }
#pragma unroll
    for (int u = 0; u < TN; ++u) {
      unsigned bits = 0;
      y[u] = sgemm_split(ahead[TM + u], bits);
      lost[1] |= (unsigned long long)sgemm_lost_rows(bits) << (u * 16);
    }
    if (t + 1 < rounds) {
      fetch((t + 1) * WAVES + wave);
    } else {
      lost_rows[wave][0] = lost[0], lost_rows[wave][1] = lost[1];
    }
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      f32x4 sum[TN];
      sgemm_run<TN>(x[i].p, y, sum);
#pragma unroll
      for (int j = 0; j < TN; ++j) *reinterpret_cast<f32x4*>(&lds[t & 1][wave][(i * TN + j) * 256 + lane * 4]) = sum[j];
    }
    __syncthreads();  // and everybody is done with the sums of the round before the last
#pragma unroll
    for (int i = 0; i < RESULTS; ++i) {
      const int q = BOTH ? threadIdx.x + i * THREADS : threadIdx.x % ELEMENTS;
      if (ELEMENTS % THREADS != 0 && q >= ELEMENTS) continue;  // the same in the wave
#pragma unroll
      for (int run = 0; run < WAVES / 2; ++run) {
        const double sum = (double)lds[t & 1][2 * run + (BOTH ? 0 : threadIdx.x / ELEMENTS)][q];
        total[i] = run & 1 ? total[i] - sum : total[i] + sum;
        if (BOTH) {
          const double other = (double)lds[t & 1][2 * run + 1][q];
          odd[i] = run & 1 ? odd[i] - other : odd[i] + other;
        }
      }
    }
  }

  if constexpr (!BOTH) {  // the odd runs' sums, to the threads that have the even ones'
    double* const shared = reinterpret_cast<double*>(lds[rounds & 1]);  // nobody reads there any more
    if (threadIdx.x >= ELEMENTS) shared[threadIdx.x - ELEMENTS] = total[0];
    __syncthreads();
    if (threadIdx.x >= ELEMENTS) return;
    odd[0] = shared[threadIdx.x];
  }
  unsigned again = 0;  // bit i: the thread's result i
#pragma unroll
  for (int i = 0; i < RESULTS; ++i) {
    const int element = threadIdx.x + i * THREADS, of = element % 256 / 4;  // the lane that had it
    const int m = m0 + element / 256 / TN * 16 + of / 16 * 4 + element % 4, n = n0 + element / 256 % TN * 16 + of % 16;
    if ((ELEMENTS % THREADS != 0 && element >= ELEMENTS) || m >= M || n >= N) continue;
    const float v = (float)(total[i] - odd[i] + (bias ? bias[n] : 0.f));
    c[(size_t)m * ldc + n] = v;
    again |= fabsf(v) < INFINITY ? 0u : 1u << i;
  }
  unsigned long long rows = 0, cols = 0;
#pragma unroll
  for (int of_wave = 0; of_wave < WAVES; ++of_wave) rows |= lost_rows[of_wave][0], cols |= lost_rows[of_wave][1];
  if (rows | cols) {  // the same in the block
#pragma unroll
    for (int i = 0; i < RESULTS; ++i) {
      const int element = threadIdx.x + i * THREADS, of = element % 256 / 4;
      const int m = element / 256 / TN * 16 + of / 16 * 4 + element % 4, n = element / 256 % TN * 16 + of % 16;
      if ((ELEMENTS % THREADS == 0 || element < ELEMENTS) && m0 + m < M && n0 + n < N) again |= (unsigned)((rows >> m | cols >> n) & 1) << i;
    }
  }
  if (__any(again)) {  // the wave has four rows of a tile: rows 4 e + lane % 4, columns lane / 4
#pragma nounroll
    for (int i = 0; i < RESULTS; ++i) {
      if (!__any(again >> i & 1)) continue;
      const int tile16 = (wave * WAVE + i * THREADS) / 256, e = wave % 4;
      const int mt = m0 + tile16 / TN * 16, nt = n0 + tile16 % TN * 16;
      const f64x4 sum = sgemm_tile_f64(a, lda, w, mt, nt, M, N, K);
      const int m = mt + 4 * e + o, n = nt + r;
      if (__shfl((int)(again >> i & 1), r * 4 + o))
        c[(size_t)m * ldc + n] = (float)((e == 0 ? sum[0] : e == 1 ? sum[1] : e == 2 ? sum[2] : sum[3]) + (bias ? bias[n] : 0.f));
    }
  }
}

template <int TM, int TN, int WAVES>
static void sgemm_few_launch(const float* a, long lda, const float* w, const float* bias, float* c, long ldc, int M, int N, int K,
                             hipStream_t stream) {
  const int m_tiles = ceil_div(M, 16 * TM), tiles = m_tiles * ceil_div(N, 16 * TN);
  sgemm_few_kernel<TM, TN, WAVES><<<8 * ceil_div(tiles, 8), WAVES * WAVE, 0, stream>>>(a, lda, w, bias, c, ldc, M, N, K, m_tiles, tiles);
}

// Many 16-byte aligned rows: 16 MT rows of x by 16 NT WN rows of W a block, two waves for each 16 NT of them: one has the even runs, the
// other the odd ones.  A wave has its rows of W to itself and a share of the rows of x: both go straight into its own LDS (tile_product_lds.h), up to
// three runs ahead, in rows of 128 bytes whose pieces of 16 bytes are XOR-swizzled with the row.  What it has of x it splits for
// all waves of its runs, into LDS, once a block; W it splits into registers.  A run's split stands beside the products of the run before it.
template <int MT, int NT, int WN>
__global__ void __launch_bounds__(2 * WN* WAVE)
    sgemm_lds_kernel(const float* __restrict__ a, long lda, const float* __restrict__ w, const float* __restrict__ bias,
                     float* __restrict__ c, long ldc, int M, int N, int K, int m_tiles, int tiles) {
  static_assert(MT % WN == 0 && MT >= 2 && NT <= MT, "every wave has as many rows of x; a tile of W is split beside a tile of x");
  constexpr int BM = 16 * MT, BN = 16 * NT * WN, UNITS = NT + MT / WN, LOADS = 2 * UNITS;
  constexpr int RAW = UNITS * 2048;                 // bytes of a wave's run: units of 16 rows of 32 k-values, of W, then of x
  constexpr int PLANE = MT * 1024;                  // one of the three parts of a run of x: 16-byte pieces in the order of the lanes
  constexpr int PLANES = 2 * WN * 2 * RAW;          // where the parts begin
  constexpr int BYTES = PLANES + 2 * 2 * 3 * PLANE;
  static_assert(BM * BN * 8 <= BYTES, "the waves of a place meet in the same LDS");
  __shared__ __attribute__((aligned(16))) char lds[BYTES];
  __shared__ unsigned lost_rows[MT + NT * WN][2];  // of x, of W, in the even and the odd runs
  const int per_die = (tiles + 7) / 8;
  const int tile = (blockIdx.x & 7) * per_die + (blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per_die || tile >= tiles) return;
  const int m0 = (tile % m_tiles) * BM, n0 = (tile / m_tiles) * BN;
  const int lane = threadIdx.x & (WAVE - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int odd = wave / WN, wn = wave % WN;
  const int r = lane % 16, o = lane / 16;

  unsigned from[LOADS];  // bytes from the block's first row to this lane's piece (sgemm asks whether 32 bits hold them)
  int piece[2];          // which k-value that is
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int row16 = h * 8 + (lane >> 3);
    piece[h] = ((lane & 7) ^ (row16 >> 1)) * 4 + odd * SG_RUN;
#pragma unroll
    for (int u = 0; u < UNITS; ++u) {
      const int row = (u < NT ? wn * NT + u : wn * (MT / WN) + u - NT) * 16 + row16, there = u < NT ? N - n0 : M - m0;
      from[u * 2 + h] = (unsigned)((row < there ? row : 0) * (u < NT ? (long)K : lda) + piece[h]) * 4;  // a row that is not there is the first one
    }
  }
  const char* const first_w = (const char*)(w + (size_t)n0 * K);
  const char* const first_x = (const char*)(a + (size_t)m0 * lda);
  const unsigned mine = wave * 2 * RAW, lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) char*)lds + mine;
  constexpr int BK = 2 * SG_RUN;
  auto fetch = [&](int s, int stage) {  // past the end: zeros, so that every step has the same number of loads under way
    const int k0 = s * BK;
    if (k0 + BK <= K) {  // uniform
#pragma unroll
      for (int i = 0; i < LOADS; ++i)
        load_to_lds((i < 2 * NT ? first_w : first_x) + (size_t)k0 * 4, from[i], lds0 + stage * RAW + i * 1024);
    } else {
#pragma unroll
      for (int i = 0; i < LOADS; ++i)
        load_to_lds(k0 + piece[i & 1] < K ? (const void*)((i < 2 * NT ? first_w : first_x) + (size_t)k0 * 4 + from[i]) : (const void*)tile_zeros,
                    lds0 + stage * RAW + i * 1024);
    }
  };
  const unsigned at0 = mine + r * 128 + ((2 * o) ^ (r >> 1)) * 16, at1 = mine + r * 128 + ((2 * o + 1) ^ (r >> 1)) * 16;
  f32x8 raw[UNITS];
  unsigned lost[UNITS] = {};
  auto read = [&](int stage) {
#pragma unroll
    for (int u = 0; u < UNITS; ++u) {
      const f32x4 lo = *reinterpret_cast<const f32x4*>(lds + stage * RAW + u * 2048 + at0);
      const f32x4 hi = *reinterpret_cast<const f32x4*>(lds + stage * RAW + u * 2048 + at1);
      raw[u] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    }
  };
  auto put = [&](int stage) {  // (a run's stage is whether its number among its wave's runs is odd)
#pragma unroll
    for (int u = 0; u < MT / WN; ++u) {
      const SgemmParts parts = sgemm_split(odd ^ stage ? -raw[NT + u] : raw[NT + u], lost[NT + u]);
#pragma unroll
      for (int p = 0; p < 3; ++p)
        *reinterpret_cast<bf16x8*>(lds + PLANES + ((stage * 2 + odd) * 3 + p) * PLANE + (wn * (MT / WN) + u) * 1024 + lane * 16) = parts.p[p];
    }
  };

  double total[MT][NT][4];
  f32x4 last[NT];  // the short sums of the tiles before
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) total[i][j][e] = 0.0, last[j][e] = 0.f;
  auto add = [&](int i, int stage) {
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const double sum = (double)last[j][e];
        total[i][j][e] = stage ? total[i][j][e] - sum : total[i][j][e] + sum;
      }
  };

  SgemmParts parts[2][NT];
  fetch(0, 0);
  fetch(1, 1);
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LOADS) : "memory");
  read(0);
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // before the next run is written there
  fetch(2, 0);
#pragma unroll
  for (int j = 0; j < NT; ++j) parts[0][j] = sgemm_split(raw[j], lost[j]);
  put(0);
  const int steps = (K + BK - 1) / BK;
  auto step = [&](int s, int stage) {
    tile_wait<LOADS>();  // run s + 1 is there, the parts of x of run s too, and everybody is done with those of s - 1
    const char* const at = lds + PLANES + (stage * 2 + odd) * 3 * PLANE + lane * 16;
    bf16x8 x[3], next[3];
#pragma unroll
    for (int p = 2; p >= 0; --p) x[p] = *reinterpret_cast<const bf16x8*>(at + p * PLANE);
    read(stage ^ 1);
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      if (i + 1 < MT) {
#pragma unroll
        for (int p = 0; p < 3; ++p) next[p] = *reinterpret_cast<const bf16x8*>(at + p * PLANE + (i + 1) * 1024);
      }
      f32x4 sum[NT];
      sgemm_run<NT>(x, parts[stage], sum);
      add(i ? i - 1 : MT - 1, i ? stage : stage ^ 1);
      if (i == (MT > NT ? MT - NT - 1 : 0)) put(stage ^ 1);
      if (i >= MT - NT) parts[stage ^ 1][i - MT + NT] = sgemm_split(raw[i - MT + NT], lost[i - MT + NT]);
#pragma unroll
      for (int j = 0; j < NT; ++j) last[j] = sum[j];
#pragma unroll
      for (int p = 0; p < 3; ++p) x[p] = next[p];
      // a product of 16 clocks, then four vector instructions (5% against the compiler's order)
#pragma unroll
      for (int p = 0; p < 6 * NT; ++p) {
        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x2, 4, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    fetch(s + 3, stage ^ 1);
  };
  for (int s = 0; s < steps; s += 2) {
    step(s, 0);
    if (s + 1 < steps) step(s + 1, 1);  // uniform
  }
  add(MT - 1, (steps - 1) & 1);
  tile_wait<0>();
#pragma unroll
  for (int u = 0; u < UNITS; ++u)
    lost_rows[u < NT ? MT + wn * NT + u : wn * (MT / WN) + u - NT][odd] = sgemm_lost_rows(lost[u]);

  // the odd runs' sums, to the waves that have the even ones'
  double* const shared = reinterpret_cast<double*>(lds) + (size_t)wn * MT * NT * 256 + lane;
  if (odd) {
#pragma unroll
    for (int i = 0; i < MT * NT * 4; ++i) shared[i * WAVE] = total[i / (4 * NT)][i / 4 % NT][i % 4];
  }
  __syncthreads();
  if (odd) return;
  auto result = [&](int i, int j, int e, float b) { return (float)(total[i][j][e] - shared[((i * NT + j) * 4 + e) * WAVE] + b); };
  float finite = 0.f;  // or a NaN
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    const int n = n0 + (wn * NT + j) * 16 + r;
    const float b = bias && n < N ? bias[n] : 0.f;
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int m = m0 + i * 16 + o * 4 + e;
        const float v = result(i, j, e, b);
        finite = fmaf(v, 0.f, finite);
        if (m < M && n < N) c[(size_t)m * ldc + n] = v;
      }
  }
  unsigned rows[MT + NT], any = 0;
#pragma unroll
  for (int u = 0; u < MT + NT; ++u) {
    const int of = u < MT ? u : u + wn * NT;
    any |= rows[u] = lost_rows[of][0] | lost_rows[of][1];
  }
  if (any == 0 && !__any(finite != 0.f)) return;  // the same in the wave
  unsigned again = 0;                             // bit 4 (j MT + i) + e
  static_assert(MT * NT * 4 <= 32, "a bit for every result");
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    const int n = n0 + (wn * NT + j) * 16 + r;
    const float b = bias && n < N ? bias[n] : 0.f;
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const bool lost_bits = (rows[i] >> (o * 4 + e) | rows[MT + j] >> r) & 1;
        if (m0 + i * 16 + o * 4 + e < M && n < N && (lost_bits || !(fabsf(result(i, j, e, b)) < INFINITY)))
          again |= 1u << (4 * (j * MT + i) + e);
      }
  }
#pragma nounroll
  for (int t = 0; t < MT * NT; ++t) {
    const int bits = again >> (4 * t) & 15;
    if (!__any(bits)) continue;
    const int mt = m0 + t % MT * 16, nt = n0 + (wn * NT + t / MT) * 16;
    const f64x4 sum = sgemm_tile_f64(a, lda, w, mt, nt, M, N, K);
#pragma unroll
    for (int e = 0; e < 4; ++e)  // row 4 e + o: lane 16 e + r had it, as its result o
      if (__shfl(bits, 16 * e + r) >> o & 1)
        c[(size_t)(mt + 4 * e + o) * ldc + nt + r] = (float)(sum[e] + (bias ? bias[nt + r] : 0.f));
  }
}

template <int MT, int NT, int WN>
static void sgemm_lds_launch(const float* a, long lda, const float* w, const float* bias, float* c, long ldc, int M, int N, int K,
                             hipStream_t stream) {
  const int m_tiles = ceil_div(M, 16 * MT), tiles = m_tiles * ceil_div(N, 16 * NT * WN);
  sgemm_lds_kernel<MT, NT, WN><<<8 * ceil_div(tiles, 8), 2 * WN * WAVE, 0, stream>>>(a, lda, w, bias, c, ldc, M, N, K, m_tiles, tiles);
}

// At most SG_TINY products: a thread has a row of W and 16 rows of x, sums in float64.  Bound by the launch and the results' bytes: all of x is
// asked for at once (a row after the other, each a round trip: 48 rows by 768 of K = 4 5.1 us, now 3.6; 2048 by 4096 12.7 and 10.7).
#define SG_TINY 4
template <int K>
__global__ void __launch_bounds__(256)
    sgemm_tiny_kernel(const float* __restrict__ a, long lda, const float* __restrict__ w, const float* __restrict__ bias,
                      float* __restrict__ c, long ldc, int M, int N, int n_blocks) {
  constexpr int ROWS = 16;
  const int n = blockIdx.x % n_blocks * 256 + threadIdx.x, m0 = blockIdx.x / n_blocks * ROWS;
  if (n >= N) return;
  float x[ROWS][K], y[K];
#pragma unroll
  for (int i = 0; i < ROWS; ++i)
#pragma unroll
    for (int k = 0; k < K; ++k) x[i][k] = a[(size_t)min(m0 + i, M - 1) * lda + k];  // a row that is not there is the last one
#pragma unroll
  for (int k = 0; k < K; ++k) y[k] = w[(size_t)n * K + k];
  const float b = bias ? bias[n] : 0.f;
#pragma unroll
  for (int i = 0; i < ROWS; ++i) {
    if (m0 + i >= M) break;  // uniform
    double sum = 0.0;
#pragma unroll
    for (int k = 0; k < K; ++k) sum += (double)x[i][k] * (double)y[k];
    c[(size_t)(m0 + i) * ldc + n] = (float)(sum + b);
  }
}

template <int K>
static void sgemm_tiny_launch(const float* a, long lda, const float* w, const float* bias, float* c, long ldc, int M, int N, hipStream_t stream) {
  const int n_blocks = ceil_div(N, 256);
  sgemm_tiny_kernel<K><<<n_blocks * ceil_div(M, 16), 256, 0, stream>>>(a, lda, w, bias, c, ldc, M, N, n_blocks);
}

// Short rows: 16 TM rows of x by 16 TN rows of W a wave, products and sums on the matrix unit in float64, four of 4 k-values at a time.
// Lane l asks for four k-values of row l % 16 at a time, from memory to registers.  Bound by the matrix unit (4.6 us for 16 k-values of
// 2048 by 4096 results) and the results' bytes.  A wave of 64 x 64 results has its unit to itself, and nothing else to do while it stores:
// 2048 by 4096 of K = 32 22 us, as waves of 32 x 32 19, of 16 x 16 22; 301 by 4096 10.9, 6.6, 5.6.
template <int TM, int TN>
__global__ void __launch_bounds__(256)
    sgemm_short_kernel(const float* __restrict__ a, long lda, const float* __restrict__ w, const float* __restrict__ bias,
                       float* __restrict__ c, long ldc, int M, int N, int K, int m_tiles, int tiles) {
  const int lane = threadIdx.x & (WAVE - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int tile = blockIdx.x * (blockDim.x / WAVE) + wave;
  if (tile >= tiles) return;
  const int m0 = tile % m_tiles * 16 * TM, n0 = tile / m_tiles * 16 * TN;
  const int r = lane % 16, o = lane / 16;
  const float* src[TM + TN];  // a row that is not there is the last one
#pragma unroll
  for (int u = 0; u < TM; ++u) src[u] = a + (size_t)min(m0 + u * 16 + r, M - 1) * lda + o * 4;
#pragma unroll
  for (int u = 0; u < TN; ++u) src[TM + u] = w + (size_t)min(n0 + u * 16 + r, N - 1) * K + o * 4;
  f32x4 ahead[TM + TN];
  auto fetch = [&](int k0) {
    if (k0 + 16 <= K) {  // uniform
#pragma unroll
      for (int u = 0; u < TM + TN; ++u) ahead[u] = *reinterpret_cast<const f32x4_at4*>(src[u] + k0);
    } else {
#pragma unroll
      for (int u = 0; u < TM + TN; ++u)
#pragma unroll
        for (int e = 0; e < 4; ++e) ahead[u][e] = k0 + o * 4 + e < K ? src[u][k0 + e] : 0.f;
    }
  };
  f64x4 sum[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) sum[i][j] = f64x4{0.0, 0.0, 0.0, 0.0};
  fetch(0);
  for (int k0 = 0; k0 < K; k0 += 16) {
    f32x4 v[TM + TN];
#pragma unroll
    for (int u = 0; u < TM + TN; ++u) v[u] = ahead[u];
    if (k0 + 16 < K) fetch(k0 + 16);
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
          sum[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)v[i][e], (double)v[TM + j][e], sum[i][j], 0, 0, 0);
  }
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int n = n0 + j * 16 + r;
    if (n >= N) continue;
    const float b = bias ? bias[n] : 0.f;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int m = m0 + i * 16 + 4 * e + o;
        if (m < M) c[(size_t)m * ldc + n] = (float)(sum[i][j][e] + b);
      }
  }
}

// Up to so many tiles a block is one wave, which spreads them over the compute units: 16 rows by 4096 of K = 64 (256 tiles) 4.2 us as blocks of four
// waves, 3.9; by 12288 (768) 4.5 either way.
#define SGEMM_SHORT_ALONE 512
template <int TM, int TN>
static void sgemm_short_launch(const float* a, long lda, const float* w, const float* bias, float* c, long ldc, int M, int N, int K,
                               hipStream_t stream) {
  const int m_tiles = ceil_div(M, 16 * TM), tiles = m_tiles * ceil_div(N, 16 * TN);
  const int waves = tiles <= SGEMM_SHORT_ALONE ? 1 : 4;  // of a block
  sgemm_short_kernel<TM, TN><<<ceil_div(tiles, waves), waves * WAVE, 0, stream>>>(a, lda, w, bias, c, ldc, M, N, K, m_tiles, tiles);
}

// Which rows are short goes with K alone, so that a row's bits go with nothing else.  Against the best block of three parts, us: 2048 by 4096 of K = 80
// 34 and 38, 48 by 11008 6.2 and 6.8; with K = 96 three parts take 10 to 15% less.  Rows that cannot all be aligned: 2048 by 4096 of K = 97 46 and 55, 129 55
// and 68, 193 73 and 73, 48 by 11008 8.6, 9.9, 12.5 and 7.5, 9.5, 10.2.
static bool sgemm_is_short(int K) { return K <= (K % 4 == 0 ? 80 : 128); }

// The block: its results, the k-values of its steps and what it costs, in microseconds: the first round of blocks over the compute units and each
// of its steps, every further round and each of its steps, fitted to 3100 products (1 to 2048 rows of x by 64 to 32000 of W, K from 84 to 8192); the
// block that is chosen by them takes 1% longer than the fastest in the mean, the slowest hundredth 15%.  Small tiles fill the chip where there are few rows,
// and their waves share K; large ones split each number less often (301 rows by 12288 of W of K = 4096: 793 us of 16 x 16, 436 of 32 x 32, 285 of 32 x 64, 268 of
// 64 x 64, 209 of 64 x 128; 16 rows by 4096: 21, 32, 53, 67, 97).  Those through LDS (the last three) want 16-byte aligned rows.
struct SgemmShape {
  int bm, bn, step;
  float first, first_step, next, next_step;
};
#define SGEMM_FEW 8  // shapes that take any rows
#define SGEMM_SHAPES_N 11
static const SgemmShape SGEMM_SHAPES[SGEMM_SHAPES_N] = {
    {16, 16, 256, 3.28f, 0.93f, 0.17f, 0.77f}, {16, 32, 256, 3.29f, 1.52f, 0.24f, 1.42f}, {16, 48, 256, 3.27f, 2.33f, 1.58f, 2.02f},
    {16, 64, 256, 3.64f, 2.60f, 1.50f, 2.68f}, {32, 32, 256, 3.60f, 2.01f, 0.52f, 1.80f}, {16, 16, 128, 3.17f, 0.60f, 0.14f, 0.37f},
    {16, 32, 128, 3.37f, 0.99f, 0.21f, 0.60f}, {32, 32, 128, 3.73f, 1.27f, 0.54f, 0.83f}, {32, 64, 64, 5.00f, 0.82f, 1.70f, 0.54f},
    {64, 64, 64, 5.47f, 1.18f, 3.54f, 1.11f},  {64, 128, 64, 8.32f, 1.68f, 5.57f, 1.59f}};
#define SGEMM_COMPUTE_UNITS 256

static int sgemm_shape(int shapes, int M, int N, int K) {
  int best = 0;
  float least = 0.f;
  for (int i = 0; i < shapes; ++i) {
    const SgemmShape& s = SGEMM_SHAPES[i];
    const long rounds = ceil_div((long)ceil_div(M, s.bm) * ceil_div(N, s.bn), SGEMM_COMPUTE_UNITS);
    const float steps = (float)ceil_div(K, s.step);
    const float cost = s.first + s.first_step * steps + (float)(rounds - 1) * (s.next + s.next_step * steps);
    if (i == 0 || cost < least) best = i, least = cost;
  }
  return best;
}

// From so many tiles of 16 x 16 results on waves of 32 x 32 fill the chip: 96 by 32000 of K = 64 (12000 tiles) 17.3
// us as waves of 16 x 16, 13.9 of 32 x 32; 512 by 4096 (8192) 11.9 and 10.6, of K = 24 9.1 and 9.0; 96 by 11008 (4128) 8.7 and 9.8.
#define SGEMM_SHORT_TILES 8192
#define SGEMM_NEAR (1 << 22)  // 128 rows of so many floats lie within 32 bits of bytes
static void sgemm(const float* a, long lda, const float* w, const float* bias, float* c, long ldc, int M, int N, int K, bool aligned,
                  hipStream_t stream) {
  if (sgemm_is_short(K)) {
    if (K <= SG_TINY) {
      switch (K) {
        case 1: sgemm_tiny_launch<1>(a, lda, w, bias, c, ldc, M, N, stream); break;
        case 2: sgemm_tiny_launch<2>(a, lda, w, bias, c, ldc, M, N, stream); break;
        case 3: sgemm_tiny_launch<3>(a, lda, w, bias, c, ldc, M, N, stream); break;
        default: sgemm_tiny_launch<SG_TINY>(a, lda, w, bias, c, ldc, M, N, stream); break;
      }
    } else if ((long)ceil_div(M, 16) * ceil_div(N, 16) >= SGEMM_SHORT_TILES) {
      sgemm_short_launch<2, 2>(a, lda, w, bias, c, ldc, M, N, K, stream);
    } else {
      sgemm_short_launch<1, 1>(a, lda, w, bias, c, ldc, M, N, K, stream);
    }
    return;
  }
  const bool any = aligned && lda < SGEMM_NEAR && K < SGEMM_NEAR;
  switch (sgemm_shape(any ? SGEMM_SHAPES_N : SGEMM_FEW, M, N, K)) {
    case 0: sgemm_few_launch<1, 1, 8>(a, lda, w, bias, c, ldc, M, N, K, stream); break;
    case 1: sgemm_few_launch<1, 2, 8>(a, lda, w, bias, c, ldc, M, N, K, stream); break;
    case 2: sgemm_few_launch<1, 3, 8>(a, lda, w, bias, c, ldc, M, N, K, stream); break;
    case 3: sgemm_few_launch<1, 4, 8>(a, lda, w, bias, c, ldc, M, N, K, stream); break;
    case 4: sgemm_few_launch<2, 2, 8>(a, lda, w, bias, c, ldc, M, N, K, stream); break;
    case 5: sgemm_few_launch<1, 1, 4>(a, lda, w, bias, c, ldc, M, N, K, stream); break;
    case 6: sgemm_few_launch<1, 2, 4>(a, lda, w, bias, c, ldc, M, N, K, stream); break;
    case 7: sgemm_few_launch<2, 2, 4>(a, lda, w, bias, c, ldc, M, N, K, stream); break;
    case 8: sgemm_lds_launch<2, 2, 2>(a, lda, w, bias, c, ldc, M, N, K, stream); break;
    case 9: sgemm_lds_launch<4, 1, 4>(a, lda, w, bias, c, ldc, M, N, K, stream); break;
    default: sgemm_lds_launch<4, 2, 4>(a, lda, w, bias, c, ldc, M, N, K, stream); break;
  }
}

// What one launch takes: its threads are counted in 32 bits (and wrap round silently), at most two for a result.
#define SGEMM_LAUNCH_TILES (1 << 22)  // of 16 x 16 results

// Many rows: bound by the vector instructions of the split and of the sums in 64 bits, which overlap with the products only in part: a step of
// 64 x 128 results and 64 k-values takes 1.5 us, of which the products alone are 0.64 (1.8 PFLOP/s in bfloat16), the sums about 0.5, the splits 0.4.
// Few rows: the weights' bytes.  Against float32 products, K 4096, weights out of memory (us): 301 rows by 22016 rows of W 604 -> 420, by 4096 131 -> 106;
// 130 rows by 12288 190 -> 160; 48 by 32000 196 -> 137; 17 by 4096 30 -> 27; 8 by 4096 27 -> 20, by 11008 39 -> 40, by 12288 39 -> 43 and by 32000
// 92 -> 99 (x's rows are split by every block); 8 by 4096 of K = 11008 73 -> 52; rows that are not aligned, 301 by 4096 of K = 4095: 302 -> 160.
extern "C" int fmsamd_gemm_f32(const float* a, long lda, const float* w, const float* bias, float* c, long ldc, int M,
                               int N, int K, hipStream_t stream) {
  if (M == 0 || N == 0) return 0;
  FMS_REQUIRE(M > 0 && N > 0 && K > 0, "gemm_f32: bad sizes M=%d N=%d K=%d", M, N, K);
  FMS_REQUIRE(lda >= K && ldc >= N, "gemm_f32: leading dimensions too small");
  const bool aligned = K % 4 == 0 && lda % 4 == 0 && ((uintptr_t)a % 16) == 0 && ((uintptr_t)w % 16) == 0;
  const long cols = N < 16L * SGEMM_LAUNCH_TILES ? N : 16L * SGEMM_LAUNCH_TILES;
  const long rows = SGEMM_LAUNCH_TILES / ceil_div(cols, 16) * 16;
  for (long n = 0; n < N; n += cols)
    for (long m = 0; m < M; m += rows)
      sgemm(a + m * lda, lda, w + n * K, bias ? bias + n : nullptr, c + m * ldc + n, ldc, (int)(M - m < rows ? M - m : rows),
            (int)(N - n < cols ? N - n : cols), K, aligned, stream);
  FMS_LAUNCH_CHECK("gemm_f32");
  return 0;
}
