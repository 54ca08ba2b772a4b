// The true 32-bit product y = x W^T (+ bias): float32 rows of x and W (K contiguous), float32 result.
//
// Sums of 16 products each in float32, added up in float64: what a long K costs is the rounding of short sums, not of
// every partial sum on the way.  The products and the short sums are the matrix unit's (mfma 32x32x2 and 16x16x4, float32
// throughout), the sums over the runs the vector unit's, side by side.
//
// Every kernel here adds in one order, so that a row's bits do not depend on how many rows there are, on the columns beside an
// element or on alignment:
//   * within a run k, k + 4, k + 8, k + 12 for k = 0 .. 3 (one 16x16x4 instruction, or two of 32x32x2, a k);
//   * the even runs in their order, the odd runs in theirs, then the two sums.
#include "common.h"
#include "fmsamd.h"
#include "tile_product_lds.h"

#define SG_RUN 16  // products of a float32 sum

// A product of TILE x TILE results, two (TILE 32) or four k-values; lane l of the result has column l % TILE and these rows.
template <int TILE>
__device__ __forceinline__ auto sgemm_mfma(float x, float w, float __attribute__((ext_vector_type(TILE * TILE / WAVE))) sum) {
  if constexpr (TILE == 32)
    return __builtin_amdgcn_mfma_f32_32x32x2f32(x, w, sum, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x4f32(x, w, sum, 0, 0, 0);
}
template <int TILE>
__device__ __forceinline__ int sgemm_row(int group, int e) {  // group: lane / TILE
  return TILE == 32 ? 8 * (e / 4) + 4 * group + e % 4 : 4 * group + e;
}

// Few rows (TILE 16), and rows that are not 16-byte aligned (VEC false).  A block's tile is TILE rows of x by TILE rows of W; its KS
// waves share K: of a step's RUNS * KS runs wave ks takes ks, ks + KS, ...  The step's rows wait in LDS while the next
// step's are on their way from memory in registers.  Rows of LDS are padded by four floats: the 16-byte reads of eight
// neighbouring rows then cover all banks.
// Two waves have the even and the odd runs and keep their sums.  Eight waves (one run each) hand the short sums over through LDS,
// where the step's rows were, and a thread adds up every second one of one element.  (Room of their own for the short sums
// leaves three blocks a compute unit where four fit: 64 rows by 4096 of K = 4096 take 55 us instead of 47.)
template <int TILE, int KS, int RUNS, bool VEC>
__global__ void __launch_bounds__(KS* WAVE)
    sgemm_kernel(const float* __restrict__ a, long lda, const float* __restrict__ w, const float* __restrict__ bias,
                 float* __restrict__ c, long ldc, int M, int N, int K, int m_tiles, int tiles) {
  constexpr bool HAND_OVER = KS > 2;
  static_assert(KS == 2 || (RUNS == 1 && KS % 2 == 0 && KS * WAVE == 2 * TILE * TILE), "a thread for the even or the odd runs of an element");
  constexpr int THREADS = KS * WAVE, BM = TILE, BN = TILE, BK = SG_RUN * RUNS * KS, LD = BK + 4;
  constexpr int PIECES = (BM + BN) * (BK / 4);  // of 16 bytes a step
  constexpr int LOADS = (PIECES + THREADS - 1) / THREADS;
  constexpr int ACC = TILE * TILE / WAVE;
  typedef float accv __attribute__((ext_vector_type(ACC)));
  constexpr int STEP = (BM + BN) * LD;  // floats
  static_assert(KS * TILE * TILE <= STEP, "the short sums, or the odd runs' sums in 64 bits, where a step's rows were");
  __shared__ __attribute__((aligned(16))) float lds[2 * STEP];

  // The tiles of x that share a tile of W follow one another on one of the eight dies (blocks are dealt to the dies in
  // turn), so that W comes from memory once.
  const int per_die = (tiles + 7) / 8;
  const int tile = (blockIdx.x & 7) * per_die + (blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per_die || tile >= tiles) return;
  const int m0 = (tile % m_tiles) * BM, n0 = (tile / m_tiles) * BN;

  const int lane = threadIdx.x & (WAVE - 1), ks = threadIdx.x / WAVE;
  const int r = lane % TILE, kq = lane / TILE;  // a lane's row and which four of a group of k-values it holds

  f32x4 ahead[LOADS];
  auto fetch = [&](int k0) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const int p = threadIdx.x + i * THREADS;
      const int row = p / (BK / 4), k = k0 + (p % (BK / 4)) * 4;
      f32x4 v = {0.f, 0.f, 0.f, 0.f};
      if (p < PIECES) {
        const bool of_x = row < BM;
        const int at = of_x ? m0 + row : n0 + row - BM;
        if (at < (of_x ? M : N)) {
          const float* src = of_x ? a + (size_t)at * lda : w + (size_t)at * K;
          if constexpr (VEC) {
            if (k < K) v = *reinterpret_cast<const f32x4*>(src + k);
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
              if (k + e < K) v[e] = src[k + e];
          }
        }
      }
      ahead[i] = v;
    }
  };
  auto put = [&](int buffer) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const int p = threadIdx.x + i * THREADS;
      if (p < PIECES) *reinterpret_cast<f32x4*>(lds + buffer * STEP + (p / (BK / 4)) * LD + (p % (BK / 4)) * 4) = ahead[i];
    }
  };

  constexpr int OWN = HAND_OVER ? 1 : ACC;  // elements that a thread keeps the sum of
  double total[OWN];
#pragma unroll
  for (int e = 0; e < OWN; ++e) total[e] = 0.0;
  // HAND_OVER: element threadIdx.x % (TILE * TILE) in the order in which the lanes hold them, even runs or odd ones
  const int odd = threadIdx.x / (TILE * TILE), element = threadIdx.x % (TILE * TILE);
  auto add = [&](int buffer) {
#pragma unroll
    for (int i = 0; i < KS / 2; ++i) total[0] += (double)lds[buffer * STEP + (2 * i + odd) * TILE * TILE + element];
  };

  fetch(0);
  put(0);
  __syncthreads();
  int buffer = 0;
  for (int k0 = 0; k0 < K; k0 += BK, buffer ^= 1) {
    const bool more = k0 + BK < K;
    if (more) fetch(k0 + BK);
    if (HAND_OVER && k0 > 0) add(buffer ^ 1);
    constexpr int GROUP = 4 * (WAVE / TILE), PARTS = SG_RUN / GROUP;  // k-values of one 16-byte piece a lane, such pieces of a run
#pragma unroll
    for (int i = 0; i < RUNS; ++i) {
      const float* sx = lds + buffer * STEP + r * LD + (i * KS + ks) * SG_RUN + kq * 4;
      f32x4 xv[PARTS], wv[PARTS];
#pragma unroll
      for (int g = 0; g < PARTS; ++g) {
        xv[g] = *reinterpret_cast<const f32x4*>(sx + g * GROUP);
        wv[g] = *reinterpret_cast<const f32x4*>(sx + BM * LD + g * GROUP);
      }
      accv acc;
#pragma unroll
      for (int e = 0; e < ACC; ++e) acc[e] = 0.f;
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int g = 0; g < PARTS; ++g) acc = sgemm_mfma<TILE>(xv[g][e], wv[g][e], acc);
      if constexpr (HAND_OVER) {
        __syncthreads();  // everybody has read the step's rows, and the short sums of the step before
        *reinterpret_cast<accv*>(lds + buffer * STEP + ks * TILE * TILE + lane * ACC) = acc;
      } else {
#pragma unroll
        for (int e = 0; e < ACC; ++e) total[e] += (double)acc[e];
      }
    }
    if (more) put(buffer ^ 1);
    __syncthreads();
  }
  if (HAND_OVER) add(buffer ^ 1);

  // the odd runs' sums, to the threads that have the even ones'
  double* const shared = reinterpret_cast<double*>(lds + buffer * STEP) + (HAND_OVER ? element : lane);
  const bool even = HAND_OVER ? odd == 0 : ks == 0;
  if (!even) {
#pragma unroll
    for (int e = 0; e < OWN; ++e) shared[e * WAVE] = total[e];
  }
  __syncthreads();
  if (!even) return;
#pragma unroll
  for (int e = 0; e < OWN; ++e) {
    const int of = HAND_OVER ? element / ACC : lane;  // the lane that had the element in the matrix unit's result
    const int m = m0 + sgemm_row<TILE>(of / TILE, HAND_OVER ? element % ACC : e), n = n0 + of % TILE;
    if (m < M && n < N) c[(size_t)m * ldc + n] = (float)(total[e] + shared[e * WAVE] + (bias ? bias[n] : 0.f));
  }
}

template <int TILE, int KS, int RUNS, bool VEC>
static void sgemm_launch(const float* a, long lda, const float* w, const float* bias, float* c, long ldc, int M, int N, int K,
                         hipStream_t stream) {
  const int m_tiles = ceil_div(M, TILE), tiles = m_tiles * ceil_div(N, TILE);
  sgemm_kernel<TILE, KS, RUNS, VEC><<<8 * ceil_div(tiles, 8), KS * WAVE, 0, stream>>>(a, lda, w, bias, c, ldc, M, N, K, m_tiles, tiles);
}

// The same for 16-byte aligned rows: the rows go from memory straight into LDS (tile_product_lds.h), STAGES - 1 steps of 32
// k-values ahead, in rows of 128 bytes whose pieces of 16 bytes are XOR-swizzled with the row.  WM x WN places of TILE x TILE results,
// two waves each: one has the even run of a step, the other the odd one.  The short sums of a step are converted and added
// while the matrix unit works on the next.
// A vector instruction costs a float32 product its own time (on this GPU a 64-bit one or a conversion 4.4 clocks, a 32-bit one 2.6, in
// kernels of nothing else, beside the 64 of a 32x32x2 product), so the loop has little but the two a result and run that the sums in 64 bits
// need: the steps are unrolled, so that places in LDS are constants and short sums stay where they are, and addresses advance in
// the scalar unit.
template <int TILE, int WM, int WN, int STAGES>
__global__ void __launch_bounds__(2 * WM* WN* WAVE) __attribute__((amdgpu_waves_per_eu(TILE == 32 ? 4 : 6)))
    sgemm_lds_kernel(const float* __restrict__ a, long lda, const float* __restrict__ w, const float* __restrict__ bias,
                     float* __restrict__ c, long ldc, int M, int N, int K, int m_tiles, int tiles) {
  constexpr int WAVES = 2 * WM * WN, BM = TILE * WM, BN = TILE * WN, BK = 2 * SG_RUN;
  constexpr int LOADS = (BM + BN) / 8 / WAVES;  // of 1 KB a step and wave, 8 rows each
  constexpr int STAGE = (BM + BN) * BK;         // floats
  constexpr int ACC = TILE * TILE / WAVE;
  typedef float accv __attribute__((ext_vector_type(ACC)));
  static_assert((BM + BN) % (8 * WAVES) == 0 && BM % 8 == 0, "whole rounds of loads, of x or of W");
  static_assert(BM * BN * 8 <= STAGES * STAGE * 4, "the waves of a place meet in the same LDS");
  __shared__ __attribute__((aligned(16))) float lds[STAGES * STAGE];
  const int per_die = (tiles + 7) / 8;
  const int tile = (blockIdx.x & 7) * per_die + (blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per_die || tile >= tiles) return;
  const int m0 = (tile % m_tiles) * BM, n0 = (tile / m_tiles) * BN;
  const int lane = threadIdx.x & (WAVE - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int ks = wave / (WM * WN), wm = (wave / WN) % WM, wn = wave % WN;
  const int r = lane % TILE, kq = lane / TILE;

  auto swizzle = [](int row) { return TILE == 32 ? (row >> 1) & 7 : row & 7; };
  const char* base[LOADS];  // the same in all lanes: of the block's first row of x or of W
  unsigned from[LOADS];     // bytes from there to this lane's piece (sgemm asks whether 32 bits hold them)
  int piece[LOADS];
  const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) float*)lds;
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int first = (wave * LOADS + i) * 8;  // of x, then of W
    const bool of_x = first < BM;              // uniform
    const int row = (of_x ? first : first - BM) + (lane >> 3), there = of_x ? M - m0 : N - n0;
    piece[i] = ((lane & 7) ^ swizzle(row)) * 4;
    base[i] = (const char*)(of_x ? a + (size_t)m0 * lda : w + (size_t)n0 * K);
    from[i] = (unsigned)((row < there ? row : 0) * (of_x ? lda : (long)K) + piece[i]) * 4;  // a row that is not there is the first one
  }
  auto fetch = [&](int s, int stage) {  // past the end: zeros, so that every step has the same number of loads under way
    const int k0 = s * BK;
    const unsigned to = lds0 + stage * (STAGE * 4) + wave * LOADS * 1024;
    if (k0 + BK <= K) {  // uniform
#pragma unroll
      for (int i = 0; i < LOADS; ++i) load_to_lds(base[i] + (size_t)k0 * 4, from[i], to + i * 1024);
    } else {
#pragma unroll
      for (int i = 0; i < LOADS; ++i)
        load_to_lds(k0 + piece[i] < K ? (const void*)(base[i] + (size_t)k0 * 4 + from[i]) : (const void*)tile_zeros, to + i * 1024);
    }
  };

  double total[ACC];
  accv sums[2];  // the short sums of this step and of the one before
#pragma unroll
  for (int e = 0; e < ACC; ++e) total[e] = 0.0, sums[0][e] = sums[1][e] = 0.f;
  const int steps = (K + BK - 1) / BK;
  for (int s = 0; s < STAGES - 1; ++s) fetch(s, s);
  constexpr int PARTS = TILE / 16;  // pieces of 16 bytes that a lane has of its row's run
  int x_at[PARTS], w_at[PARTS];
#pragma unroll
  for (int g = 0; g < PARTS; ++g) {
    const int at = r * BK + ((ks * 4 + g * (WAVE / TILE) + kq) ^ swizzle(r)) * 4;
    x_at[g] = wm * TILE * BK + at, w_at[g] = (BM + wn * TILE) * BK + at;
  }
  auto step = [&](int s, int stage, accv& sum, const accv& last) {
    tile_wait<(STAGES - 2) * LOADS>();  // step s is there, and everybody is done with step s - 1
    fetch(s + STAGES - 1, stage == 0 ? STAGES - 1 : stage - 1);
    f32x4 xv[PARTS], wv[PARTS];
#pragma unroll
    for (int g = 0; g < PARTS; ++g) {
      xv[g] = *reinterpret_cast<const f32x4*>(lds + stage * STAGE + x_at[g]);
      wv[g] = *reinterpret_cast<const f32x4*>(lds + stage * STAGE + w_at[g]);
    }
    __builtin_amdgcn_sched_barrier(0);  // all pieces are asked for before the first product (5% at 128 rows by 32000)
#pragma unroll
    for (int e = 0; e < ACC; ++e) sum[e] = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int g = 0; g < PARTS; ++g) sum = sgemm_mfma<TILE>(xv[g][e], wv[g][e], sum);
#pragma unroll
    for (int e = 0; e < ACC; ++e) total[e] += (double)last[e];
  };
  constexpr int ROUND = STAGES % 2 ? 2 * STAGES : STAGES;  // steps after which places and short sums are where they were
  for (int s0 = 0; s0 < steps; s0 += ROUND) {
#pragma unroll
    for (int u = 0; u < ROUND; ++u)
      if (s0 + u < steps) step(s0 + u, u % STAGES, sums[u & 1], sums[~u & 1]);  // uniform
  }
  if (steps & 1) {
#pragma unroll
    for (int e = 0; e < ACC; ++e) total[e] += (double)sums[0][e];
  } else {
#pragma unroll
    for (int e = 0; e < ACC; ++e) total[e] += (double)sums[1][e];
  }
  tile_wait<0>();

  // the odd runs' sums, to the waves that have the even ones'
  double* const shared = reinterpret_cast<double*>(lds) + (size_t)(wm * WN + wn) * TILE * TILE + lane;
  if (ks == 1) {
#pragma unroll
    for (int e = 0; e < ACC; ++e) shared[e * WAVE] = total[e];
  }
  __syncthreads();
  const int n = n0 + wn * TILE + r;
  if (ks == 1 || n >= N) return;
  const float b = bias ? bias[n] : 0.f;
#pragma unroll
  for (int e = 0; e < ACC; ++e) {
    const int m = m0 + wm * TILE + sgemm_row<TILE>(kq, e);
    if (m < M) c[(size_t)m * ldc + n] = (float)(total[e] + shared[e * WAVE] + b);
  }
}

template <int TILE, int WM, int WN, int STAGES>
static void sgemm_lds_launch(const float* a, long lda, const float* w, const float* bias, float* c, long ldc, int M, int N, int K,
                             hipStream_t stream) {
  const int m_tiles = ceil_div(M, TILE * WM), tiles = m_tiles * ceil_div(N, TILE * WN);
  sgemm_lds_kernel<TILE, WM, WN, STAGES><<<8 * ceil_div(tiles, 8), 2 * WM * WN * WAVE, 0, stream>>>(a, lda, w, bias, c, ldc, M, N, K, m_tiles, tiles);
}

// The tile shape.  What a compute unit needs for its blocks was measured at K = 4096 (8 to 512 rows of x, 4096 to 32000 of W):
// the first block costs `first` microseconds, every further one `next`, whatever the rows.  Small tiles fill the chip where
// there are few rows, large ones read less from LDS and the caches per product (301 rows by 32000: 73 TFLOP/s of 16 x 16, 85 of 32 x 32, 92 of
// 32 x 64; blocks of 64 x 64 and of 64 x 32 are within two per cent of the last, with four stages it takes a tenth longer).  Rows that are not 16-byte aligned have
// tiles of their own.
struct SgemmShape {
  int bm, bn;
  float first, next;
};
static const SgemmShape SGEMM_SHAPES[3] = {{16, 16, 22.f, 8.5f}, {32, 32, 39.f, 24.f}, {32, 64, 58.f, 45.f}};
static const SgemmShape SGEMM_UNALIGNED[2] = {{16, 16, 34.f, 28.f}, {32, 32, 126.f, 45.f}};
#define SGEMM_COMPUTE_UNITS 256

static int sgemm_rounds(const SgemmShape& s, int M, int N) {
  return (int)ceil_div((long)ceil_div(M, s.bm) * ceil_div(N, s.bn), SGEMM_COMPUTE_UNITS);
}

template <int SHAPES>
static int sgemm_shape(const SgemmShape (&shapes)[SHAPES], int M, int N) {
  int best = 0;
  float least = 0.f;
  for (int i = 0; i < SHAPES; ++i) {
    const float cost = shapes[i].first + shapes[i].next * (float)(sgemm_rounds(shapes[i], M, N) - 1);
    if (i == 0 || cost < least) best = i, least = cost;
  }
  return best;
}

#define SGEMM_NEAR (1 << 23)  // 64 rows of so many floats
static void sgemm(const float* a, long lda, const float* w, const float* bias, float* c, long ldc, int M, int N, int K, bool aligned,
                  hipStream_t stream) {
  if (aligned) {
    const bool near = lda < SGEMM_NEAR && K < SGEMM_NEAR;  // a tile's rows lie within 32 bits of bytes
    switch (near ? sgemm_shape(SGEMM_SHAPES, M, N) : 0) {
      case 0: sgemm_launch<16, 8, 1, true>(a, lda, w, bias, c, ldc, M, N, K, stream); break;
      case 1: sgemm_lds_launch<16, 2, 2, 4>(a, lda, w, bias, c, ldc, M, N, K, stream); break;
      default: sgemm_lds_launch<32, 1, 2, 3>(a, lda, w, bias, c, ldc, M, N, K, stream); break;
    }
  } else if (sgemm_shape(SGEMM_UNALIGNED, M, N) == 0) {
    sgemm_launch<16, 8, 1, false>(a, lda, w, bias, c, ldc, M, N, K, stream);
  } else if (sgemm_rounds(SGEMM_UNALIGNED[1], M, N) <= 2) {
    // a block or two a compute unit: long steps (128 rows by 4096 of K = 4095 150 us, 184 in short ones); more of them
    // hide one another's waits in short steps (301 rows: 423 against 290)
    sgemm_launch<32, 2, 4, false>(a, lda, w, bias, c, ldc, M, N, K, stream);
  } else {
    sgemm_launch<32, 2, 1, false>(a, lda, w, bias, c, ldc, M, N, K, stream);
  }
}

// What one launch takes: its threads are counted in 32 bits (and wrap round silently), at most two for a result.
#define SGEMM_LAUNCH_TILES (1 << 22)  // of 16 x 16 results

// Bound by the matrix unit's float32 rate (154 TFLOP/s for the vendor's product of 8192^3) and the vector instructions beside it, which
// take its time: with the 32 that the sums in 64 bits are for a run of 32 x 32 results some 120 would be left, and 110 are reached
// for 2048 rows (99 with the 57 of a loop that moved short sums and addresses); with few rows by the weights' bytes.  301 rows, K 4096: 630 us for 22016 rows of W (705),
// 134 for 4096 (144); 160 rows: 326 for 22016 (370), 82 for 4096 (85); 8 rows: 39 us for 12288 rows of W (5.0 TB/s), 23 for 4096.
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
