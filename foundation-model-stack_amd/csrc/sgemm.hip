// The true 32-bit product y = x W^T (+ bias): float32 rows of x and W (K contiguous), float32 result.
//
// Sums of 16 products each in float32, added up in float64: what a long K costs is the rounding of short sums, not of
// every partial sum on the way.  The products and the short sums are the matrix unit's (mfma 32x32x2 and 16x16x4, float32
// throughout), the sums over the runs the vector unit's, side by side.
#include "common.h"
#include "fmsamd.h"
#include "tile_product_lds.h"

#define SG_RUN 16  // products of a float32 sum

// Few rows, and rows that are not 16-byte aligned (VEC false).  A block's tile is TILE rows of x by TILE rows of W; its KS waves
// share K: of a step's SG_RUN * RUNS * KS k-values each takes SG_RUN * RUNS.  The step's rows wait in LDS while the next
// step's are on their way from memory in registers.  Rows of LDS are padded by four floats: the 16-byte reads of eight
// neighbouring rows then cover all banks.
template <int TILE, int KS, int RUNS, bool VEC>
__global__ void __launch_bounds__(KS* WAVE)
    sgemm_kernel(const float* __restrict__ a, long lda, const float* __restrict__ w, const float* __restrict__ bias,
                 float* __restrict__ c, long ldc, int M, int N, int K, int m_tiles, int tiles) {
  constexpr int THREADS = KS * WAVE, BM = TILE, BN = TILE, BK = SG_RUN * RUNS * KS, LD = BK + 4;
  constexpr int PIECES = (BM + BN) * (BK / 4);  // of 16 bytes a step
  constexpr int LOADS = (PIECES + THREADS - 1) / THREADS;
  constexpr int ACC = TILE * TILE / WAVE;
  typedef float accv __attribute__((ext_vector_type(ACC)));
  constexpr int REDUCE_BYTES = TILE * TILE * 8;
  constexpr int STEP_BYTES = 2 * (BM + BN) * LD * 4;
  __shared__ __attribute__((aligned(16))) unsigned char lds[STEP_BYTES > REDUCE_BYTES ? STEP_BYTES : REDUCE_BYTES];
  float* const steps = reinterpret_cast<float*>(lds);

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
      if (p < PIECES) *reinterpret_cast<f32x4*>(steps + buffer * (BM + BN) * LD + (p / (BK / 4)) * LD + (p % (BK / 4)) * 4) = ahead[i];
    }
  };

  double total[ACC];
#pragma unroll
  for (int e = 0; e < ACC; ++e) total[e] = 0.0;

  fetch(0);
  put(0);
  __syncthreads();
  int buffer = 0;
  for (int k0 = 0; k0 < K; k0 += BK, buffer ^= 1) {
    const bool more = k0 + BK < K;
    if (more) fetch(k0 + BK);
    const float* sx = steps + buffer * (BM + BN) * LD + r * LD + ks * SG_RUN * RUNS + kq * 4;
    const float* sw = sx + BM * LD;
    constexpr int GROUP = 4 * (WAVE / TILE);  // k-values of one 16-byte piece a lane
#pragma unroll
    for (int run = 0; run < RUNS; ++run) {
      accv acc;
#pragma unroll
      for (int e = 0; e < ACC; ++e) acc[e] = 0.f;
#pragma unroll
      for (int g = 0; g < SG_RUN / GROUP; ++g) {
        const f32x4 xv = *reinterpret_cast<const f32x4*>(sx + run * SG_RUN + g * GROUP);
        const f32x4 wv = *reinterpret_cast<const f32x4*>(sw + run * SG_RUN + g * GROUP);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if constexpr (TILE == 32)
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(xv[e], wv[e], acc, 0, 0, 0);
          else
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(xv[e], wv[e], acc, 0, 0, 0);
        }
      }
#pragma unroll
      for (int e = 0; e < ACC; ++e) total[e] += (double)acc[e];
    }
    if (more) put(buffer ^ 1);
    __syncthreads();
  }

  // the waves add up, in their order
  double* const shared = reinterpret_cast<double*>(lds) + lane;
#pragma unroll 1
  for (int s = 1; s < KS; ++s) {
    if (ks == s) {
#pragma unroll
      for (int e = 0; e < ACC; ++e) shared[e * WAVE] = total[e];
    }
    __syncthreads();
    if (ks == 0) {
#pragma unroll
      for (int e = 0; e < ACC; ++e) total[e] += shared[e * WAVE];
    }
    __syncthreads();
  }
  if (ks != 0) return;
  const int n = n0 + r;
  if (n >= N) return;
  const float b = bias ? bias[n] : 0.f;
#pragma unroll
  for (int e = 0; e < ACC; ++e) {
    // the matrix unit's result: column lane % TILE, rows in groups of four
    const int m = m0 + (TILE == 32 ? 8 * (e / 4) + 4 * kq + e % 4 : 4 * kq + e);
    if (m < M) c[(size_t)m * ldc + n] = (float)(total[e] + b);
  }
}

template <int TILE, int KS, int RUNS, bool VEC>
static void sgemm_launch(const float* a, long lda, const float* w, const float* bias, float* c, long ldc, int M, int N, int K,
                         hipStream_t stream) {
  const int m_tiles = ceil_div(M, TILE), tiles = m_tiles * ceil_div(N, TILE);
  sgemm_kernel<TILE, KS, RUNS, VEC><<<8 * ceil_div(tiles, 8), KS * WAVE, 0, stream>>>(a, lda, w, bias, c, ldc, M, N, K, m_tiles, tiles);
}

// The same for 16-byte aligned rows and tiles of 32 x 32 a wave: the rows go from memory straight into LDS (tile_product_lds.h),
// STAGES - 1 steps of 32 k-values ahead, in rows of 128 bytes whose pieces of 16 bytes are XOR-swizzled with the row.  The KS
// waves of a place share a step's two runs.  The short sums of one run are converted and added while the matrix unit
// works on the other.
template <int WM, int WN, int KS, int STAGES>
__global__ void __launch_bounds__(WM* WN* KS* WAVE)
    sgemm_lds_kernel(const float* __restrict__ a, long lda, const float* __restrict__ w, const float* __restrict__ bias,
                     float* __restrict__ c, long ldc, int M, int N, int K, int m_tiles, int tiles) {
  constexpr int WAVES = WM * WN * KS, BM = 32 * WM, BN = 32 * WN, BK = 32;
  constexpr int LOADS = (BM + BN) / 8 / WAVES;  // of 1 KB a step and wave, 8 rows each
  constexpr int STAGE = (BM + BN) * BK;         // floats
  static_assert((BM + BN) % (8 * WAVES) == 0, "whole rounds of loads");
  static_assert(KS == 1 || WM * WN * 32 * 32 * 8 <= STAGES * STAGE * 4, "the waves of a place meet in the same LDS");
  __shared__ __attribute__((aligned(16))) float lds[STAGES * STAGE];
  const int per_die = (tiles + 7) / 8;
  const int tile = (blockIdx.x & 7) * per_die + (blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per_die || tile >= tiles) return;
  const int m0 = (tile % m_tiles) * BM, n0 = (tile / m_tiles) * BN;
  const int lane = threadIdx.x & (WAVE - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int ks = wave / (WM * WN), wm = (wave / WN) % WM, wn = wave % WN;
  const int r = lane & 31, h = lane >> 5;

  const int piece = (lane & 7) ^ ((lane >> 3) & 7);
  const float* src[LOADS];
  const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) float*)lds;
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int row = (wave * LOADS + i) * 8 + (lane >> 3);  // of x, then of W; a row that is not there is the first one
    const bool of_x = row < BM;
    const int at = of_x ? m0 + row : n0 + row - BM;
    src[i] = (of_x ? a + (size_t)(at < M ? at : 0) * lda : w + (size_t)(at < N ? at : 0) * K) + piece * 4;
  }
  auto fetch = [&](int s, int stage) {  // past the end: zeros, so that every step has the same number of loads under way
    const int k0 = s * BK;
    const unsigned to = lds0 + stage * (STAGE * 4) + wave * LOADS * 1024;
    if (k0 + BK <= K) {  // uniform
#pragma unroll
      for (int i = 0; i < LOADS; ++i) load_to_lds(src[i] + k0, to + i * 1024);
    } else {
      const bool in = k0 + piece * 4 < K;
#pragma unroll
      for (int i = 0; i < LOADS; ++i) load_to_lds(in ? (const void*)(src[i] + k0) : (const void*)tile_zeros, to + i * 1024);
    }
  };

  double total[16];
#pragma unroll
  for (int e = 0; e < 16; ++e) total[e] = 0.0;
  constexpr int RUNS = 2 / KS;  // of a wave in a step
  f32x16 acc[2];
#pragma unroll
  for (int e = 0; e < 16; ++e) acc[1][e] = 0.f;
  const int steps = (K + BK - 1) / BK;
  for (int s = 0; s < STAGES - 1; ++s) fetch(s, s);
  int stage = 0;
  // the sum of a run, from the four pieces of 16 bytes that this lane's row has in it
  auto multiply = [&](const float* base, int run, f32x16& sum) {
    f32x4 xv[2], wv[2];
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      const int at = r * BK + ((run * 4 + g * 2 + h) ^ (r & 7)) * 4;
      xv[g] = *reinterpret_cast<const f32x4*>(base + wm * 32 * BK + at);
      wv[g] = *reinterpret_cast<const f32x4*>(base + (BM + wn * 32) * BK + at);
    }
#pragma unroll
    for (int e = 0; e < 16; ++e) sum[e] = 0.f;
#pragma unroll
    for (int g = 0; g < 2; ++g)
#pragma unroll
      for (int e = 0; e < 4; ++e) sum = __builtin_amdgcn_mfma_f32_32x32x2f32(xv[g][e], wv[g][e], sum, 0, 0, 0);
  };
  auto add = [&](const f32x16& sum) {
#pragma unroll
    for (int e = 0; e < 16; ++e) total[e] += (double)sum[e];
  };
  for (int s = 0; s < steps; ++s) {
    tile_wait<(STAGES - 2) * LOADS>();  // step s is there, and everybody is done with step s - 1
    fetch(s + STAGES - 1, stage == 0 ? STAGES - 1 : stage - 1);
    const float* base = lds + stage * STAGE;
    if constexpr (RUNS == 2) {
      multiply(base, 0, acc[0]);
      add(acc[1]);
      multiply(base, 1, acc[1]);
      add(acc[0]);
    } else {
      multiply(base, ks, acc[0]);
      add(acc[1]);
      acc[1] = acc[0];
    }
    stage = stage == STAGES - 1 ? 0 : stage + 1;
  }
  add(acc[1]);
  tile_wait<0>();

  if constexpr (KS > 1) {  // the waves of a place add up, in their order
    double* const shared = reinterpret_cast<double*>(lds) + (size_t)(wm * WN + wn) * 32 * 32 + lane;
#pragma unroll 1
    for (int s = 1; s < KS; ++s) {
      if (ks == s) {
#pragma unroll
        for (int e = 0; e < 16; ++e) shared[e * WAVE] = total[e];
      }
      __syncthreads();
      if (ks == 0) {
#pragma unroll
        for (int e = 0; e < 16; ++e) total[e] += shared[e * WAVE];
      }
      __syncthreads();
    }
    if (ks != 0) return;
  }
  const int n = n0 + wn * 32 + r;
  if (n >= N) return;
  const float b = bias ? bias[n] : 0.f;
#pragma unroll
  for (int e = 0; e < 16; ++e) {
    const int m = m0 + wm * 32 + 8 * (e / 4) + 4 * h + e % 4;
    if (m < M) c[(size_t)m * ldc + n] = (float)(total[e] + b);
  }
}

template <int WM, int WN, int KS, int STAGES>
static void sgemm_lds_launch(const float* a, long lda, const float* w, const float* bias, float* c, long ldc, int M, int N, int K,
                             hipStream_t stream) {
  const int m_tiles = ceil_div(M, 32 * WM), tiles = m_tiles * ceil_div(N, 32 * WN);
  sgemm_lds_kernel<WM, WN, KS, STAGES><<<8 * ceil_div(tiles, 8), WM * WN * KS * WAVE, 0, stream>>>(a, lda, w, bias, c, ldc, M, N, K, m_tiles, tiles);
}

// The tile shape.  What a compute unit needs for its blocks was measured at K = 4096 (8 to 512 rows of x, 4096 to 32000 of W):
// the first block costs `first` microseconds, every further one `next`, whatever the rows.  Small tiles fill the chip where
// there are few rows, large ones read less from LDS and the caches per product (100 TFLOP/s of 64 x 64, 60 of 16 x 16).
struct SgemmShape {
  int bm, bn;
  float first, next;
};
static const SgemmShape SGEMM_SHAPES[3] = {{16, 16, 22.f, 8.5f}, {32, 64, 67.f, 39.f}, {64, 64, 102.f, 81.f}};
#define SGEMM_COMPUTE_UNITS 256

static int sgemm_shape(int M, int N) {
  int best = 0;
  float least = 0.f;
  for (int i = 0; i < 3; ++i) {
    const SgemmShape& s = SGEMM_SHAPES[i];
    const long blocks = (long)ceil_div(M, s.bm) * ceil_div(N, s.bn);
    const float cost = s.first + s.next * (float)(ceil_div(blocks, SGEMM_COMPUTE_UNITS) - 1);
    if (i == 0 || cost < least) best = i, least = cost;
  }
  return best;
}

// Bound by the matrix unit's float32 rate (154 TFLOP/s for the vendor's product of 8192^3, 100 here; without the conversions and
// additions in float64 the same); with few rows by the weights' bytes.  301 rows, K 4096: 587 us for 22016 rows of W (92
// TFLOP/s; 2450 with one float32 product a thread and instruction, 614 with the rows through registers), 142 for 4096 (152);
// 160 rows: 310 for 22016 (386); 8 rows: 34 us for 12288 rows of W (5.9 TB/s), 22 for 4096.
extern "C" int fmsamd_gemm_f32(const float* a, long lda, const float* w, const float* bias, float* c, long ldc, int M,
                               int N, int K, hipStream_t stream) {
  if (M == 0 || N == 0) return 0;
  FMS_REQUIRE(M > 0 && N > 0 && K > 0, "gemm_f32: bad sizes M=%d N=%d K=%d", M, N, K);
  FMS_REQUIRE(lda >= K && ldc >= N, "gemm_f32: leading dimensions too small");
  FMS_REQUIRE((long)ceil_div(M, 16) * ceil_div(N, 16) <= 0x7ffffff0L, "gemm_f32: M=%d N=%d exceed one launch", M, N);
  const bool aligned = K % 4 == 0 && lda % 4 == 0 && ((uintptr_t)a % 16) == 0 && ((uintptr_t)w % 16) == 0;
  const int shape = sgemm_shape(M, N);
  if (shape == 0) {
    if (aligned)
      sgemm_launch<16, 8, 1, true>(a, lda, w, bias, c, ldc, M, N, K, stream);
    else
      sgemm_launch<16, 8, 1, false>(a, lda, w, bias, c, ldc, M, N, K, stream);
  } else if (!aligned) {
    sgemm_launch<32, 4, 2, false>(a, lda, w, bias, c, ldc, M, N, K, stream);
  } else if (shape == 1) {
    sgemm_lds_launch<1, 2, 2, 3>(a, lda, w, bias, c, ldc, M, N, K, stream);
  } else {
    sgemm_lds_launch<2, 2, 2, 3>(a, lda, w, bias, c, ldc, M, N, K, stream);
  }
  FMS_LAUNCH_CHECK("gemm_f32");
  return 0;
}
