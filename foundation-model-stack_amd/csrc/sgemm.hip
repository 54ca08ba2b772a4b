// The true 32-bit product y = x W^T (+ bias): float32 rows of x and W (K contiguous), float32 result.
//
// Sums of 16 products each in float32, added up in float64: what a long K costs is the rounding of short sums, not of
// every partial sum on the way.  The products and the short sums are the matrix unit's (mfma 32x32x2 and 16x16x4, float32
// throughout), the sums over the runs the vector unit's, side by side.
#include "common.h"
#include "fmsamd.h"

typedef double f64x4 __attribute__((ext_vector_type(4)));

#define SG_RUN 16  // products of a float32 sum

// A block's tile is TILE * WM * RM rows of x by TILE * WN * RN rows of W; its WM x WN x KS waves have RM x RN tiles each, the
// KS waves of a place share K: of a step's SG_RUN * RUNS * KS k-values each takes SG_RUN * RUNS.  The step's rows wait in
// LDS while the next step's are on their way from memory in registers.  Rows of LDS are padded by four floats: the 16-byte
// reads of eight neighbouring rows then cover all banks.
template <int TILE, int WM, int WN, int RM, int RN, int KS, int RUNS, bool VEC>
__global__ void __launch_bounds__(WM* WN* KS* WAVE)
    sgemm_kernel(const float* __restrict__ a, long lda, const float* __restrict__ w, const float* __restrict__ bias,
                 float* __restrict__ c, long ldc, int M, int N, int K, int m_tiles, int tiles) {
  constexpr int THREADS = WM * WN * KS * WAVE;
  constexpr int BM = TILE * WM * RM, BN = TILE * WN * RN, BK = SG_RUN * RUNS * KS, LD = BK + 4;
  constexpr int PIECES = (BM + BN) * (BK / 4);  // of 16 bytes a step
  constexpr int LOADS = (PIECES + THREADS - 1) / THREADS;
  constexpr int ACC = TILE * TILE / WAVE;
  typedef float accv __attribute__((ext_vector_type(ACC)));
  constexpr int REDUCE_BYTES = KS > 1 ? WM * WN * RM * RN * TILE * TILE * 8 : 0;
  constexpr int STEP_BYTES = 2 * (BM + BN) * LD * 4;
  __shared__ __attribute__((aligned(16))) unsigned char lds[STEP_BYTES > REDUCE_BYTES ? STEP_BYTES : REDUCE_BYTES];
  float* const steps = reinterpret_cast<float*>(lds);

  // The tiles of x that share a tile of W follow one another on one of the eight dies (blocks are dealt to the dies in
  // turn), so that W comes from memory once.
  const int per_die = (tiles + 7) / 8;
  const int tile = (blockIdx.x & 7) * per_die + (blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per_die || tile >= tiles) return;
  const int m0 = (tile % m_tiles) * BM, n0 = (tile / m_tiles) * BN;

  const int lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x / WAVE;
  const int ks = wave / (WM * WN), wm = (wave / WN) % WM, wn = wave % WN;
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

  double total[RM][RN][ACC];
#pragma unroll
  for (int i = 0; i < RM; ++i)
#pragma unroll
    for (int j = 0; j < RN; ++j)
#pragma unroll
      for (int e = 0; e < ACC; ++e) total[i][j][e] = 0.0;

  fetch(0);
  put(0);
  __syncthreads();
  int buffer = 0;
  for (int k0 = 0; k0 < K; k0 += BK, buffer ^= 1) {
    const bool more = k0 + BK < K;
    if (more) fetch(k0 + BK);
    const float* sx = steps + buffer * (BM + BN) * LD + (wm * RM * TILE + r) * LD + ks * SG_RUN * RUNS + kq * 4;
    const float* sw = steps + buffer * (BM + BN) * LD + (BM + wn * RN * TILE + r) * LD + ks * SG_RUN * RUNS + kq * 4;
    constexpr int GROUP = 4 * (WAVE / TILE);  // k-values of one 16-byte piece a lane
#pragma unroll
    for (int run = 0; run < RUNS; ++run) {
      accv acc[RM][RN];
#pragma unroll
      for (int i = 0; i < RM; ++i)
#pragma unroll
        for (int j = 0; j < RN; ++j)
#pragma unroll
          for (int e = 0; e < ACC; ++e) acc[i][j][e] = 0.f;
#pragma unroll
      for (int g = 0; g < SG_RUN / GROUP; ++g) {
        f32x4 xv[RM], wv[RN];
#pragma unroll
        for (int i = 0; i < RM; ++i) xv[i] = *reinterpret_cast<const f32x4*>(sx + i * TILE * LD + run * SG_RUN + g * GROUP);
#pragma unroll
        for (int j = 0; j < RN; ++j) wv[j] = *reinterpret_cast<const f32x4*>(sw + j * TILE * LD + run * SG_RUN + g * GROUP);
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int i = 0; i < RM; ++i)
#pragma unroll
            for (int j = 0; j < RN; ++j) {
              if constexpr (TILE == 32)
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(xv[i][e], wv[j][e], acc[i][j], 0, 0, 0);
              else
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(xv[i][e], wv[j][e], acc[i][j], 0, 0, 0);
            }
      }
#pragma unroll
      for (int i = 0; i < RM; ++i)
#pragma unroll
        for (int j = 0; j < RN; ++j)
#pragma unroll
          for (int e = 0; e < ACC; ++e) total[i][j][e] += (double)acc[i][j][e];
    }
    if (more) put(buffer ^ 1);
    __syncthreads();
  }

  if constexpr (KS > 1) {  // the waves of a place add up, in their order
    double* const shared = reinterpret_cast<double*>(lds) + (size_t)(wm * WN + wn) * RM * RN * TILE * TILE + lane;
#pragma unroll 1
    for (int s = 1; s < KS; ++s) {
      if (ks == s) {
#pragma unroll
        for (int i = 0; i < RM; ++i)
#pragma unroll
          for (int j = 0; j < RN; ++j)
#pragma unroll
            for (int e = 0; e < ACC; ++e) shared[((i * RN + j) * ACC + e) * WAVE] = total[i][j][e];
      }
      __syncthreads();
      if (ks == 0) {
#pragma unroll
        for (int i = 0; i < RM; ++i)
#pragma unroll
          for (int j = 0; j < RN; ++j)
#pragma unroll
            for (int e = 0; e < ACC; ++e) total[i][j][e] += shared[((i * RN + j) * ACC + e) * WAVE];
      }
      __syncthreads();
    }
    if (ks != 0) return;
  }
#pragma unroll
  for (int j = 0; j < RN; ++j) {
    const int n = n0 + (wn * RN + j) * TILE + r;
    if (n >= N) continue;
    const float b = bias ? bias[n] : 0.f;
#pragma unroll
    for (int i = 0; i < RM; ++i)
#pragma unroll
      for (int e = 0; e < ACC; ++e) {
        // the matrix unit's result: column lane % TILE, rows in groups of four
        const int row = TILE == 32 ? 8 * (e / 4) + 4 * kq + e % 4 : 4 * kq + e;
        const int m = m0 + (wm * RM + i) * TILE + row;
        if (m < M) c[(size_t)m * ldc + n] = (float)(total[i][j][e] + b);
      }
  }
}

template <int TILE, int WM, int WN, int RM, int RN, int KS, int RUNS>
static void sgemm_launch(const float* a, long lda, const float* w, const float* bias, float* c, long ldc, int M, int N, int K,
                         hipStream_t stream) {
  constexpr int BM = TILE * WM * RM, BN = TILE * WN * RN;
  const int m_tiles = ceil_div(M, BM), tiles = m_tiles * ceil_div(N, BN);
  const bool vec = K % 4 == 0 && lda % 4 == 0 && ((uintptr_t)a % 16) == 0 && ((uintptr_t)w % 16) == 0;
  const int blocks = 8 * ceil_div(tiles, 8);
  if (vec)
    sgemm_kernel<TILE, WM, WN, RM, RN, KS, RUNS, true><<<blocks, WM * WN * KS * WAVE, 0, stream>>>(a, lda, w, bias, c, ldc, M, N, K, m_tiles, tiles);
  else
    sgemm_kernel<TILE, WM, WN, RM, RN, KS, RUNS, false><<<blocks, WM * WN * KS * WAVE, 0, stream>>>(a, lda, w, bias, c, ldc, M, N, K, m_tiles, tiles);
}

// The tile shape.  What a compute unit needs for its blocks was measured at K = 4096 (7 to 500 rows of x, 4096 to 32000 of W):
// the first block costs `first` microseconds, every further one `next`, whatever the rows.  Small tiles fill the chip where
// there are few rows, large ones read less from LDS and the caches per product (97 TFLOP/s of 64 x 64, 72 of 32 x 32).
struct SgemmShape {
  int bm, bn;
  float first, next;
};
static const SgemmShape SGEMM_SHAPES[4] = {{16, 16, 22.f, 8.5f}, {32, 32, 41.f, 30.f}, {32, 64, 73.f, 45.f}, {64, 64, 126.f, 82.f}};
#define SGEMM_COMPUTE_UNITS 256

static int sgemm_shape(int M, int N) {
  int best = 0;
  float least = 0.f;
  for (int i = 0; i < 4; ++i) {
    const SgemmShape& s = SGEMM_SHAPES[i];
    const long blocks = (long)ceil_div(M, s.bm) * ceil_div(N, s.bn);
    const float cost = s.first + s.next * (float)(ceil_div(blocks, SGEMM_COMPUTE_UNITS) - 1);
    if (i == 0 || cost < least) best = i, least = cost;
  }
  return best;
}

// Bound by the matrix unit's float32 rate (154 TFLOP/s for the vendor's product of 8192^3) and, in its shadow, the vector
// unit's conversions and additions in float64; with few rows by the weights' bytes.  301 rows, K 4096: 614 us for 22016 rows of
// W (88 TFLOP/s; 2450 with one float32 product a thread and instruction), 154 for 4096; 8 rows: 34 us for 12288 rows of W
// (5.9 TB/s), 22 for 4096.
extern "C" int fmsamd_gemm_f32(const float* a, long lda, const float* w, const float* bias, float* c, long ldc, int M,
                               int N, int K, hipStream_t stream) {
  if (M == 0 || N == 0) return 0;
  FMS_REQUIRE(M > 0 && N > 0 && K > 0, "gemm_f32: bad sizes M=%d N=%d K=%d", M, N, K);
  FMS_REQUIRE(lda >= K && ldc >= N, "gemm_f32: leading dimensions too small");
  FMS_REQUIRE((long)ceil_div(M, 16) * ceil_div(N, 16) <= 0x7ffffff0L, "gemm_f32: M=%d N=%d exceed one launch", M, N);
  switch (sgemm_shape(M, N)) {
    case 0: sgemm_launch<16, 1, 1, 1, 1, 8, 1>(a, lda, w, bias, c, ldc, M, N, K, stream); break;
    case 1: sgemm_launch<32, 1, 1, 1, 1, 4, 2>(a, lda, w, bias, c, ldc, M, N, K, stream); break;
    case 2: sgemm_launch<32, 1, 2, 1, 1, 2, 2>(a, lda, w, bias, c, ldc, M, N, K, stream); break;
    default: sgemm_launch<32, 2, 2, 1, 1, 1, 2>(a, lda, w, bias, c, ldc, M, N, K, stream); break;
  }
  FMS_LAUNCH_CHECK("gemm_f32");
  return 0;
}
