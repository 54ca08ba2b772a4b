// bfloat16 products of many rows, out = x W^T (+ bias) and act(x Wg^T + bg) * (x Wu^T + bu), from the ring of ring_product.h.
//
// 256 blocks, one a compute unit, walk over the tiles.  Of the tiles behind the last whole round every one may be cut into two or four,
// so that the last round is short and full.  A product with rows for one round of smaller tiles takes those.
//
// Measured (the vendor library's product in turn, for the gated one with the activation kernel behind it; microseconds):
//   rows  columns x K       library   here
//   2048  6144 x 4096          82      77
//   2048  4096 x 4096          59      56
//   2048  4096 x 14336        196     181
//   2048  2 x 14336 x 4096    375     337
//   4689  4096 x 4096         141     120
//   4689  4096 x 14336        443     404
//   4689  2 x 14336 x 4096    869     789
//   2277  6176 x 2048 float32  64      56
// 8192 x 8192 x 8192 runs at 1.5 PFLOP/s, in the library at 1.6: either is bound by the chip's power.
#include "fmsamd.h"
#include "gemm_epilogue.h"
#include "ring_product.h"

struct TallArgs {
  const bf16 *x, *w;
  const void* bias;
  int bias_f32;
  void* out;
  long ldx, ldo;  // elements
  int M, N, K;    // N: columns of out
  int row_tiles, col_tiles, group;  // group: row tiles that are walked through together
  int full, split;                  // tiles that are whole; into how many parts the others are cut (1: none are)
  OutAct act;
};

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

// The tiles from `first` to `last`, cut into `parts` parts each (2: rows in halves; 4: columns as well), dealt to the blocks: in every
// round the blocks of one XCD (block % 8) take neighbours, which share rows of x and of W in its L2.  The corner of the n-th part of a
// block, of bm rows and bn columns; false behind the last one.  A part may lie behind the last row or column as a whole.
__host__ __device__ __forceinline__ bool tall_corner(const TallArgs& g, int first, int last, int parts, int bm, int bn, int blocks, int block, int n,
                                                     int& m0, int& n0) {
  const int row_parts = parts > 1 ? 2 : 1, col_parts = parts / row_parts, xcd = block % 8, nth = block / 8, count = (last - first) * parts;
  const int left = count - n * blocks, per = ((left < blocks ? left : blocks) + 7) / 8, in_round = xcd * per + nth;
  if (nth >= per || in_round >= left) return false;
  const int u = n * blocks + in_round;
  const int t = first + u / parts, part = u % parts;
  const int top = t / (g.group * g.col_tiles) * g.group, rows = g.row_tiles - top < g.group ? g.row_tiles - top : g.group;
  const int in = t - top * g.col_tiles;
  m0 = ((top + in % rows) * row_parts + part % row_parts) * bm;
  n0 = ((in / rows) * col_parts + part / row_parts) * bn;
  return true;
}

// How many bytes of out a part of bm rows may store to, from its first result on: to the end of its last row that exists.  What lies
// behind is left out by the store.  None for a part without rows or columns.  (The store takes the number as unsigned: it must not be
// negative, as it would be for one row whose columns all lie behind N.)  Below 2^31, so that TALL_ABSENT lies behind it.
__host__ __device__ __forceinline__ unsigned tall_reach(const TallArgs& g, int m0, int n0, int bm, int size) {
  const int rows = g.M - m0 < bm ? g.M - m0 : bm;
  return rows <= 0 || n0 >= g.N ? 0 : (unsigned)((rows * g.ldo - n0) * size);
}

// Where in there a piece of eight results is stored: of columns that do not exist, behind the reach.
#define TALL_ABSENT 0x80000000u
__host__ __device__ __forceinline__ unsigned tall_offset(const TallArgs& g, int n0, int row, int col, int size) {
  return n0 + col < g.N ? (unsigned)(((long)row * g.ldo + col) * size) : TALL_ABSENT;
}

template <typename R, bool GATED, typename O, int PARTS>
__device__ __forceinline__ void tall_tiles(const TallArgs& g, int first, int last, char* lds) {
  constexpr int BN = GATED ? R::HN : R::BN;
  auto corner = [&](int n, int& m0, int& n0) __attribute__((always_inline)) {
    return tall_corner(g, first, last, PARTS, R::BM, BN, gridDim.x, blockIdx.x, n, m0, n0);
  };
  auto bytes = [](long there, int most, long stride) { return (unsigned)((there < 0 ? 0 : there < most ? there : most) * stride * 2); };
  auto place = [&](int n, RingTile& t) __attribute__((always_inline)) {
    int m0, n0;
    if (!corner(n, m0, n0)) return false;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      t.a[i] = g.x + (long)(m0 + i * R::HM) * g.ldx;
      t.a_bytes[i] = bytes((long)g.M - m0 - i * R::HM, R::HM, g.ldx);
      const long row = GATED ? n0 + (long)i * g.N : n0 + i * R::HN;  // gated: the other half is the "up" rows
      t.w[i] = g.w + row * g.K;
      t.w_bytes[i] = bytes(GATED ? g.N - n0 : (long)g.N - row, R::HN, g.K);
    }
    return true;
  };
  auto finish = [&](int n, auto& sums) __attribute__((always_inline)) {
    // (from a value that the compiler does not know before: registers that hold a lane's place all through the loop would be too many)
    int thread = threadIdx.x;
    asm volatile("" : "+v"(thread));
    const int lane = thread & 63, wave = __builtin_amdgcn_readfirstlane(thread / 64), r = lane & 15, h = lane >> 4;
    const int row0 = (wave / R::WN) * R::QM * 16 + r, col0 = (wave % R::WN) * R::QN * 32 + h * 8;
    int m0, n0;
    corner(n, m0, n0);
    const unsigned reach = tall_reach(g, m0, n0, R::BM, sizeof(O));
    if (reach == 0) return;
    const auto to = __builtin_amdgcn_make_buffer_rsrc((O*)g.out + (long)m0 * g.ldo + n0, 0, (int)reach, 0x00020000);
    auto store = [&](u32x4 v, unsigned offset) __attribute__((always_inline)) { __builtin_amdgcn_raw_buffer_store_b128(v, to, offset, 0, 0); };
    auto write = [&](auto unit) __attribute__((always_inline)) {
      ring_for<(GATED ? 1 : 2) * R::QN>([&](auto bjc) __attribute__((always_inline)) {
        constexpr int b = decltype(bjc)::value / R::QN, j = decltype(bjc)::value % R::QN * 2;
        const int col = col0 + b * R::HN + j * 16;
        float add[8], up[8];
        const bool there = n0 + col < g.N;
        if (g.bias) {
          const int at = there ? n0 + col : 0;
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            add[e] = g.bias_f32 ? ((const float*)g.bias)[at + e] : (float)((const bf16*)g.bias)[at + e];
            if (GATED) up[e] = g.bias_f32 ? ((const float*)g.bias)[g.N + at + e] : (float)((const bf16*)g.bias)[g.N + at + e];
          }
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e) add[e] = up[e] = 0.f;
        }
        ring_for<2 * R::QM>([&](auto aic) __attribute__((always_inline)) {
          constexpr int a = decltype(aic)::value / R::QM, i = decltype(aic)::value % R::QM;
          const int row = row0 + a * R::HM + i * 16;
          const unsigned offset = tall_offset(g, n0, row, col, sizeof(O));
          float v[8];
          const f32x4 lo = sums[R::at(a, b, i, j)], hi = sums[R::at(a, b, i, j + 1)];
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] = (e < 4 ? lo[e % 4] : hi[e % 4]) + add[e];
          if constexpr (GATED) {
            const f32x4 ulo = sums[R::at(a, 1, i, j)], uhi = sums[R::at(a, 1, i, j + 1)];
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = unit(v[e], (e < 4 ? ulo[e % 4] : uhi[e % 4]) + up[e]);
          }
          if constexpr (sizeof(O) == 2) {
            bf16x8 o;
#pragma unroll
            for (int e = 0; e < 8; ++e) o[e] = (bf16)v[e];
            store(__builtin_bit_cast(u32x4, o), offset);
          } else {
            store(__builtin_bit_cast(u32x4, f32x4{v[0], v[1], v[2], v[3]}), offset);
            store(__builtin_bit_cast(u32x4, f32x4{v[4], v[5], v[6], v[7]}), offset + 16);
          }
          __builtin_amdgcn_sched_barrier(0);
        });
      });
    };
    // (a choice for the whole tile: one for every element costs more than the products of a tile.  The fast exponential and the
    // reciprocal are within 7e-6 of the sigmoid wherever it is above 2^-126, the result is rounded to 2^-9; expf and a division take
    // 354 us instead of 342 for 2048 rows by 2 x 14336 of K = 4096, 809 instead of 778 for 4689.)
    if (!GATED || g.act.kind == FMS_ACT_SILU)
      write([&](float gate, float up) { return gate * __builtin_amdgcn_rcpf(1.f + __expf(-gate)) * up; });
    else if (g.act.kind == FMS_ACT_CLAMPED_GATE)
      write([&](float gate, float up) {
        const float z = fminf(gate, g.act.limit), u = fminf(fmaxf(up, -g.act.limit), g.act.limit);
        return z * __builtin_amdgcn_rcpf(1.f + __expf(-g.act.alpha * z)) * (u + g.act.shift);
      });
    else
      write([&](float gate, float up) { return sk_gated(gate, up, g.act); });
  };
  ring_product<R>((unsigned)(g.ldx * 2), (unsigned)(g.K * 2), g.K, lds, place, finish);
}

// R: the whole tiles.
template <typename R, bool GATED, typename O>
__global__ void __launch_bounds__(R::THREADS) tall_kernel(TallArgs g) {
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  const int tiles = g.row_tiles * g.col_tiles;
  tall_tiles<R, GATED, O, 1>(g, 0, g.full, lds);
  if constexpr (R::BM == 256 && R::BN == 256) {
    if (g.split == 2) tall_tiles<Ring<2, 4, 2, 1>, GATED, O, 2>(g, g.full, tiles, lds);
    if (g.split == 4) tall_tiles<Ring<4, 2, 1, 1>, GATED, O, 4>(g, g.full, tiles, lds);
  }
}

typedef Ring<2, 4, 4, 1> TallSquare;  // 256 x 256
template <bool GATED> using TallMiddle = std::conditional_t<GATED, Ring<8, 1, 1, 3>, Ring<4, 1, 2, 3>>;
typedef Ring<2, 2, 4, 1> TallNarrow;  // 256 x 128

#define TALL_COMPUTE_UNITS 256
#define TALL_LONGEST (1 << 22)  // a row's elements, or bytes of out: offsets inside a tile are 32-bit

static bool tall_countable(int M, int N) { return (long)ceil_div(M, 256) * ceil_div(2L * N, 128) < (1 << 24); }

// Which tiles a product is cut into, and about how long it takes.
struct TallPlan {
  int shape, split;  // 0 square, 1 middle, 2 narrow; parts of the tiles behind the last whole round of square ones
  double us;
};

// A round of tiles, one a compute unit: microseconds a step of 64 k-values with few tiles (the rest of the chip idle) and what a full
// chip adds (less power for each), and what begins and ends a tile.  Measured over 192 to 4689 rows, 784 to 32064 columns, K = 256 to
// 14336.  Square tiles move the fewest bytes a product: two of 128 x 256 take 1.25 times as long as one of 256 x 256.
static double tall_rounds(long tiles, int steps, double few, double more, double ends) {
  const double last = (double)(tiles % TALL_COMPUTE_UNITS) / TALL_COMPUTE_UNITS;
  return (double)(tiles / TALL_COMPUTE_UNITS) * (steps * (few + more) + ends) + (last > 0 ? steps * (few + more * last) + ends : 0);
}

static TallPlan tall_plan(int M, int N, int K, bool gated) {
  const int wide = gated ? 2 : 1, steps = K / 64;
  auto tiles = [&](int bm, int bn) { return (long)ceil_div(M, bm) * ceil_div((long)N * wide, bn); };
  const long square = tiles(256, 256), whole = square / TALL_COMPUTE_UNITS * TALL_COMPUTE_UNITS, rest = square - whole;
  const TallPlan plans[5] = {
      {0, 1, tall_rounds(square, steps, 1.10, 0.32, 7)},
      {0, 2, tall_rounds(whole, steps, 1.10, 0.32, 7) + tall_rounds(2 * rest, steps, 0.74, 0.18, 4)},
      {0, 4, tall_rounds(whole, steps, 1.10, 0.32, 7) + tall_rounds(4 * rest, steps, whole ? 0.45 : 0.53, 0.08, 3)},
      {1, 1, tall_rounds(tiles(256, 192), steps, gated ? 0.93 : 0.89, gated ? 0.30 : 0.27, 6)},
      {2, 1, tall_rounds(tiles(256, 128), steps, 0.72, 0.12, 4)},
  };
  int best = 0;
  for (int i = 1; i < 5; ++i)
    if (plans[i].us < plans[best].us) best = i;
  return plans[best];
}

// Which tiles: 0 to 2 256 x 256 (the last ones whole, halved, quartered), 3 256 x 192, 4 256 x 128.
extern "C" int fmsamd_gemm_tall_plan(int M, int N, int K, int gated) {
  const TallPlan plan = tall_plan(M, N, K, gated != 0);
  return plan.shape ? plan.shape + 2 : plan.split / 2;
}

// Whether a product is better here than in the vendor library, which cuts K where rows and columns give few tiles: from the share of
// the chip that the tiles here use.  Of shapes timed in turn, 512 rows by 4096 columns of K = 2048 are equal (16 us, a share of 0.31), 1024
// by 4096 of K = 4096 too (39 us, 0.56), and of K = 14336 3000 rows lose (292 us, library 249; 0.77) where 2048 win (181, 196; 0.84).  A
// gated product saves the kernel behind it and its bytes as well: half of the share will do.
//
// The products of every registered configuration at 33 numbers of rows from 193 to 4689, between a kernel that writes x and one that
// reads the results: of 1556 that are taken 960 are more than 3 % faster here and 245 slower, 7.7 % faster on average.  The slower ones are
// whole squares of bfloat16 results with many rows (3000 x 4096 x 4096 84, library 76; K = 5120 and 128256 columns are 4 to 18 % faster
// here: equal on average) and 256 x 128 tiles with a share below 0.55 (5 % slower on average).  Leaving the first to the library
// makes a pass of 8 layers of 4096 wide 0.3 % slower to 1.3 % faster (2277 to 4096 rows), the second one of 2048 wide 1.0 % slower to
// 0.5 % faster (512 to 1280 rows): the kernels behind read the library's results more slowly.  So there is no line for them.
extern "C" int fmsamd_gemm_tall_pays(int M, int N, int K, int gated) {
  if (M <= FMS_SKINNY_MAX_ROWS || N < 128 || K < 256 || N % 8 || K % 128 || K >= TALL_LONGEST || !tall_countable(M, N)) return 0;
  const double ideal = (double)M * N * (gated ? 2 : 1) / (256. * 256 * TALL_COMPUTE_UNITS) * (K / 64) * 1.36;
  const double share = K < 1280 ? 0.1875 : K > 5051 ? 0.74 : 0.15 * K / 1024;
  return ideal >= tall_plan(M, N, K, gated != 0).us * share * (gated ? 0.5 : 1.0);
}

// The tiles, of bm rows and bn columns, that a product is cut into, and how many of them stay whole.
static int tall_cut(TallArgs& g, int bm, int bn, int split) {
  g.row_tiles = ceil_div(g.M, bm);
  g.col_tiles = ceil_div(g.N, bn);
  g.group = ceil_div(g.row_tiles, ceil_div(g.row_tiles, 8));
  const int tiles = g.row_tiles * g.col_tiles, units = TALL_COMPUTE_UNITS;
  g.split = split;
  g.full = split == 1 ? tiles : tiles / units * units;
  const long parts = (long)tiles * split;
  return parts < units ? ((int)parts + 7) / 8 * 8 : units;  // blocks
}

template <typename R, bool GATED, typename O>
static int tall_launch(TallArgs g, int split, hipStream_t stream) {
  const int blocks = tall_cut(g, R::BM, GATED ? R::HN : R::BN, split);
  auto kernel = tall_kernel<R, GATED, O>;
  // more than 64 KB of LDS a block has to be asked for, once a kernel
  static const hipError_t sized = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, R::LDS_BYTES);
  FMS_REQUIRE(sized == hipSuccess, "gemm_tall: %d bytes of LDS refused: %s", R::LDS_BYTES, hipGetErrorString(sized));
  kernel<<<blocks, R::THREADS, R::LDS_BYTES, stream>>>(g);
  FMS_LAUNCH_CHECK("gemm_tall");
  return 0;
}

template <bool GATED, typename O>
static int tall_choose(const TallArgs& g, hipStream_t stream) {
  const TallPlan plan = tall_plan(g.M, g.N, g.K, GATED);
  if (plan.shape == 1) return tall_launch<TallMiddle<GATED>, GATED, O>(g, 1, stream);
  if (plan.shape == 2) return tall_launch<TallNarrow, GATED, O>(g, 1, stream);
  return tall_launch<TallSquare, GATED, O>(g, plan.split, stream);
}

static int tall_check(const char* name, const TallArgs& g, int size) {
  FMS_REQUIRE(g.M > 0 && g.N > 0 && g.K >= 256 && g.K % 128 == 0 && g.N % 8 == 0,
              "%s: bad sizes M=%d N=%d K=%d (N a multiple of 8, K one of 128 and at least 256)", name, g.M, g.N, g.K);
  FMS_REQUIRE(g.ldx >= g.K && g.ldo >= g.N && g.ldx % 8 == 0 && g.ldo * size % 16 == 0, "%s: row strides %ld and %ld", name, g.ldx, g.ldo);
  FMS_REQUIRE(!((uintptr_t)g.x % 16 || (uintptr_t)g.w % 16 || (uintptr_t)g.out % 16), "%s: x, W and out start at 16-byte addresses", name);
  // (of a store the upper half of the offsets lies outside)
  FMS_REQUIRE(g.ldx < TALL_LONGEST && g.K < TALL_LONGEST && g.ldo * size < TALL_LONGEST, "%s: rows are too long (%ld, %d, %ld)", name, g.ldx, g.K,
              g.ldo);
  FMS_REQUIRE(tall_countable(g.M, g.N), "%s: too many tiles (M=%d N=%d)", name, g.M, g.N);
  return 0;
}

// out [M, N] = x W^T (+ bias), bfloat16 or float32.
extern "C" int fmsamd_gemm_tall_bf16(const void* x, long ldx, const void* w, const void* bias, int bias_dtype, void* out, int out_dtype, long ldo,
                                     int M, int N, int K, hipStream_t stream) {
  if (M == 0 || N == 0) return 0;
  FMS_REQUIRE(out_dtype == FMS_BF16 || out_dtype == FMS_F32, "gemm_tall_bf16: unknown output dtype %d", out_dtype);
  const TallArgs g{(const bf16*)x, (const bf16*)w, bias, bias_dtype == FMS_F32, out, ldx, ldo, M, N, K, 0, 0, 0, 0, 0, plain_act(FMS_ACT_IDENTITY)};
  if (tall_check("gemm_tall_bf16", g, out_dtype == FMS_F32 ? 4 : 2)) return -1;
  return out_dtype == FMS_F32 ? tall_choose<false, float>(g, stream) : tall_choose<false, bf16>(g, stream);
}

// out [M, hidden] = act(x Wg^T + bg) * (x Wu^T + bu) or the clamped unit of the two, W and bias stacked as [gate; up].
extern "C" int fmsamd_gemm_tall_gated_bf16(const void* x, long ldx, const void* w, const void* bias, int bias_dtype, void* out, long ldo, int M,
                                           int hidden, int K, int act, const fmsamd_gate_clamp* clamp, hipStream_t stream) {
  if (M == 0 || hidden == 0) return 0;
  FMS_REQUIRE(act >= FMS_ACT_SILU && act <= FMS_ACT_LAST, "gemm_tall_gated_bf16: unknown activation %d", act);
  FMS_REQUIRE(clamp == nullptr || clamp->limit > 0.f, "gemm_tall_gated_bf16: a limit of %g", (double)clamp->limit);
  const OutAct unit = clamp ? OutAct{FMS_ACT_CLAMPED_GATE, clamp->limit, clamp->alpha, clamp->shift} : plain_act(act);
  const TallArgs g{(const bf16*)x, (const bf16*)w, bias, bias_dtype == FMS_F32, out, ldx, ldo, M, hidden, K, 0, 0, 0, 0, 0, unit};
  if (tall_check("gemm_tall_gated_bf16", g, 2)) return -1;
  return tall_choose<true, bf16>(g, stream);
}

// How many pieces of eight results a product of this kind of tiles (as fmsamd_gemm_tall_plan names them) stores, walked through on the host
// with what the kernels compute their stores from: M N / 8.  -1: one would lie outside its row, behind the last row or behind its part's reach.
extern "C" long fmsamd_gemm_tall_stores(int M, int N, long ldo, int size, int gated, int tiles) {
  TallArgs g{};
  g.M = M, g.N = N, g.ldo = ldo;
  const int split = tiles == 1 ? 2 : tiles == 2 ? 4 : 1, bn = (tiles < 3 ? 256 : tiles == 3 ? 192 : 128) / (gated ? 2 : 1);
  const int blocks = tall_cut(g, 256, bn, split);
  long stored = 0;
  for (int rest = 0; rest < 2; ++rest) {  // the whole tiles, and the parts of the others
    const int first = rest ? g.full : 0, last = rest ? g.row_tiles * g.col_tiles : g.full, parts = rest ? split : 1;
    const int part_rows = parts > 1 ? 128 : 256, part_cols = parts == 4 ? bn / 2 : bn;
    for (int block = 0; block < blocks; ++block) {
      int m0, n0;
      for (int n = 0; tall_corner(g, first, last, parts, part_rows, part_cols, blocks, block, n, m0, n0); ++n) {
        const unsigned reach = tall_reach(g, m0, n0, part_rows, size);
        if (reach > TALL_ABSENT) return -1;
        for (int row = 0; row < part_rows; ++row)
          for (int col = 0; col < part_cols; col += 8) {
            const unsigned offset = tall_offset(g, n0, row, col, size);
            if (offset >= reach) continue;
            if (m0 + row >= M || n0 + col + 8 > N || offset + 8u * size > reach) return -1;
            ++stored;
          }
      }
    }
  }
  return stored;
}
