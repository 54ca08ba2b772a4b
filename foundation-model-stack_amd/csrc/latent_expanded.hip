// Attention over a latent cache for prompts, with keys and values expanded for the step.
//
// latent_attention.hip never forms keys or values: it takes every query into the latent space, where a pair of query and key
// costs 2 R + P products a head (R the latent, P the shared key part).  With the head's own keys [Uk_h c | shared part] and values
// Uv_h c a pair costs D + P + V, 3.4 times less for R = 512 and heads of 128 + 64, and the queries and results need no product of
// their own on the way in and out of the latent space.  What it costs is one product of every cached row with Uk and Uv and room
// for its result, so it is for steps that bring most of the tokens that they look at.
//
//   latent_expand:  keys [seq][page][H][token][D] and values, transposed, [seq][page][H][V][token] of every row that the
//                   step's tokens look at (with a window from the pair of pages on that the sequence's first token of the step sees);
//                   rows behind a sequence's last token are zeros, up to an even number of pages
//   latent_prompt:  causal softmax attention over them: rotation of the queries on the way in, the gate on the way out
#include "common.h"
#include "fmsamd.h"
#include "tile_product_lds.h"

#define LX_STEP 128  // keys of a step: two pages

struct ExpandArgs {
  const bf16* cache;  // [page][64][width]
  long width;
  const bf16 *uk, *uv;  // [H * D, R], [H * V, R]
  bf16 *keys, *values;
  const int *positions, *seq_starts, *block_table;
  int table_stride, pages, H, D, V, R, window;
};

// The first pair of pages that a sequence's tokens of the step look at, which its room begins with.
__device__ __forceinline__ int first_pair(int first_position, int window) {
  return window > 0 && first_position - window + 1 > 0 ? (first_position - window + 1) / LX_STEP : 0;
}

// A block: 128 tokens (two pages) by 128 columns of Uk, or 128 rows of Uv by 128 tokens, so that either result is written in runs
// of 64 bytes.  K is the latent's size, eight steps for R = 512, so a block is mostly its first loads and its stores and two of them
// share a compute unit (one with twice the steps under way: 20 us instead of 16; blocks of 256 columns 16, and 12 instead of 9 for a
// single block of tokens).  16 heads of 128: 9.5 us for 32 rows, 12 for 1000, 16 for 2048 (4.3e9 multiply-adds, 17 MB written).
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) latent_expand_kernel(ExpandArgs a) {
  constexpr int COLS = 128;
  typedef TileLds<2, 2, 2, 2, 2> S;
  __shared__ __attribute__((aligned(16))) bf16 lds[S::LDS_ELEMENTS];
  const int col_tiles = (a.H * a.D + COLS - 1) / COLS;
  const int seq = blockIdx.x / (a.pages / 2), pair = blockIdx.x % (a.pages / 2);
  const bool of_keys = (int)blockIdx.y < col_tiles;
  const int n0 = ((int)blockIdx.y - (of_keys ? 0 : col_tiles)) * COLS;
  const int begin = uniform_load(a.seq_starts + seq), last = uniform_load(a.seq_starts + seq + 1) - 1;
  if (last < begin) return;  // uniform
  const int context = uniform_load(a.positions + last) + 1;
  const int of_sequence = first_pair(uniform_load(a.positions + begin), a.window) + pair, first = of_sequence * LX_STEP;
  if (first >= context) return;  // uniform
  const int* bt = a.block_table + (size_t)seq * a.table_stride + 2 * of_sequence;
  const size_t page0 = readable_page(bt[0]), page1 = readable_page(bt[first + PAGE_TOKENS < context ? 1 : 0]);
  auto token_row = [&](int i) { return a.cache + ((i < PAGE_TOKENS ? page0 : page1) * PAGE_TOKENS + i % PAGE_TOKENS) * a.width; };
  const int rows = a.H * (of_keys ? a.D : a.V);
  const bf16* const w = of_keys ? a.uk : a.uv;
  auto weight_row = [&](int n) { return w + (size_t)(n0 + n < rows ? n0 + n : 0) * a.R; };
  f32x16 acc[2][2];
  if (of_keys)
    tile_product_lds<2, 2, 2, 2, 2>(token_row, weight_row, a.R, lds, acc);
  else
    tile_product_lds<2, 2, 2, 2, 2>(weight_row, token_row, a.R, lds, acc);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r0 = (wave >> 1) * 64 + 4 * (lane >> 5), c0 = (wave & 1) * 64 + (lane & 31);
  const size_t slot = (size_t)seq * a.pages + 2 * pair;
  // (a row or column of 128 tokens lies in one page in runs of 64: a wave's tiles are on one side)
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int c = c0 + j * 32;
    if (of_keys) {
      const int n = n0 + c;
      if (n >= rows) continue;
      const int left = context - first - r0;  // of this lane's first row
      bf16* const to = a.keys + (((slot + r0 / PAGE_TOKENS) * a.H + n / a.D) * PAGE_TOKENS + r0 % PAGE_TOKENS) * a.D + n % a.D;
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int at = i * 32 + 8 * (e / 4) + e % 4;
          to[at * a.D] = at < left ? (bf16)acc[i][j][e] : (bf16)0.f;
        }
    } else {
      bf16* const to = a.values + ((slot + c / PAGE_TOKENS) * a.H * a.V + n0 + r0) * PAGE_TOKENS + c % PAGE_TOKENS;
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int at = i * 32 + 8 * (e / 4) + e % 4;
          if (n0 + r0 + at < rows) to[at * PAGE_TOKENS] = first + c < context ? (bf16)acc[i][j][e] : (bf16)0.f;
        }
    }
  }
}

struct PromptArgs {
  const bf16* q;  // [T, ldq]: head h's D + P elements at h (D + P), not rotated
  long ldq;
  bf16* out;  // [T, ldo]: head h's V elements at h V
  long ldo;
  const bf16 *keys, *values, *cache;
  const int *positions, *seq_of_token, *seq_starts, *qblock_start, *qblock_len, *block_table;
  const float *cos_t, *sin_t, *sink, *gate;  // gate: logits [T, ldg] or null
  long ldg;
  int n_qblocks, table_stride, pages, H, rank, window;
  float scale2;  // times log2(e)
};

// (fmaxf and not inline assembly: the compiler forms v_max3_f32, behind the wait between a matrix instruction and the first read of its
// result, which it does not put in front of assembly)
__device__ __forceinline__ float max3(float a, float b, float c) { return fmaxf(fmaxf(a, b), c); }

// Scores S^T = K Q^T of 32 keys by 32 queries, O^T += V^T P^T, both 32x32x16: the lane layout is that of the prompts' attention with
// head sizes up to 128 (attention.hip).  A block is 64 queries of one head and walks 128 keys a step: two runs of 32 queries by four
// runs of 32 keys, whose waves meet at the end.  (Blocks of 128 queries by 64 keys, three pages ahead in LDS: 15 us for 300 tokens, 29 for
// 1000, 51 for 2048, 385 for 8192: with one sequence the longest block, of twice as many steps, is what the kernel takes.)  The
// longest blocks go first; the heads follow one another on the dies (blocks are dealt to them in turn), so that a head's keys stay in one L2.
// 16 heads of 128 + 64: 8 us for 32 tokens, 12 for 300, 22 for 1000, 46 for 2048, 456 for 8192; in the latent space 10, 62, 134 and 1751, with 17 to
// 55 us more for the products into the latent space and out of it.
// Keys, shared parts and values go from memory straight into LDS, one step ahead: 80 KB a step for 128 + 64 and 128, twice, is all of a
// compute unit's LDS.  Their pieces of 16 bytes are XOR-swizzled with the row, so that the operand reads of 16 neighbouring rows cover
// all 64 banks (with 8 of them 48 us for 2048 tokens and 476 for 8192).
// NC, RC: pieces of 16 of a key's own and shared part; DT: tiles of 32 value elements.
template <int NC, int RC, int DT>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) latent_prompt_kernel(PromptArgs a) {
  constexpr int D = NC * 16, P = RC * 16, V = DT * 32;
  constexpr int KN_BYTES = LX_STEP * D * 2, KR_BYTES = LX_STEP * P * 2, V_BYTES = V * LX_STEP * 2, STAGE = KN_BYTES + KR_BYTES + V_BYTES;
  constexpr int KN_LOADS = KN_BYTES / 8192, KR_LOADS = KR_BYTES / 8192, V_LOADS = V_BYTES / 8192;  // of 1 KB, a wave
  constexpr int KN_PIECES = D / 8, KR_PIECES = P > 0 ? P / 8 : 8;
  static_assert(KN_BYTES % 8192 == 0 && KR_BYTES % 8192 == 0 && V_BYTES % 8192 == 0, "whole loads");
  static_assert((KN_PIECES == 16 || KN_PIECES == 8) && KR_PIECES == 8 && 64 % KN_PIECES == 0 && 64 % KR_PIECES == 0, "whole groups of pieces, whole rows a load");
  static_assert(2 * STAGE <= 160 * 1024 && 6 * (DT * 16 + 2) * 256 <= 2 * STAGE, "a compute unit's LDS; the waves meet in it");
  extern __shared__ __attribute__((aligned(16))) unsigned char lx_lds[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int j = lane & 31, hb = lane >> 5;
  const int unit = wave & 1, quarter = wave >> 1;  // which 32 queries, which 32 keys of a step
  const int qb = a.n_qblocks - 1 - (int)(blockIdx.x / a.H), h = blockIdx.x % a.H;
  const int t_begin = uniform_load(a.qblock_start + qb), t_end = t_begin + uniform_load(a.qblock_len + qb);
  const int seq = uniform_load(a.seq_of_token + t_begin);
  if (seq < 0) return;  // whole block
  const int* bt = a.block_table + (size_t)seq * a.table_stride;
  const int t0 = t_begin + unit * 32, t = t0 + j;
  const bool has_work = t0 < t_end, valid = t < t_end;
  const int blk_first = uniform_load(a.positions + t_begin), blk_last = uniform_load(a.positions + t_end - 1);

  bf16x8 q[NC + RC];
  const int pos = valid ? a.positions[t] : -1;
  {
    const bf16* row = a.q + (size_t)(valid ? t : t_begin) * a.ldq + (size_t)h * (D + P) + hb * 8;
#pragma unroll
    for (int c = 0; c < NC + RC; ++c) q[c] = *reinterpret_cast<const bf16x8*>(row + c * 16);
    const size_t angle = (size_t)(valid ? pos : blk_first) * (P / 2) + hb * 4;
#pragma unroll
    for (int c = 0; c < RC; ++c) {
      const f32x4 cs = *reinterpret_cast<const f32x4*>(a.cos_t + angle + c * 8), sn = *reinterpret_cast<const f32x4*>(a.sin_t + angle + c * 8);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float u = (float)q[NC + c][2 * e], w = (float)q[NC + c][2 * e + 1];
        q[NC + c][2 * e] = (bf16)(u * cs[e] - w * sn[e]);
        q[NC + c][2 * e + 1] = (bf16)(w * cs[e] + u * sn[e]);
      }
    }
  }
  auto lowest = [&](int p) { return a.window > 0 && p - a.window + 1 > 0 ? p - a.window + 1 : 0; };
  const int lo = lowest(pos);
  int wave_hi = -1, wave_lo = 0, full_hi = -1, full_lo = 0;  // keys that some, that all queries of the wave see
  if (has_work) {
    wave_hi = uniform_load(a.positions + (t0 + 32 < t_end ? t0 + 32 : t_end) - 1), full_hi = uniform_load(a.positions + t0);
    wave_lo = lowest(full_hi), full_lo = lowest(wave_hi);
  }

  // what this lane loads: which row of a load's and which piece of it
  // (rows of 256 bytes by their number, rows of 128 by half of it: sixteen neighbouring rows then cover all 64 banks)
  auto swizzle = [](int row, int pieces) { return pieces == 16 ? row & 15 : (row >> 1) & 7; };
  const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)lx_lds;
  const size_t page_keys = (size_t)a.H * PAGE_TOKENS * D, page_values = (size_t)a.H * V * PAGE_TOKENS;
  const int half = wave >> 2;  // the page of the two whose keys this wave loads
  unsigned kn_from[KN_LOADS], kr_from[RC > 0 ? KR_LOADS : 1], v_from[V_LOADS];
#pragma unroll
  for (int n = 0; n < KN_LOADS; ++n) {
    const int key = (wave * KN_LOADS + n) * (64 / KN_PIECES) + lane / KN_PIECES;
    kn_from[n] = ((key & 63) * D + ((lane % KN_PIECES) ^ swizzle(key, KN_PIECES)) * 8) * 2;
  }
#pragma unroll
  for (int n = 0; n < (RC > 0 ? KR_LOADS : 0); ++n) {
    const int key = (wave * KR_LOADS + n) * (64 / KR_PIECES) + lane / KR_PIECES;
    kr_from[n] = ((key & 63) * (a.rank + P) + a.rank + ((lane % KR_PIECES) ^ swizzle(key, KR_PIECES)) * 8) * 2;
  }
#pragma unroll
  for (int n = 0; n < V_LOADS; ++n) {
    const int d = (wave * V_LOADS + n) * 4 + (lane >> 4), piece = (lane & 15) ^ swizzle(d, 16);
    v_from[n] = (unsigned)((piece >> 3) * page_values + d * PAGE_TOKENS + (piece & 7) * 8) * 2;
  }
  const int room_first = a.window > 0 ? first_pair(uniform_load(a.positions + uniform_load(a.seq_starts + seq)), a.window) : 0;
  const char* const own_keys = (const char*)(a.keys + ((size_t)seq * a.pages + half) * page_keys + (size_t)h * PAGE_TOKENS * D);
  const char* const own_values = (const char*)(a.values + (size_t)seq * a.pages * page_values + (size_t)h * V * PAGE_TOKENS);
  // (the second page of the last step may not be there: nobody sees its keys)
  auto entry_of = [&](int step) { return RC > 0 ? uniform_load(bt + step * 2 + (step * LX_STEP + half * PAGE_TOKENS <= blk_last ? half : 0)) : 0; };
  auto fetch = [&](int step, int buffer, int entry) {
    const unsigned to = lds0 + buffer * STAGE;
    const char* const kp = own_keys + (size_t)(step - room_first) * 2 * page_keys * 2;
    const char* const vp = own_values + (size_t)(step - room_first) * 2 * page_values * 2;
#pragma unroll
    for (int n = 0; n < KN_LOADS; ++n) load_to_lds(kp, kn_from[n], to + (wave * KN_LOADS + n) * 1024);
    if constexpr (RC > 0) {
      const char* const rp = (const char*)(a.cache + readable_page(entry) * PAGE_TOKENS * (size_t)(a.rank + P));
#pragma unroll
      for (int n = 0; n < KR_LOADS; ++n) load_to_lds(rp, kr_from[n], to + KN_BYTES + (wave * KR_LOADS + n) * 1024);
    }
#pragma unroll
    for (int n = 0; n < V_LOADS; ++n) load_to_lds(vp, v_from[n], to + KN_BYTES + KR_BYTES + (wave * V_LOADS + n) * 1024);
  };

  // operand reads.  Which key sits in which row of a score tile is free: dealt so that lane half hb holds the probabilities of the
  // keys 8 hb .. 8 hb + 7 and 16 + 8 hb .. of the 32, each eight an operand of the second product as they are
  const int key_row = quarter * 32 + 16 * (j >> 4) + 8 * ((j >> 2) & 1) + 4 * ((j >> 3) & 1) + (j & 3);
  const int n_swizzle = swizzle(key_row, KN_PIECES), r_swizzle = swizzle(key_row, KR_PIECES);

  f32x16 acc[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[dt][v] = 0.f;
  float m = -1e30f, l = 0.f;

  const int step_first = lowest(blk_first) / LX_STEP, step_last = blk_last / LX_STEP;
  fetch(step_first, 0, entry_of(step_first));
  int buffer = 0, entry = step_first < step_last ? entry_of(step_first + 1) : 0;  // a step before it is needed
  for (int step = step_first; step <= step_last; ++step, buffer ^= 1) {
    tile_wait<0>();  // the step is there, and everybody has read the one before
    if (step < step_last) fetch(step + 1, buffer ^ 1, entry);
    if (step + 1 < step_last) entry = entry_of(step + 2);
    const int key0 = step * LX_STEP + quarter * 32;
    if (!has_work || key0 > wave_hi || key0 + 31 < wave_lo) continue;  // the same in all lanes
    const unsigned char* const kn = lx_lds + buffer * STAGE + key_row * (D * 2);
    const unsigned char* const kr = lx_lds + buffer * STAGE + KN_BYTES + key_row * (P * 2);
    const unsigned char* const vs = lx_lds + buffer * STAGE + KN_BYTES + KR_BYTES;
    f32x16 sc;
#pragma unroll
    for (int v = 0; v < 16; ++v) sc[v] = 0.f;
    {
      bf16x8 k[NC + RC];
#pragma unroll
      for (int c = 0; c < NC; ++c) k[c] = *reinterpret_cast<const bf16x8*>(kn + ((2 * c + hb) ^ n_swizzle) * 16);
#pragma unroll
      for (int c = 0; c < RC; ++c) k[NC + c] = *reinterpret_cast<const bf16x8*>(kr + ((2 * c + hb) ^ r_swizzle) * 16);
      __builtin_amdgcn_sched_barrier(0);  // all of them are asked for before the first product
#pragma unroll
      for (int c = 0; c < NC + RC; ++c) sc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(k[c], q[c], sc, 0, 0, 0);
    }
    bf16x8 values[DT][2];  // on their way during the softmax
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int n = 0; n < 2; ++n)
        values[dt][n] = *reinterpret_cast<const bf16x8*>(vs + (dt * 32 + j) * (LX_STEP * 2) + ((quarter * 4 + 2 * n + hb) ^ swizzle(j, 16)) * 16);
    __builtin_amdgcn_sched_barrier(0);
    if (!(key0 + 31 <= full_hi && key0 >= full_lo)) {  // the same in all lanes
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int key = key0 + 16 * (v >> 3) + 8 * hb + (v & 7);
        sc[v] = key <= pos && key >= lo ? sc[v] : -INFINITY;
      }
    }
    float top = max3(max3(sc[0], sc[1], sc[2]), max3(sc[3], sc[4], sc[5]), max3(sc[6], sc[7], sc[8]));
    top = max3(top, max3(sc[9], sc[10], sc[11]), max3(sc[12], sc[13], fmaxf(sc[14], sc[15])));
    {
      const unsigned u = __float_as_uint(top);
      const auto halves = __builtin_amdgcn_permlane32_swap(u, u, false, false);  // the column's other lane
      top = fmaxf(__uint_as_float(halves[0]), __uint_as_float(halves[1]));
    }
    const float m_new = fmaxf(m, top * a.scale2);  // (the scale is positive)
    const float alpha = __builtin_amdgcn_exp2f(m - m_new);
    m = m_new;
    float psum = 0.f;
    bf16x8 p[2];
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const float e = __builtin_amdgcn_exp2f(fmaf(sc[v], a.scale2, -m_new));
      psum += e;
      p[v >> 3][v & 7] = (bf16)e;
    }
    l = l * alpha + psum;
    if (__any(alpha != 1.f)) {  // the running maximum seldom moves after the first keys
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[dt][v] *= alpha;
    }
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int n = 0; n < 2; ++n) acc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(values[dt][n], p[n], acc[dt], 0, 0, 0);
  }
  __syncthreads();  // everybody has read the last step

  // the four waves of a run of queries meet: all but the first hand over
  float* const hand = reinterpret_cast<float*>(lx_lds) + (size_t)unit * 3 * (DT * 16 + 2) * 64 + lane;
  if (quarter > 0) {
    float* const to = hand + (size_t)(quarter - 1) * (DT * 16 + 2) * 64;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int v = 0; v < 16; ++v) to[(dt * 16 + v) * 64] = acc[dt][v];
    to[DT * 16 * 64] = m, to[(DT * 16 + 1) * 64] = l;
  }
  __syncthreads();
  if (quarter > 0 || !has_work) return;
  float f[4], top = m;
#pragma unroll
  for (int n = 0; n < 3; ++n) f[n + 1] = hand[((size_t)n * (DT * 16 + 2) + DT * 16) * 64], top = fmaxf(top, f[n + 1]);
  f[0] = __builtin_amdgcn_exp2f(m - top);
  float sum = l * f[0];
#pragma unroll
  for (int n = 0; n < 3; ++n) {
    f[n + 1] = __builtin_amdgcn_exp2f(f[n + 1] - top);
    sum += hand[((size_t)n * (DT * 16 + 2) + DT * 16 + 1) * 64] * f[n + 1];
  }
  sum += __shfl_xor(sum, 32, WAVE);
  if (a.sink != nullptr) sum += __builtin_amdgcn_exp2f(a.sink[h] * 1.4426950408889634f - top);  // the sink counts once a query
  if (!valid) return;
  float by = sum > 0.f ? 1.f / sum : 0.f;
  if (a.gate != nullptr) by /= 1.f + expf(-a.gate[(size_t)t * a.ldg + h]);
  bf16* const row = a.out + (size_t)t * a.ldo + (size_t)h * V;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      bf16x4 o;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float v = acc[dt][4 * b + e] * f[0];
#pragma unroll
        for (int n = 0; n < 3; ++n) v += hand[((size_t)n * (DT * 16 + 2) + dt * 16 + 4 * b + e) * 64] * f[n + 1];
        o[e] = (bf16)(v * by);
      }
      *reinterpret_cast<bf16x4*>(row + dt * 32 + 8 * b + 4 * hb) = o;
    }
}

// 1 if there is a kernel for these sizes: heads of 128 with a shared part of 64 or none, values of 128
extern "C" int fmsamd_latent_prompt_fits(int dim, int rot, int vdim, int rank) {
  return dim == 128 && (rot == 64 || rot == 0) && vdim == 128 && rank >= TL_BK && rank % 8 == 0;
}

// pages: of every sequence in keys and values, even, at least as many as the step's tokens of any sequence look at, from an even page on.
// Every row of q belongs to a query block (qblock_start, qblock_len: at most 64 tokens of one sequence each).
extern "C" int fmsamd_latent_prompt(const void* q, long ldq, void* out, long ldo, const void* cache, const void* uk, const void* uv,
                                    void* keys, void* values, const int* positions, const int* seq_of_token, const int* seq_starts,
                                    const int* qblock_start, const int* qblock_len, int n_qblocks, const int* block_table,
                                    int table_stride, int pages, const float* cos_t, const float* sin_t, const float* sink,
                                    const float* gate, long ldg, int n_seqs, int nheads, int dim, int rot, int vdim, int rank, float scale,
                                    int window, hipStream_t stream) {
  if (n_qblocks == 0 || n_seqs == 0) return 0;
  FMS_REQUIRE(fmsamd_latent_prompt_fits(dim, rot, vdim, rank), "latent_prompt: no kernel for heads of %d + %d, values of %d, a latent of %d", dim, rot,
              vdim, rank);
  FMS_REQUIRE(n_qblocks > 0 && n_seqs > 0 && nheads > 0 && pages > 0 && pages % 2 == 0 && table_stride > 0 && scale > 0.f && window >= 0,
              "latent_prompt: bad sizes");
  FMS_REQUIRE(ldq >= (long)nheads * (dim + rot) && ldq % 8 == 0 && ldo >= (long)nheads * vdim && ldo % 4 == 0, "latent_prompt: rows too short or not aligned");
  FMS_REQUIRE((((uintptr_t)q | (uintptr_t)cache | (uintptr_t)uk | (uintptr_t)uv | (uintptr_t)keys | (uintptr_t)values) & 15) == 0 && ((uintptr_t)out & 7) == 0 &&
                  ((uintptr_t)cos_t & 15) == 0 && ((uintptr_t)sin_t & 15) == 0,
              "latent_prompt: addresses not aligned");
  FMS_REQUIRE(rot == 0 || (cos_t != nullptr && sin_t != nullptr), "latent_prompt: a rotation needs its tables");
  FMS_REQUIRE(gate == nullptr || ldg >= nheads, "latent_prompt: rows of gates too short");
  // offsets from a sequence's first key or value of a page pair are counted in 32 bits
  FMS_REQUIRE((long)nheads * PAGE_TOKENS * (dim > vdim ? dim : vdim) * 4 < (1l << 31) && (long)n_seqs * (pages / 2) < (1l << 31) &&
                  (long)n_qblocks * nheads < (1l << 31) && nheads <= 16384,
              "latent_prompt: too much for one launch");
  const ExpandArgs e{(const bf16*)cache, rank + rot, (const bf16*)uk, (const bf16*)uv, (bf16*)keys, (bf16*)values, positions, seq_starts,
                     block_table, table_stride, pages, nheads, dim, vdim, rank, window};
  latent_expand_kernel<<<dim3(n_seqs * (pages / 2), ceil_div((long)nheads * dim, 128) + ceil_div((long)nheads * vdim, 128)), 256, 0, stream>>>(e);
  FMS_LAUNCH_CHECK("latent_expand");
  const PromptArgs a{(const bf16*)q, ldq, (bf16*)out, ldo, (const bf16*)keys, (const bf16*)values, (const bf16*)cache, positions, seq_of_token,
                     seq_starts, qblock_start, qblock_len, block_table, cos_t, sin_t, sink, gate, ldg, n_qblocks, table_stride, pages, nheads, rank, window,
                     scale * 1.4426950408889634f};
#define LAUNCH_PROMPT(RC)                                                                                                     \
  do {                                                                                                                        \
    const int bytes = 2 * LX_STEP * (128 + RC * 16 + 128) * 2;                                                                \
    /* more than 64 KB of LDS a block has to be asked for */                                                                  \
    const hipError_t err = hipFuncSetAttribute((const void*)latent_prompt_kernel<8, RC, 4>, hipFuncAttributeMaxDynamicSharedMemorySize, bytes); \
    FMS_REQUIRE(err == hipSuccess, "latent_prompt: the kernel's LDS could not be sized: %s", hipGetErrorString(err));          \
    latent_prompt_kernel<8, RC, 4><<<(unsigned)(n_qblocks * nheads), 512, bytes, stream>>>(a);                                 \
  } while (0)
  if (rot == 64)
    LAUNCH_PROMPT(4);
  else
    LAUNCH_PROMPT(0);
#undef LAUNCH_PROMPT
  FMS_LAUNCH_CHECK("latent_prompt");
  return 0;
}
