// A feed-forward of many small experts of which every token uses a few.
//
//   route:    float32 router logits [T, E] -> the `top` largest per token (ties: the lower index) and their weights:
//             the softmax over those `top` logits alone, or every chosen logit's sigmoid (as it is, or divided by the
//             sum of the chosen ones).
//   group:    the T * top (token, choice) pairs sorted by expert, cut into tiles of rows that belong to one expert
//             each.  It runs on the device, in one block, so a step never waits for the host (and can be captured).
//   gate_up:  for every tile, hidden = clamp-gated activation of (x Wg_e^T, x Wu_e^T)
//   down:     for every tile, y[pair] = hidden Wd_e^T, float32, at the pair's own place (token * top + choice)
//   combine:  out[t] = sum_j weight[t, j] y[t * top + j]  (+ sigmoid(shared_gate[t]) * shared[t]), summed in the order
//             of j: a token's result does not depend on what else is in the batch.
//
// The products take their rows through tile_product.h (float32 FMA for the 32-bit path and for bfloat16 rows that are not
// aligned to 16 bytes) and tile_product_lds.h (MFMA 32x32x16 for bfloat16).
// The grids are sized for the worst case (every expert with a ragged last tile); tiles that do not exist leave at once.
#include "common.h"
#include "fmsamd.h"
#include "tile_product.h"
#include "tile_product_lds.h"

// rows of the matrix-core kernels' tiles
#define TILE_SMALL_ROWS 32
#define TILE_BIG_ROWS 128
#define EXPERT_COMPUTE_UNITS 256

#define ROUTE_MAX_EXPERTS 1024
#define ROUTE_MAX_TOP 64

// The largest of a wave's values, in all lanes: rows of 16 lanes in the vector unit, then their four results.
__device__ __forceinline__ float route_max(float v) {
#define ROUTE_DPP_MAX(ctrl) v = fmaxf(v, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), ctrl, 0xF, 0xF, true)))
  ROUTE_DPP_MAX(0xB1);   // quad_perm [1, 0, 3, 2]
  ROUTE_DPP_MAX(0x4E);   // quad_perm [2, 3, 0, 1]
  ROUTE_DPP_MAX(0x141);  // row_half_mirror
  ROUTE_DPP_MAX(0x140);  // row_mirror
#undef ROUTE_DPP_MAX
  auto of = [&](int lane) { return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane)); };
  return fmaxf(fmaxf(of(0), of(16)), fmaxf(of(32), of(48)));
}

// The `top` largest of the values z(e), e < n_experts <= 64 PER, and their weights, by a wave that keeps them in registers: a round is the largest
// value, the lanes that have it and the lowest index among them (a chain of shuffles through LDS with value and index takes 0.6 us a round).
template <int PER, typename Value>
__device__ __forceinline__ void route_row(Value z, int lane, int n_experts, int top, int score, int* ids, float* weights) {
  float v[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) v[i] = lane + i * WAVE < n_experts ? z(lane + i * WAVE) : 0.f;
  float mine = 0.f;  // lane j: the j-th chosen one
  int my_id = 0;
  for (int j = 0; j < top; ++j) {
    float best = -INFINITY;
    int at = 0x7fffffff;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int e = lane + i * WAVE;
      if (e < n_experts && (v[i] > best || (v[i] == best && e < at))) best = v[i], at = e;
    }
    if (at == 0x7fffffff) at = lane < n_experts ? lane : 0;  // only NaNs left in this lane's share
    const float largest = route_max(best);
    unsigned long long have = __ballot(best == largest);
    int chosen = 0x7fffffff;
    for (; have != 0; have &= have - 1) {  // one lane, but for ties
      const int other = __builtin_amdgcn_readlane(at, __builtin_ctzll(have));
      chosen = other < chosen ? other : chosen;
    }
    if (lane == j) mine = largest, my_id = chosen;
#pragma unroll
    for (int i = 0; i < PER; ++i) v[i] = lane + i * WAVE == chosen ? -INFINITY : v[i];
  }
  auto of = [&](float x, int j) { return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), j)); };
  const float m = of(mine, 0);  // the largest comes first
  // softmax over the chosen ones, or sigmoid scores (the order of the logits is the order of their sigmoids); sums in the order of j
  const float one = score == FMS_ROUTE_SOFTMAX ? expf(mine - m) : 1.f / (1.f + expf(-mine));
  float sum = 0.f;
  for (int j = 0; j < top; ++j) sum += of(one, j);
  const float norm = score == FMS_ROUTE_SIGMOID_NORMED ? 1.f / sum : 1.f;
  if (lane < top) {
    ids[lane] = my_id;
    weights[lane] = score == FMS_ROUTE_SOFTMAX ? one / sum : norm / (1.f + expf(-mine));
  }
}

// One wave per token.
template <int PER>
__global__ void __launch_bounds__(256)
    route_kernel(const float* __restrict__ logits, long ld, int n_tokens, int n_experts, int top, int score, int* __restrict__ ids,
                 float* __restrict__ weights) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int t = blockIdx.x * 4 + wave;
  if (t >= n_tokens) return;
  route_row<PER>([&](int e) { return logits[(size_t)t * ld + e]; }, lane, n_experts, top, score, ids + (size_t)t * top, weights + (size_t)t * top);
}

// The smallest number of values a lane that a kernel is built for.
#define ROUTE_PER(n_experts, CALL)     \
  do {                                 \
    if ((n_experts) <= WAVE) CALL(1);  \
    else if ((n_experts) <= 4 * WAVE) CALL(4); \
    else CALL(16);                     \
  } while (0)
static_assert(ROUTE_MAX_EXPERTS <= 16 * WAVE && ROUTE_MAX_TOP <= WAVE, "values a lane, and a lane for every choice");

// The router's product and the choice as one kernel, for the few tokens of a decode step: a block of sixteen waves a token, a row of W a wave
// at a time, three rows asked for at once.  Bound by a launch, the round trip for x and W together and the chain of the choice.  Width 2048, 33
// outputs, 4 chosen, us, the two kernels and this one: 1 token 5.6 and 4.8, 8 5.6 and 5.0, 32 7.4 and 5.1, 128 10.9 and 5.3 (the
// two with the choice's shuffles through LDS 7.9, 9.3, 10.5, 14.1).  Every token reads all of W: 128 outputs of width 1024 7.5 and 7.7 for 16
// tokens, 8.1 and 7.7 for 32; 65 of width 4096 10 and 14.
#define ROUTER_WAVES 16
#define ROUTER_WIDEST 2048
// CHUNKS: of 512 elements of a row; PER: route_row's
template <int CHUNKS, int PER>
__global__ void __launch_bounds__(ROUTER_WAVES* WAVE)
    router_kernel(const bf16* __restrict__ x, long ldx, const bf16* __restrict__ w, int K, int n_out, int n_experts, int top, int score,
                  float* __restrict__ logits, int* __restrict__ ids, float* __restrict__ weights) {
  __shared__ float z[PER * WAVE];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), lane = threadIdx.x & (WAVE - 1), t = blockIdx.x;
  const bf16x8 zero = __builtin_bit_cast(bf16x8, f32x4{0.f, 0.f, 0.f, 0.f});
  auto row = [&](const bf16* from, bf16x8 (&to)[CHUNKS]) {
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
      const int k = c * 512 + lane * 8;
      to[c] = k < K ? *reinterpret_cast<const bf16x8*>(from + k) : zero;
    }
  };
  bf16x8 v[CHUNKS];
  row(x + (size_t)t * ldx, v);
  constexpr int AT_ONCE = 3;
  for (int n0 = wave; n0 < n_out; n0 += ROUTER_WAVES * AT_ONCE) {
    bf16x8 u[AT_ONCE][CHUNKS];
#pragma unroll
    for (int i = 0; i < AT_ONCE; ++i) row(w + (size_t)(n0 + i * ROUTER_WAVES < n_out ? n0 + i * ROUTER_WAVES : n0) * K, u[i]);
#pragma unroll
    for (int i = 0; i < AT_ONCE; ++i) {
      float sum = 0.f;
#pragma unroll
      for (int c = 0; c < CHUNKS; ++c)
#pragma unroll
        for (int e = 0; e < 8; ++e) sum = fmaf((float)v[c][e], (float)u[i][c][e], sum);
      sum = row16_sum(sum);
      sum += __shfl_xor(sum, 16, WAVE);
      sum += __shfl_xor(sum, 32, WAVE);
      const int n = n0 + i * ROUTER_WAVES;
      if (lane == 0 && n < n_out) {
        logits[(size_t)t * n_out + n] = sum;
        if (n < n_experts) z[n] = sum;
      }
    }
  }
  __syncthreads();
  if (wave == 0) route_row<PER>([&](int e) { return z[e]; }, lane, n_experts, top, score, ids + (size_t)t * top, weights + (size_t)t * top);
}

// logits [n_tokens, n_out] = x W^T in float32 (bfloat16 x and W, K a multiple of 8 up to 2048, 16-byte addresses), and the choice among
// the first n_experts of them as fmsamd_moe_route makes it.
extern "C" int fmsamd_moe_router(const void* x, long ldx, const void* w, int n_tokens, int K, int n_out, int n_experts, int top, int score,
                                 float* logits, int* ids, float* weights, hipStream_t stream) {
  if (n_tokens == 0) return 0;
  FMS_REQUIRE(n_tokens > 0 && n_experts > 0 && n_experts <= n_out && n_out <= ROUTE_MAX_EXPERTS + 1 && top > 0 && top <= n_experts && top <= ROUTE_MAX_TOP,
              "moe_router: %d experts of %d outputs (at most %d), top %d (at most %d and the experts)", n_experts, n_out, ROUTE_MAX_EXPERTS, top,
              ROUTE_MAX_TOP);
  FMS_REQUIRE(K > 0 && K % 8 == 0 && K <= ROUTER_WIDEST && ldx >= K && ldx % 8 == 0 && (uintptr_t)x % 16 == 0 && (uintptr_t)w % 16 == 0,
              "moe_router: K=%d (a multiple of 8, at most %d), row stride %ld", K, ROUTER_WIDEST, ldx);
  FMS_REQUIRE(score >= FMS_ROUTE_SOFTMAX && score <= FMS_ROUTE_SIGMOID_NORMED, "moe_router: unknown score %d", score);
#define FMS_ROUTER(CHUNKS, PER)                                                                                                             \
  router_kernel<CHUNKS, PER><<<n_tokens, ROUTER_WAVES * WAVE, 0, stream>>>((const bf16*)x, ldx, (const bf16*)w, K, n_out, n_experts, top, score, \
                                                                           logits, ids, weights)
#define FMS_ROUTER_OF(PER)                   \
  do {                                       \
    if (K <= 1024) FMS_ROUTER(2, PER);       \
    else FMS_ROUTER(4, PER);                 \
  } while (0)
  ROUTE_PER(n_experts, FMS_ROUTER_OF);
#undef FMS_ROUTER_OF
#undef FMS_ROUTER
  FMS_LAUNCH_CHECK("moe_router");
  return 0;
}

extern "C" int fmsamd_moe_route(const float* logits, long ld, int n_tokens, int n_experts, int top, int score, int* ids,
                                float* weights, hipStream_t stream) {
  if (n_tokens == 0) return 0;
  FMS_REQUIRE(n_tokens > 0 && n_experts > 0 && n_experts <= ROUTE_MAX_EXPERTS && top > 0 && top <= n_experts && top <= ROUTE_MAX_TOP,
              "moe_route: %d experts (at most %d), top %d (at most %d and the experts)", n_experts, ROUTE_MAX_EXPERTS, top, ROUTE_MAX_TOP);
  FMS_REQUIRE(ld >= n_experts, "moe_route: rows of %ld for %d experts", ld, n_experts);
  FMS_REQUIRE(score >= FMS_ROUTE_SOFTMAX && score <= FMS_ROUTE_SIGMOID_NORMED, "moe_route: unknown score %d", score);
#define FMS_ROUTE(PER) route_kernel<PER><<<ceil_div(n_tokens, 4), 256, 0, stream>>>(logits, ld, n_tokens, n_experts, top, score, ids, weights)
  ROUTE_PER(n_experts, FMS_ROUTE);
#undef FMS_ROUTE
  FMS_LAUNCH_CHECK("moe_route");
  return 0;
}

// The wave's largest value and where it is (ties: the lower index); every lane gets both.
__device__ __forceinline__ void wave_argmax(float& best, int& at) {
#pragma unroll
  for (int off = WAVE / 2; off > 0; off >>= 1) {
    const float ov = __shfl_xor(best, off, WAVE);
    const int oa = __shfl_xor(at, off, WAVE);
    if (ov > best || (ov == best && oa < at)) best = ov, at = oa;
  }
}

__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_wave_barrier();
  __threadfence_block();
}

// Routing over groups of experts.  s = softmax over all n router outputs; an output is chosen by s + correction, but
// weighted by s.  The outputs form `groups` equal runs of neighbours; a group's score is its largest choice score, and
// only outputs of the `keep` best groups can be chosen (the others count as minus infinity).  The weights of the `top`
// chosen are their s divided by their sum (+ 1e-20), times `scale`.  One wave per token; ties go to the lower index.
__global__ void __launch_bounds__(256)
    route_grouped_kernel(const float* __restrict__ logits, long ld, int n_tokens, int n, int top, const float* __restrict__ correction,
                         int groups, int keep, float scale, int* __restrict__ ids, float* __restrict__ weights) {
  extern __shared__ float lds[];  // 4 waves x (2 n + 2 groups + top)
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int t = blockIdx.x * 4 + wave;
  if (t >= n_tokens) return;
  float* s = lds + (size_t)wave * (2 * n + 2 * groups + top);
  float* choice = s + n;
  float* gscore = choice + n;
  float* kept = gscore + groups;
  float* chosen = kept + groups;
  float m = -INFINITY;
  for (int e = lane; e < n; e += WAVE) {
    const float z = logits[(size_t)t * ld + e];
    s[e] = z;
    m = fmaxf(m, z);
  }
  m = wave_max(m);
  float sum = 0.f;
  for (int e = lane; e < n; e += WAVE) {
    const float p = expf(s[e] - m);
    s[e] = p;
    sum += p;
  }
  sum = wave_sum(sum);
  for (int e = lane; e < n; e += WAVE) {
    const float p = s[e] / sum;
    float c = p + (correction ? correction[e] : 0.f);
    if (!(c >= -3.0e38f)) c = -3.0e38f;  // not a number (a padding row's logits): still a candidate, the last of all
    s[e] = p;
    choice[e] = c;
  }
  wave_lds_fence();
  if (groups > 1) {
    const int per = n / groups;
    for (int g = lane; g < groups; g += WAVE) {
      float best = -INFINITY;
      for (int e = g * per; e < (g + 1) * per; ++e) best = fmaxf(best, choice[e]);
      gscore[g] = best;
      kept[g] = 0.f;
    }
    wave_lds_fence();
    for (int j = 0; j < keep; ++j) {
      float best = -INFINITY;
      int at = 0x7fffffff;
      for (int g = lane; g < groups; g += WAVE) {
        const float v = gscore[g];
        if (v > best || (v == best && g < at)) best = v, at = g;
      }
      wave_argmax(best, at);
      if (lane == 0 && at < groups) kept[at] = 1.f, gscore[at] = -INFINITY;
      wave_lds_fence();
    }
    for (int e = lane; e < n; e += WAVE)
      if (kept[e / per] == 0.f) choice[e] = -INFINITY;
    wave_lds_fence();
  }
  for (int j = 0; j < top; ++j) {
    float best = -INFINITY;
    int at = 0x7fffffff;
    for (int e = lane; e < n; e += WAVE) {
      const float v = choice[e];
      if (v > best || (v == best && e < at)) best = v, at = e;
    }
    wave_argmax(best, at);
    if (at >= n) at = 0;  // nothing left to choose from: the configuration allows fewer outputs than `top`
    if (lane == 0) {
      ids[(size_t)t * top + j] = at;
      chosen[j] = s[at];
      choice[at] = -INFINITY;
    }
    wave_lds_fence();
  }
  if (lane == 0) {
    float total = 0.f;
    for (int j = 0; j < top; ++j) total += chosen[j];
    const float norm = scale / (total + 1e-20f);
    for (int j = 0; j < top; ++j) weights[(size_t)t * top + j] = chosen[j] * norm;
  }
}

extern "C" int fmsamd_moe_route_grouped(const float* logits, long ld, int n_tokens, int n_outputs, int top, const float* correction,
                                        int groups, int keep, float scale, int* ids, float* weights, hipStream_t stream) {
  if (n_tokens == 0) return 0;
  FMS_REQUIRE(n_tokens > 0 && n_outputs > 0 && n_outputs <= ROUTE_MAX_EXPERTS && top > 0 && top <= n_outputs && top <= ROUTE_MAX_TOP,
              "moe_route_grouped: %d outputs (at most %d), top %d (at most %d and the outputs)", n_outputs, ROUTE_MAX_EXPERTS, top,
              ROUTE_MAX_TOP);
  FMS_REQUIRE(ld >= n_outputs, "moe_route_grouped: rows of %ld for %d outputs", ld, n_outputs);
  FMS_REQUIRE(groups >= 1 && n_outputs % groups == 0 && keep >= 1 && keep <= groups && (long)keep * (n_outputs / groups) >= top,
              "moe_route_grouped: %d groups of %d outputs, %d kept, cannot give %d choices", groups, n_outputs / (groups > 0 ? groups : 1),
              keep, top);
  const size_t lds = 4 * (size_t)(2 * n_outputs + 2 * groups + top) * sizeof(float);
  route_grouped_kernel<<<ceil_div(n_tokens, 4), 256, lds, stream>>>(logits, ld, n_tokens, n_outputs, top, correction, groups, keep, scale,
                                                                    ids, weights);
  FMS_LAUNCH_CHECK("moe_route_grouped");
  return 0;
}

// --------------------------------------------------------------------------
// group: order[0 .. n) = the pairs sorted by expert; tiles[i] = (expert, first row in order, rows), rows 0: no tile.  The last
// of the max_tiles places never holds one (fmsamd_moe_max_tiles asks for more than there can be): its second number says
// how many tiles there are.
// --------------------------------------------------------------------------
// One block.  Its time is round trips: a thread asks for eight ids at a time, and the experts' places come from a scan over
// the threads (an expert each).  8192 pairs of 32 experts: 7.6 us (12.6 with ids one by one and one thread adding up); 32 pairs:
// 4.9 (5.9).
#define GROUP_THREADS 1024
__global__ void __launch_bounds__(GROUP_THREADS)
    group_kernel(const int* __restrict__ ids, int n_pairs, int n_experts, int* __restrict__ order, int* __restrict__ tiles,
                 int max_tiles, int tile_rows) {
  __shared__ int counts[ROUTE_MAX_EXPERTS];
  __shared__ int cursor[ROUTE_MAX_EXPERTS];
  __shared__ int wave_pairs[GROUP_THREADS / WAVE], wave_tiles[GROUP_THREADS / WAVE];
  const int tid = threadIdx.x, lane = tid & (WAVE - 1), wave = tid / WAVE;
  for (int e = tid; e < n_experts; e += GROUP_THREADS) counts[e] = 0;
  __syncthreads();
  constexpr int AHEAD = 8;
  for (int a0 = tid; a0 < n_pairs; a0 += AHEAD * GROUP_THREADS) {
    int e[AHEAD];
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) {
      const int a = a0 + i * GROUP_THREADS;
      e[i] = a < n_pairs ? ids[a] : -1;
    }
#pragma unroll
    for (int i = 0; i < AHEAD; ++i)
      if (e[i] >= 0 && e[i] < n_experts) atomicAdd(&counts[e[i]], 1);
  }
  __syncthreads();
  // thread e: how many pairs and tiles the experts before e have (there are no more experts than threads)
  const int c = tid < n_experts ? counts[tid] : 0, t = (c + tile_rows - 1) / tile_rows;
  int pairs = c, some = t;
#pragma unroll
  for (int off = 1; off < WAVE; off <<= 1) {
    const int p = __shfl_up(pairs, off, WAVE), q = __shfl_up(some, off, WAVE);
    if (lane >= off) pairs += p, some += q;
  }
  if (lane == WAVE - 1) wave_pairs[wave] = pairs, wave_tiles[wave] = some;
  __syncthreads();
  int before = pairs - c, nt = some - t, all = 0;
  for (int w = 0; w < GROUP_THREADS / WAVE; ++w) {
    if (w < wave) before += wave_pairs[w], nt += wave_tiles[w];
    all += wave_tiles[w];
  }
  all = all < max_tiles ? all : max_tiles;
  if (tid < n_experts) {
    cursor[tid] = before;
    for (int r = 0; r < c && nt < max_tiles; r += tile_rows, ++nt) {
      tiles[3 * nt] = tid;
      tiles[3 * nt + 1] = before + r;
      tiles[3 * nt + 2] = c - r < tile_rows ? c - r : tile_rows;
    }
  }
  for (int i = 3 * all + tid; i < 3 * max_tiles; i += GROUP_THREADS) tiles[i] = i == 3 * max_tiles - 2 ? all : 0;
  __syncthreads();
  for (int a0 = tid; a0 < n_pairs; a0 += AHEAD * GROUP_THREADS) {
    int e[AHEAD];
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) {
      const int a = a0 + i * GROUP_THREADS;
      e[i] = a < n_pairs ? ids[a] : -1;
    }
#pragma unroll
    for (int i = 0; i < AHEAD; ++i)
      if (e[i] >= 0 && e[i] < n_experts) order[atomicAdd(&cursor[e[i]], 1)] = a0 + i * GROUP_THREADS;
  }
}

// Rows of a tile.  The matrix-core kernels (wide_ok: bfloat16, everything aligned to 16 bytes) take large tiles where experts fill
// more than one small one on average and read their weights twice, and there are pairs enough to give the compute units work in
// large tiles.  Both products and the grouping, us, small tiles and large ones, weights out of memory: 32 experts, 4 a token, width 2048,
// hidden 1024, 150 tokens (18 rows an expert) 78, 85, 200 (25) 96, 88, 256 (32) 116, 89; 64 experts, 8 a token, hidden 768, 200 tokens
// (25) 136, 144, 256 (32) 158, 147; 8 experts, 2 a token, width 768, hidden 2048, 256 tokens (512 pairs) 50, 57, 512 (1024 pairs) 63,
// 63; width 1024, hidden 512, 512 tokens 26, 36, 1024 tokens 43, 38.
#define TILE_BIG_PAIRS 1024
extern "C" int fmsamd_moe_tile_rows(int n_pairs, int n_experts, int wide_ok) {
  if (!wide_ok) return TILE_ROWS;
  return n_pairs >= TILE_BIG_PAIRS && n_pairs >= (long)TILE_SMALL_ROWS * n_experts ? TILE_BIG_ROWS : TILE_SMALL_ROWS;
}

// More than there can be: an expert with c pairs has at most (c + tile_rows - 1) / tile_rows tiles, less than c / tile_rows + 1.
extern "C" int fmsamd_moe_max_tiles(int n_pairs, int n_experts, int tile_rows) {
  if (tile_rows <= 0) return 0;
  return (n_pairs + tile_rows - 1) / tile_rows + (n_experts < n_pairs ? n_experts : n_pairs);
}

extern "C" int fmsamd_moe_group(const int* ids, int n_pairs, int n_experts, int* order, int* tiles, int max_tiles,
                                int tile_rows, hipStream_t stream) {
  if (n_pairs == 0) return 0;
  FMS_REQUIRE(n_pairs > 0 && n_experts > 0 && n_experts <= ROUTE_MAX_EXPERTS, "moe_group: %d pairs, %d experts (at most %d)", n_pairs,
              n_experts, ROUTE_MAX_EXPERTS);
  FMS_REQUIRE(tile_rows == TILE_ROWS || tile_rows == TILE_SMALL_ROWS || tile_rows == TILE_BIG_ROWS, "moe_group: tiles of %d rows", tile_rows);
  FMS_REQUIRE(max_tiles >= fmsamd_moe_max_tiles(n_pairs, n_experts, tile_rows), "moe_group: room for %d tiles, %d may be needed", max_tiles,
              fmsamd_moe_max_tiles(n_pairs, n_experts, tile_rows));
  static_assert(ROUTE_MAX_EXPERTS <= GROUP_THREADS, "an expert a thread");
  group_kernel<<<1, GROUP_THREADS, 0, stream>>>(ids, n_pairs, n_experts, order, tiles, max_tiles, tile_rows);
  FMS_LAUNCH_CHECK("moe_group");
  return 0;
}

// --------------------------------------------------------------------------
// the experts' products
// --------------------------------------------------------------------------
struct ExpertArgs {
  const void* x;  // gate_up: [T, ldx] token rows; down: hidden [pairs, ldx] in sorted order
  long ldx;
  const void* w1;  // gate_up: gate weights [E, N, K]; down: down weights [E, N, K]
  const void* w2;  // gate_up: up weights [E, N, K]
  void* y;  // gate_up: hidden [pairs, N] in sorted order; down: float32 [pairs, N] by pair
  const int* order;
  const int* tiles;
  int top, N, K;
  float limit, alpha, shift;
  const float* in_scale;  // gate_up: a factor per pair on the expert's input (applied to both float32 sums), or null
  int act;  // gate_up without up weights (w2 null): hidden = act(x W1^T), one of FMS_ACT_*
};

// (the matrix-core kernels look a tile's pairs and their factors up at the start: at the end, a row after the other, they are a chain of
// round trips to memory, some 10 us of a large tile)
__device__ __forceinline__ float pair_scale(const ExpertArgs& a, int sorted_row) {
  return a.in_scale ? a.in_scale[a.order[sorted_row]] : 1.f;
}

__device__ __forceinline__ float clamp_gated(float g, float u, float limit, float alpha, float shift) {
  g = fminf(g, limit);
  u = fminf(fmaxf(u, -limit), limit);
  return g / (1.f + expf(-alpha * g)) * (u + shift);
}

// what an expert keeps between its two products: the clamped gated activation of (gate, up), or act(the one product)
__device__ __forceinline__ float hidden_value(const ExpertArgs& a, bool gated, float g, float u) {
  return gated ? clamp_gated(g, u, a.limit, a.alpha, a.shift) : fms_activate(g, a.act);
}

template <typename T>
__global__ void __launch_bounds__(TILE_THREADS) expert_gate_up_fma_kernel(ExpertArgs a) {
  const int e = a.tiles[3 * blockIdx.x], start = a.tiles[3 * blockIdx.x + 1], rows = a.tiles[3 * blockIdx.x + 2];
  if (rows == 0) return;
  const int n0 = blockIdx.y * TILE_FMA_COLS;
  const T* x = (const T*)a.x;
  const T* wg = (const T*)a.w1 + (size_t)e * a.N * a.K;
  const T* wu = (const T*)a.w2 + (size_t)e * a.N * a.K;
  auto a_row = [&](int m) { return m < rows ? x + (size_t)(a.order[start + m] / a.top) * a.ldx : (const T*)nullptr; };
  const bool gated = a.w2 != nullptr;
  float g[4], u[4] = {0.f, 0.f, 0.f, 0.f};
  tile_product_fma<T>(a_row, [&](int n) { return n0 + n < a.N ? wg + (size_t)(n0 + n) * a.K : (const T*)nullptr; }, a.K, g);
  if (gated) tile_product_fma<T>(a_row, [&](int n) { return n0 + n < a.N ? wu + (size_t)(n0 + n) * a.K : (const T*)nullptr; }, a.K, u);
  const int n = n0 + threadIdx.x % 64;
  if (n >= a.N) return;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int m = (threadIdx.x / 64) * 4 + i;
    if (m < rows) {
      const float sc = pair_scale(a, start + m);
      ((T*)a.y)[(size_t)(start + m) * a.N + n] = from_f32<T>(hidden_value(a, gated, g[i] * sc, u[i] * sc));
    }
  }
}

template <typename T>
__global__ void __launch_bounds__(TILE_THREADS) expert_down_fma_kernel(ExpertArgs a) {
  const int e = a.tiles[3 * blockIdx.x], start = a.tiles[3 * blockIdx.x + 1], rows = a.tiles[3 * blockIdx.x + 2];
  if (rows == 0) return;
  const int n0 = blockIdx.y * TILE_FMA_COLS;
  const T* x = (const T*)a.x;
  const T* w = (const T*)a.w1 + (size_t)e * a.N * a.K;
  float acc[4];
  tile_product_fma<T>([&](int m) { return m < rows ? x + (size_t)(start + m) * a.ldx : (const T*)nullptr; },
                      [&](int n) { return n0 + n < a.N ? w + (size_t)(n0 + n) * a.K : (const T*)nullptr; }, a.K, acc);
  const int n = n0 + threadIdx.x % 64;
  if (n >= a.N) return;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int m = (threadIdx.x / 64) * 4 + i;
    if (m < rows) ((float*)a.y)[(size_t)a.order[start + m] * a.N + n] = acc[i];
  }
}

// The same two products in bfloat16: tiles of 32 or 128 rows, through LDS (tile_product_lds.h).  For the gated product half of a
// wave's tiles are gate columns and the others the up columns of the same elements, so that both meet in one lane.  The
// column blocks of a tile follow one another on one of the eight dies (blocks are dealt to the dies in turn), the tiles of
// an expert behind each other, so that rows and weights come from memory once.
//
// Few rows an expert (decode) are bound by the weights' bytes: tiles of 32 rows by 64 rows of W, one wave and three stages of 12 KB a
// block, four blocks a compute unit.  Many rows (prompts) by the matrix unit, the rounds of blocks over the compute units and the start
// and end of a block together: 128 rows by 256 rows of W; the waves whose rows a short tile does not have load for the others and
// multiply nothing.  Blocks start their walk over K at different steps (expert_first_step).
// Measured with weights out of memory, 32 experts, 4 a token, width 2048, hidden 1024, grouping, gate and up and down together (in
// brackets the same without that start, with 128 rows of W a small block and the pairs looked up at the end of a block): 8 tokens 52 us
// (65), 32 tokens 70 (89; 5.8 TB/s), 128 tokens 72 (92), 300 tokens 89 (111), 1000 140 (158), 2048 206 (230), 2277 with scaled inputs
// 218 (253), 4096 334 (356).  Small tiles with four stages: 85 for 32 tokens; by 128 rows of W: 56 for 8 tokens, the rest as it is.
// Large ones as waves of 64 x 64: 203 for 2048 tokens, 226 for 2277; 128 x 128 with two blocks a compute unit 224, 238.
__device__ __forceinline__ bool expert_place(const ExpertArgs& a, int max_tiles, int col_blocks, int& tile, int& col) {
  const int total = uniform_load(a.tiles + 3 * max_tiles - 2) * col_blocks;  // the tiles there are (group_kernel)
  const int per_die = (total + 7) / 8;
  const int at = (blockIdx.x & 7) * per_die + (blockIdx.x >> 3);
  tile = at / col_blocks, col = at % col_blocks;
  return (int)(blockIdx.x >> 3) < per_die && at < total;
}

// Are the weight rows of this tile loaded as bytes that are not read again?  Where a tile of 32 rows is the only one of its expert,
// nobody else reads them; the other tiles of a popular expert do.  And with fewer blocks than compute units (of which each can take four) such loads
// take longer.  Grouping, gate, up and down together, us, weights out of memory, with this rule, no load marked and every load marked: 32 experts, 4 a
// token, width 2048, hidden 1024, 4 tokens 42, 46, 41, 32 tokens 69, 77, 68, 128 tokens 74, 84, 73, 128 tokens of which most go to a few
// experts 101, 103, 109; 64 experts, 8 a token, hidden 768, 32 tokens 110, 121, 110, 128 such tokens 123, 135, 139, one token (192 and 256
// blocks) 30, 27, 30; 8 experts, 2 a token, width 768, hidden 2048, 256 tokens 49, 48, 55.  Two or four times as many blocks as the line: a token
// of the 64 experts 27, 4 to 32 tokens of the 32 up to 77.
template <int BM>
__device__ __forceinline__ bool expert_reads_once(const ExpertArgs& a, int max_tiles, int col_blocks, int tile, int e) {
  if (BM != TILE_SMALL_ROWS) return false;
  const int* const t = a.tiles + 3 * tile;  // (the place behind the last tile is there: fmsamd_moe_max_tiles)
  const bool alone = !(tile > 0 && t[-3] == e) && !(t[3] == e && t[5] > 0);
  return alone && a.tiles[3 * max_tiles - 2] * col_blocks >= EXPERT_COMPUTE_UNITS;
}

// The step of K that a block starts with: weight rows lie a multiple of kilobytes apart, and the blocks of all experts in step crowd into few
// memory channels.  It goes with the expert alone: the blocks of a tile share its rows, and those of an expert its weights, while they are in
// an L2.  Grouping, gate, up and down together, us, all blocks at the start of K, this, and another start for every column: 32 experts, 4 a token, width
// 2048, hidden 1024, 32 tokens 85, 75, 76, 2048 tokens 205, 199, 203; 4 experts, 2 a token, width 4096, hidden 3584, 1024 tokens 275, 273, 309, 4096 tokens
// 895, 895, 1065.  And a pair has the same bits in any tile.
__device__ __forceinline__ int expert_first_step(int e, int K) { return 3 * e % ((K + TL_BK - 1) / TL_BK); }

template <int WM, int WN, int TM, int TN, int ST, bool GATED>
__global__ void __launch_bounds__(WM* WN* WAVE) __attribute__((amdgpu_waves_per_eu(2))) expert_gate_up_lds_kernel(ExpertArgs a, int max_tiles, int col_blocks) {
  typedef TileLds<WM, WN, TM, TN, ST> S;
  __shared__ __attribute__((aligned(16))) bf16 lds[S::LDS_ELEMENTS];
  __shared__ int pairs[S::BM];  // of the tile's rows
  int tile, col;
  if (!expert_place(a, max_tiles, col_blocks, tile, col)) return;
  const int e = uniform_load(a.tiles + 3 * tile), start = uniform_load(a.tiles + 3 * tile + 1), rows = uniform_load(a.tiles + 3 * tile + 2);
  const int own_pair = (int)threadIdx.x < S::BM ? a.order[start + ((int)threadIdx.x < rows ? threadIdx.x : 0)] : 0;
  const float own_scale = (int)threadIdx.x < S::BM && a.in_scale ? a.in_scale[own_pair] : 1.f;
  __shared__ float scales[S::BM];
  if ((int)threadIdx.x < S::BM) pairs[threadIdx.x] = own_pair;
  __syncthreads();
  const bf16* x = (const bf16*)a.x;
  const bf16* wg = (const bf16*)a.w1 + (size_t)e * a.N * a.K;
  const bf16* wu = (const bf16*)a.w2 + (size_t)e * a.N * a.K;
  // gated: a wave's first TN / 2 tiles are gate columns, the others the up columns of the same elements
  const int n0 = col * (GATED ? S::BN / 2 : S::BN);
  f32x16 acc[TM][TN];
  const bool works = (int)(threadIdx.x / WAVE) / WN * TM * 32 < rows;
  auto a_row = [&](int m) { return x + (size_t)(pairs[m] / a.top) * a.ldx; };
  auto w_row = [&](int n) {
    const int t = n / 32;
    const bool up = GATED && t % TN >= TN / 2;
    const int c = n0 + (GATED ? ((t / TN) * (TN / 2) + t % (TN / 2)) * 32 + n % 32 : n);
    return (up ? wu : wg) + (size_t)(c < a.N ? c : 0) * a.K;
  };
  const int first = expert_first_step(e, a.K);
  if (expert_reads_once<S::BM>(a, max_tiles, col_blocks, tile, e))
    tile_product_lds<WM, WN, TM, TN, ST, true, (TM * WM > 1)>(a_row, w_row, a.K, lds, acc, works, first);
  else
    tile_product_lds<WM, WN, TM, TN, ST, false, (TM * WM > 1)>(a_row, w_row, a.K, lds, acc, works, first);
  if ((int)threadIdx.x < S::BM) scales[threadIdx.x] = own_scale;
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int i = 0; i < TM; ++i) {
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int m = ((wave / WN) * TM + i) * 32 + 8 * (v / 4) + 4 * (lane >> 5) + v % 4;
      if (m >= rows) continue;
      const float sc = scales[m];
      bf16* to = (bf16*)a.y + (size_t)(start + m) * a.N;
      if constexpr (GATED) {
#pragma unroll
        for (int j = 0; j < TN / 2; ++j) {
          const int n = n0 + ((wave % WN) * (TN / 2) + j) * 32 + (lane & 31);
          if (n < a.N) to[n] = (bf16)clamp_gated(acc[i][j][v] * sc, acc[i][TN / 2 + j][v] * sc, a.limit, a.alpha, a.shift);
        }
      } else {
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          const int n = n0 + ((wave % WN) * TN + j) * 32 + (lane & 31);
          if (n < a.N) to[n] = (bf16)fms_activate(acc[i][j][v] * sc, a.act);
        }
      }
    }
  }
}

template <int WM, int WN, int TM, int TN, int ST>
__global__ void __launch_bounds__(WM* WN* WAVE) __attribute__((amdgpu_waves_per_eu(2))) expert_down_lds_kernel(ExpertArgs a, int max_tiles, int col_blocks) {
  typedef TileLds<WM, WN, TM, TN, ST> S;
  __shared__ __attribute__((aligned(16))) bf16 lds[S::LDS_ELEMENTS];
  __shared__ int pairs[S::BM];  // of the tile's rows
  int tile, col;
  if (!expert_place(a, max_tiles, col_blocks, tile, col)) return;
  const int e = uniform_load(a.tiles + 3 * tile), start = uniform_load(a.tiles + 3 * tile + 1), rows = uniform_load(a.tiles + 3 * tile + 2);
  const int own_pair = (int)threadIdx.x < S::BM ? a.order[start + ((int)threadIdx.x < rows ? threadIdx.x : 0)] : 0;
  const int n0 = col * S::BN;
  const bf16* x = (const bf16*)a.x;
  const bf16* w = (const bf16*)a.w1 + (size_t)e * a.N * a.K;
  f32x16 acc[TM][TN];
  const bool works = (int)(threadIdx.x / WAVE) / WN * TM * 32 < rows;
  auto a_row = [&](int m) { return x + (size_t)(start + (m < rows ? m : 0)) * a.ldx; };
  auto w_row = [&](int n) { return w + (size_t)(n0 + n < a.N ? n0 + n : 0) * a.K; };
  const int first = expert_first_step(e, a.K);
  if (expert_reads_once<S::BM>(a, max_tiles, col_blocks, tile, e))
    tile_product_lds<WM, WN, TM, TN, ST, true, (TM * WM > 1)>(a_row, w_row, a.K, lds, acc, works, first);
  else
    tile_product_lds<WM, WN, TM, TN, ST, false, (TM * WM > 1)>(a_row, w_row, a.K, lds, acc, works, first);
  if ((int)threadIdx.x < S::BM) pairs[threadIdx.x] = own_pair;
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int i = 0; i < TM; ++i) {
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int m = ((wave / WN) * TM + i) * 32 + 8 * (v / 4) + 4 * (lane >> 5) + v % 4;
      if (m >= rows) continue;
      float* to = (float*)a.y + (size_t)pairs[m] * a.N;
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int n = n0 + ((wave % WN) * TN + j) * 32 + (lane & 31);
        if (n < a.N) to[n] = acc[i][j][v];
      }
    }
  }
}

template <int WM, int WN, int TM, int TN, int ST>
static int launch_lds(int stage, const ExpertArgs& a, int max_tiles, hipStream_t stream) {
  typedef TileLds<WM, WN, TM, TN, ST> S;
  const int col_blocks = ceil_div(a.N, stage == 0 && a.w2 != nullptr ? S::BN / 2 : S::BN);
  // (a launch's threads are counted in 32 bits)
  FMS_REQUIRE((long)max_tiles * col_blocks <= 0xffffffffL / S::THREADS - 8, "moe_experts: %d tiles of %d columns are too many for one launch", max_tiles, a.N);
  const int blocks = 8 * ceil_div((long)max_tiles * col_blocks, 8);
  if (stage == 1)
    expert_down_lds_kernel<WM, WN, TM, TN, ST><<<blocks, S::THREADS, 0, stream>>>(a, max_tiles, col_blocks);
  else if (a.w2 != nullptr)
    expert_gate_up_lds_kernel<WM, WN, TM, TN, ST, true><<<blocks, S::THREADS, 0, stream>>>(a, max_tiles, col_blocks);
  else
    expert_gate_up_lds_kernel<WM, WN, TM, TN, ST, false><<<blocks, S::THREADS, 0, stream>>>(a, max_tiles, col_blocks);
  return 0;
}

// stage 0: hidden = act(x Wg^T, x Wu^T) for the tiles' rows; stage 1: y = hidden Wd^T
// tile_rows: what fmsamd_moe_tile_rows said when the tiles were made
extern "C" int fmsamd_moe_experts(int stage, const void* x, long ldx, const void* w1, const void* w2, void* y, int dtype,
                                  const int* order, const int* tiles, int max_tiles, int tile_rows, int top, int N, int K,
                                  float limit, float alpha, float shift, const float* in_scale, int act, hipStream_t stream) {
  if (max_tiles == 0) return 0;
  FMS_REQUIRE(act >= 0 && act <= FMS_ACT_LAST, "moe_experts: unknown activation %d", act);
  FMS_REQUIRE(stage == 0 || stage == 1, "moe_experts: stage %d", stage);
  FMS_REQUIRE(tile_rows == TILE_ROWS || tile_rows == TILE_SMALL_ROWS || tile_rows == TILE_BIG_ROWS, "moe_experts: tiles of %d rows", tile_rows);
  FMS_REQUIRE(max_tiles > 0 && top > 0 && N > 0 && K > 0 && ldx >= K, "moe_experts: bad sizes tiles=%d top=%d N=%d K=%d ldx=%ld", max_tiles,
              top, N, K, ldx);
  ExpertArgs a{x, ldx, w1, w2, y, order, tiles, top, N, K, limit, alpha, shift, stage == 0 ? in_scale : nullptr, act};
  const bool mfma = dtype == FMS_BF16 && K % 8 == 0 && ldx % 8 == 0 && ((uintptr_t)x % 16) == 0 && ((uintptr_t)w1 % 16) == 0 &&
                    (w2 == nullptr || ((uintptr_t)w2 % 16) == 0);
  const dim3 grid(max_tiles, ceil_div(N, TILE_FMA_COLS));
  FMS_REQUIRE(grid.y <= 65535, "moe_experts: %d columns are too many for one launch", N);
  if (tile_rows != TILE_ROWS) {
    // the larger tiles are made for the matrix-core kernels only
    FMS_REQUIRE(mfma, "moe_experts: tiles of %d rows need bfloat16 rows aligned to 16 bytes", tile_rows);
    const int st = tile_rows == TILE_BIG_ROWS ? launch_lds<4, 2, 1, 4, 3>(stage, a, max_tiles, stream)
                                              : launch_lds<1, 1, 1, 2, 3>(stage, a, max_tiles, stream);
    if (st) return st;
  } else if (dtype == FMS_F32) {
    if (stage == 0) expert_gate_up_fma_kernel<float><<<grid, TILE_THREADS, 0, stream>>>(a);
    else expert_down_fma_kernel<float><<<grid, TILE_THREADS, 0, stream>>>(a);
  } else if (dtype == FMS_BF16) {
    if (stage == 0) expert_gate_up_fma_kernel<bf16><<<grid, TILE_THREADS, 0, stream>>>(a);
    else expert_down_fma_kernel<bf16><<<grid, TILE_THREADS, 0, stream>>>(a);
  } else {
    FMS_REQUIRE(false, "moe_experts: unknown dtype %d", dtype);
  }
  FMS_LAUNCH_CHECK("moe_experts");
  return 0;
}

// --------------------------------------------------------------------------
// combine
// --------------------------------------------------------------------------
template <typename T>
__global__ void __launch_bounds__(256)
    combine_kernel(const float* __restrict__ y, const float* __restrict__ weights, int top, const T* __restrict__ shared,
                   const float* __restrict__ shared_gate, long ldg, T* __restrict__ out, int width, const int* __restrict__ ids,
                   int n_experts, const T* __restrict__ x_in, long ldx) {
  const int t = blockIdx.x;
  const float sg = shared ? (shared_gate ? 1.f / (1.f + expf(-shared_gate[(size_t)t * ldg])) : 1.f) : 0.f;
  for (int i = threadIdx.x; i < width; i += blockDim.x) {
    float v = 0.f;
    for (int j = 0; j < top; ++j) {
      // a choice past the experts is an identity expert: its output is the token's input
      const bool same = ids != nullptr && ids[(size_t)t * top + j] >= n_experts;
      const float yj = same ? to_f32(x_in[(size_t)t * ldx + i]) : y[((size_t)t * top + j) * width + i];
      v = fmaf(weights ? weights[(size_t)t * top + j] : 1.f, yj, v);
    }
    if (shared) v = fmaf(sg, to_f32(shared[(size_t)t * width + i]), v);
    out[(size_t)t * width + i] = from_f32<T>(v);
  }
}

// The same for rows of at most 1024 * KEEP elements (a multiple of 4): a thread's elements wait in registers, four a
// load, and every choice's row is asked for at once, so the kernel pays the memory's latency once a choice instead of
// once an element and choice.
template <typename T, int KEEP>
__global__ void __launch_bounds__(256)
    combine_small_kernel(const float* __restrict__ y, const float* __restrict__ weights, int top, const T* __restrict__ shared,
                         const float* __restrict__ shared_gate, long ldg, T* __restrict__ out, int width, const int* __restrict__ ids,
                         int n_experts, const T* __restrict__ x_in, long ldx) {
  const int t = blockIdx.x;
  f32x4 acc[KEEP], sh[KEEP];
#pragma unroll
  for (int n = 0; n < KEEP; ++n) {
    const int i = (threadIdx.x + n * 256) * 4;
    acc[n] = f32x4{0.f, 0.f, 0.f, 0.f};
    sh[n] = acc[n];
    if (shared && i < width) {
      if constexpr (sizeof(T) == 4) {
        sh[n] = *reinterpret_cast<const f32x4*>(shared + (size_t)t * width + i);
      } else {
        const bf16x4 v = *reinterpret_cast<const bf16x4*>(shared + (size_t)t * width + i);
        sh[n] = f32x4{(float)v[0], (float)v[1], (float)v[2], (float)v[3]};
      }
    }
  }
  const float sg = shared ? (shared_gate ? 1.f / (1.f + expf(-shared_gate[(size_t)t * ldg])) : 1.f) : 0.f;
  for (int j = 0; j < top; ++j) {
    const float wj = weights ? weights[(size_t)t * top + j] : 1.f;  // no weights: the plain sum
    const float* row = y + ((size_t)t * top + j) * width;
    // a choice past the experts is an identity expert: its output is the token's input
    const bool same = ids != nullptr && ids[(size_t)t * top + j] >= n_experts;
#pragma unroll
    for (int n = 0; n < KEEP; ++n) {
      const int i = (threadIdx.x + n * 256) * 4;
      if (i < width) {
        f32x4 v;
        if (same) {
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = to_f32(x_in[(size_t)t * ldx + i + e]);
        } else {
          v = *reinterpret_cast<const f32x4*>(row + i);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[n][e] = fmaf(wj, v[e], acc[n][e]);
      }
    }
  }
#pragma unroll
  for (int n = 0; n < KEEP; ++n) {
    const int i = (threadIdx.x + n * 256) * 4;
    if (i < width) {
      f32x4 r;
#pragma unroll
      for (int e = 0; e < 4; ++e) r[e] = fmaf(sg, sh[n][e], acc[n][e]);
      if constexpr (sizeof(T) == 4) {
        *reinterpret_cast<f32x4*>(out + (size_t)t * width + i) = r;
      } else {
        *reinterpret_cast<bf16x4*>(out + (size_t)t * width + i) = bf16x4{(bf16)r[0], (bf16)r[1], (bf16)r[2], (bf16)r[3]};
      }
    }
  }
}

extern "C" int fmsamd_moe_combine(const float* y, const float* weights, int top, const void* shared, const float* shared_gate,
                                  long ldg, void* out, int dtype, int n_tokens, int width, const int* ids, int n_experts,
                                  const void* x_in, long ldx, hipStream_t stream) {
  if (n_tokens == 0) return 0;
  FMS_REQUIRE(n_tokens > 0 && top > 0 && width > 0, "moe_combine: bad sizes T=%d top=%d width=%d", n_tokens, top, width);
  FMS_REQUIRE(ids == nullptr || (x_in != nullptr && ldx >= width && n_experts >= 0), "moe_combine: identity experts need the tokens' inputs");
  if (width <= 1024 * 4 && width % 4 == 0 && dtype == FMS_F32)
    combine_small_kernel<float, 4><<<n_tokens, 256, 0, stream>>>(y, weights, top, (const float*)shared, shared_gate, ldg, (float*)out, width, ids, n_experts, (const float*)x_in, ldx);
  else if (width <= 1024 * 4 && width % 4 == 0 && dtype == FMS_BF16)
    combine_small_kernel<bf16, 4><<<n_tokens, 256, 0, stream>>>(y, weights, top, (const bf16*)shared, shared_gate, ldg, (bf16*)out, width, ids, n_experts, (const bf16*)x_in, ldx);
  else if (dtype == FMS_F32)
    combine_kernel<float><<<n_tokens, 256, 0, stream>>>(y, weights, top, (const float*)shared, shared_gate, ldg, (float*)out, width, ids, n_experts, (const float*)x_in, ldx);
  else if (dtype == FMS_BF16)
    combine_kernel<bf16><<<n_tokens, 256, 0, stream>>>(y, weights, top, (const bf16*)shared, shared_gate, ldg, (bf16*)out, width, ids, n_experts, (const bf16*)x_in, ldx);
  else
    FMS_REQUIRE(false, "moe_combine: unknown dtype %d", dtype);
  FMS_LAUNCH_CHECK("moe_combine");
  return 0;
}
