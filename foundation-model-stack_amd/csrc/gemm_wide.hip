// bfloat16 products y = x W^T for 17 to 192 rows of x, weights [rows, K] with K contiguous.
//
// With this many rows of x the activations are no longer small beside the weights: a block that owns 16 weight rows and all
// of K (gemm.hip) reads four times as many bytes of x as of W.  Here a block owns up to 128 weight rows and a slice of K, and
// its waves share the x rows of the slice through LDS, so x is read once per 128 weight rows.  When K has to be cut into
// slices to fill the compute units, the slices meet in memory: the product kernel leaves float32 partial sums in a workspace,
// and a second kernel adds them in a fixed order (the same bits whatever the launch looks like) and applies the epilogue.
// A product with enough weight rows for one slice (the gated feed-forward product, the output head) is finished by the
// product kernel itself.
//
// The rows go from memory straight into LDS, several steps of 64 k-values ahead (tile_product_lds.h has the layout), and the
// products are 32x32x16 matrix instructions on tiles of 32 weight rows and 32 rows of x.  What bounds a block is what its
// compute unit can take in: its weight rows and, out of L2, the rows of x; from three tiles of x on, the operands' way from LDS
// to the matrix units.  Measured beside the kernel that came before (rows through registers, 16x16x32 products), 64 rows of x:
// the gated product of 14336 columns and K = 4096 in 42.7 us (5.5 TB/s of weights) against 46.7, an output head of 128256
// rows in 187 against 202, 4096 rows of K = 14336 with their finish in 31 against 35.  The weights are loaded as bytes that
// nobody reads again; without that mark the gated product takes 47.2 us and the long K 32.8.  Steps of 128 k-values, half as
// many deep, take 45.0 for the gated product.
#include "gemm_epilogue.h"
#include "tile_product_lds.h"

#define WD_ROWS 128   // weight rows per block
#define WD_GROUP 128  // k-values a slice of K is a multiple of (the last one may be shorter)
#define WD_COMPUTE_UNITS 256
#define WD_MAX_ROWS FMS_SKINNY_MAX_ROWS  // rows of x: six tiles of 32
#define WD_TILE_LD 132   // floats per row of the block's result tile in LDS: 128 and a shift of the banks

// What the product kernel does with its block's result tile.
#define WD_PARTIAL 0  // a slice of K: float32 partial sums into the workspace
#define WD_PLAIN 1    // all of K: row scale, bias, store
#define WD_GATED 2    // all of K; the block owns 64 gate rows and their 64 up rows: act(gate) * up

struct WideOut {
  void* out;
  long ldo;
  const void* bias;
  int bias_f32;
  int N, tile2_offset;
  OutAct act;
  int own;  // weight rows a block owns, a multiple of 4, at most WD_ROWS (WD_GATED: gate rows, and as many up rows)
  int aligned;  // x and w start at 16-byte addresses (their rows are multiples of 16 bytes apart)
  int vec;  // rows of the destination start 16-byte aligned: four elements at a time
  RowScale scale;
};

__device__ __forceinline__ float wide_bias(const WideOut& o, int n) {
  return o.bias_f32 ? ((const float*)o.bias)[n] : to_f32(((const bf16*)o.bias)[n]);
}
__device__ __forceinline__ void store4(float* p, f32x4 v) { *reinterpret_cast<f32x4*>(p) = v; }
__device__ __forceinline__ void store4(bf16* p, f32x4 v) {
  const bf16x4 b = {(bf16)v[0], (bf16)v[1], (bf16)v[2], (bf16)v[3]};
  *reinterpret_cast<bf16x4*>(p) = b;
}

// MT: tiles of 32 rows of x.  The waves form four rows of two: a pair shares 32 weight rows and deals the tiles of x between
// its two waves.  STAGES steps of rows in LDS, as many as fit.  FOLD: every group of WD_GROUP k-values is a sum of its own, and
// the groups are added up in their order (wide_plan says when).
template <int MT, int MODE, typename OutT, bool FOLD>
__global__ void __launch_bounds__(512)
    wide_kernel(const bf16* __restrict__ x, long ldx, const bf16* __restrict__ w, float* __restrict__ part, int M,
                int rows, int K, int groups_per_slice, WideOut o) {
  constexpr int BK = TL_BK;  // k-values per step of the stream
  constexpr int XROWS = MT * 32;
  constexpr int STAGE = (XROWS + WD_ROWS) * BK;  // elements: the step's rows of x, then the block's weight rows
  constexpr int STAGES = 160 * 1024 / (STAGE * 2) < 7 ? 160 * 1024 / (STAGE * 2) : 7;
  constexpr int TILE_BYTES = XROWS * WD_TILE_LD * 4;  // the block's results, once the stream has ended
  // The rows' scales (1 / rms, if the norm of x was left to this product) are worked out while the first loads are
  // under way, kept one a lane, and put into LDS behind the result tile when the stream has ended.
  constexpr int STREAM_BYTES = STAGES * STAGE * 2;
  constexpr int SMEM = STREAM_BYTES > TILE_BYTES + XROWS * 4 ? STREAM_BYTES : TILE_BYTES + XROWS * 4;
  static_assert(SMEM <= 160 * 1024, "the stream's buffers must fit the LDS of a compute unit");
  __shared__ __attribute__((aligned(16))) char smem[SMEM];
  float* const row_scale = reinterpret_cast<float*>(smem + TILE_BYTES);
  float my_scale = 1.f;  // of row wave * RPW + lane, for lane < RPW
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), lane = threadIdx.x & (WAVE - 1);
  float* const tile = reinterpret_cast<float*>(smem);
  const int li = lane & 31, kb = lane >> 5;     // the lane's row of a 32-row tile and its half of a product's 16 values
  const int pair = wave >> 1, side = wave & 1;  // the wave's row of waves, and which of its two waves it is

  // what the wave loads of a step: RX instructions of 8 rows of x (with few rows some waves load the same ones) and RW of 8
  // weight rows.  Which piece of its row a lane asks for is swizzled with half the row's number (tile_product_lds.h; the groups of 8 rows that a
  // wave loads are all even or all odd ones); a row that is not there is one that is.
  constexpr int GX = XROWS / 8, RX = (GX + 7) / 8, RW = WD_ROWS / 64, R = RX + RW;
  const int lrow = lane >> 3, piece = (lane & 7) ^ ((wave & 1) * 4 + (lrow >> 1));
  static_assert(GX % 2 == 0, "even groups of rows of x stay even");
  const bf16* src[R];
  unsigned put[R];
  const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) char*)smem;
#pragma unroll
  for (int i = 0; i < RX; ++i) {
    const int gr = (wave + i * 8) % GX, m = gr * 8 + lrow;
    src[i] = x + (size_t)(m < M ? m : M - 1) * ldx + piece * 8;
    put[i] = lds0 + gr * 8 * BK * 2;
  }
#pragma unroll
  for (int i = 0; i < RW; ++i) {
    const int gr = wave + i * 8, row = gr * 8 + lrow;
    // (the places behind the rows that the block owns take its last row again: their results are not stored)
    const int r = MODE == WD_GATED ? row & 63 : row;  // WD_GATED: 64 places for gate rows and 64 for their up rows
    int n = (int)blockIdx.x * o.own + (r < o.own ? r : o.own - 1);
    if (MODE == WD_GATED) n = (n < o.N ? n : o.N - 1) + (row < 64 ? 0 : o.tile2_offset);
    src[RX + i] = w + (size_t)(n < rows ? n : rows - 1) * K + piece * 8;
    put[RX + i] = lds0 + (XROWS + gr * 8) * BK * 2;
  }

  const int ngroups = (K + BK - 1) / BK, per_slice = groups_per_slice * (WD_GROUP / BK);
  const int g_begin = blockIdx.y * per_slice;
  const int g_end = g_begin + per_slice < ngroups ? g_begin + per_slice : ngroups;
  // The blocks walk their slice from different starting steps and wrap around: blocks that all read the same
  // bytes of their rows at the same time (rows lie a multiple of kilobytes apart) crowd into few memory
  // channels.  The start depends on the block's place only, so the order of the sum does too.
  const int n_steps = g_end - g_begin;
  // (by whole groups; the groups that are folded keep their order)
  const int rot = FOLD ? 0 : WD_GROUP / BK * ((blockIdx.x * 5) % ((n_steps + WD_GROUP / BK - 1) / (WD_GROUP / BK)));
  auto fetch = [&](int t, int stage) {  // past the end: zeros, so that every step has the same number of loads under way
    const int u = t + rot;
    const int k0 = (g_begin + (u >= n_steps ? u - n_steps : u)) * BK;
    const unsigned to = stage * (STAGE * 2);
    if (t < n_steps && k0 + BK <= K) {  // uniform
#pragma unroll
      for (int i = 0; i < RX; ++i) load_to_lds(src[i] + k0, put[i] + to);
#pragma unroll
      for (int i = RX; i < R; ++i) load_once_to_lds(src[i] + k0, put[i] + to);
    } else {
      const bool in = t < n_steps && k0 + piece * 8 < K;
#pragma unroll
      for (int i = 0; i < R; ++i) load_to_lds(in ? (const void*)(src[i] + k0) : (const void*)tile_zeros, put[i] + to);
    }
  };

  // The way straight to LDS wants 16-byte addresses.  Where x or w starts at another one the rows go through registers, AHEAD steps
  // before they are put into LDS: 33 rows of such x by 4096 and 28672 weight rows of K = 4096 17 and 49 us (24 and 79 with every step's
  // loads waited for; 14 for the first where both are aligned).
  constexpr int AHEAD = 3;
  bf16x8 held[AHEAD][R];
  auto ask = [&](int t, bf16x8 (&to)[R]) {
    const int u = t + rot;
    const int k0 = (g_begin + (u >= n_steps ? u - n_steps : u)) * BK;
    const bool in = t < n_steps && k0 + piece * 8 < K;
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const bf16x8* const from = reinterpret_cast<const bf16x8*>(in ? src[i] + k0 : (const bf16*)tile_zeros);
      to[i] = i < RX ? *from : __builtin_nontemporal_load(from);
    }
  };
  auto put_held = [&](int stage, const bf16x8 (&of)[R]) {
#pragma unroll
    for (int i = 0; i < R; ++i) *reinterpret_cast<bf16x8*>(smem + (put[i] - lds0) + stage * (STAGE * 2) + lane * 16) = of[i];
  };

  constexpr int NT = (MT + 1) / 2;  // tiles of x a wave takes at most (tiles side, side + 2, ...)
  f32x16 acc[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[j][v] = 0.f;
  f32x16 folded[FOLD ? NT : 1];  // the groups before this one
#pragma unroll
  for (int j = 0; j < (FOLD ? NT : 1); ++j) folded[j] = acc[0];

  if (o.aligned) {  // uniform
#pragma unroll
    for (int s = 0; s < STAGES - 1; ++s) fetch(s, s);
  } else {
#pragma unroll
    for (int d = 0; d < AHEAD; ++d) ask(d, held[d]);
  }
  constexpr int RPW = MT * 4;  // rows a wave works out the scale of
  if (MODE != WD_PARTIAL) {
    // 1 / rms of the rows of x, if their norm was left to this product.  The partial sums are asked for behind the
    // stream's first loads and all at once.
    constexpr int PRE = MT > 4 ? 2 : 4;  // loads a row that are under way together
    if (o.scale.partials != nullptr) {
      float pre[RPW][PRE];
#pragma unroll
      for (int k = 0; k < RPW; ++k)
#pragma unroll
        for (int j = 0; j < PRE; ++j) {
          const int m = wave * RPW + k < M ? wave * RPW + k : M - 1, i = lane + j * WAVE;
          pre[k][j] = o.scale.partials[(size_t)m * o.scale.count + (i < o.scale.count ? i : 0)];
        }
#pragma unroll
      for (int k = 0; k < RPW; ++k) {
        const int m = wave * RPW + k < M ? wave * RPW + k : M - 1;
        float sum = 0.f;
#pragma unroll
        for (int j = 0; j < PRE; ++j) sum += lane + j * WAVE < o.scale.count ? pre[k][j] : 0.f;
        for (int i = lane + PRE * WAVE; i < o.scale.count; i += WAVE) sum += o.scale.partials[(size_t)m * o.scale.count + i];
        const float total = wave_sum(sum);
        if (lane == k) my_scale = rsqrtf(total * o.scale.inv_width + o.scale.eps);
      }
    }
  }
  auto multiply = [&](int t, int stage) {
    const bf16* const xs = reinterpret_cast<const bf16*>(smem) + stage * STAGE;
    const bf16* const ws = xs + (XROWS + pair * 32) * BK;
    auto operand = [&](const bf16* rows32, int st) {
      return *reinterpret_cast<const bf16x8*>(rows32 + li * BK + ((st * 2 + kb) ^ ((li >> 1) & 7)) * 8);
    };
    bf16x8 a[4];
#pragma unroll
    for (int st = 0; st < 4; ++st) a[st] = operand(ws, st);
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      if (side + 2 * j < MT) {  // uniform over the wave
        bf16x8 b[4];
#pragma unroll
        for (int st = 0; st < 4; ++st) b[st] = operand(xs + (side + 2 * j) * 32 * BK, st);
#pragma unroll
        for (int st = 0; st < 4; ++st) acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[st], b[st], acc[j], 0, 0, 0);
      }
    }
    if (FOLD && ((t + 1) % (WD_GROUP / BK) == 0 || t + 1 == n_steps)) {  // uniform
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) folded[j][v] += acc[j][v], acc[j][v] = 0.f;
    }
  };
  if (o.aligned) {  // uniform
    int stage = 0;
    for (int t = 0; t < n_steps; ++t) {
      tile_wait<(STAGES - 2) * R>();  // step t is there, and everybody is done with step t - 1
      fetch(t + STAGES - 1, stage == 0 ? STAGES - 1 : stage - 1);
      multiply(t, stage);
      stage = stage == STAGES - 1 ? 0 : stage + 1;
    }
  } else {
    put_held(0, held[0]);
    ask(AHEAD, held[0]);
    block_sync_lds();
    for (int t0 = 0; t0 < n_steps; t0 += AHEAD) {
#pragma unroll
      for (int d = 0; d < AHEAD; ++d) {
        // step t + 1 into the buffer that step t - 1 was in; loads and stores stand behind no branch, so that the compiler can wait
        // for the oldest loads alone (steps past the end are zeros)
        const int t = t0 + d;
        put_held((t + 1) & 1, held[(d + 1) % AHEAD]);
        ask(t + 1 + AHEAD, held[(d + 1) % AHEAD]);
        if (t < n_steps) multiply(t, t & 1);  // uniform
        block_sync_lds();
      }
    }
  }
  if (FOLD) {
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[j] = folded[j];
  }
  tile_wait<0>();  // nothing is on its way to LDS any more, and everybody has read the last step

  // The block's results meet in LDS (where the stream's buffers were): row m of x, then the block's 128
  // weight rows in their order; from there they leave in whole rows of 256 or 512 bytes.
  // acc[j][v]: x row 32 (side + 2 j) + li, the pair's weight row 8 (v / 4) + 4 kb + v % 4
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    const int jt = side + 2 * j;
    if (jt < MT)
#pragma unroll
      for (int u = 0; u < 4; ++u)
        *reinterpret_cast<f32x4*>(tile + (jt * 32 + li) * WD_TILE_LD + pair * 32 + 8 * u + 4 * kb) =
            f32x4{acc[j][4 * u], acc[j][4 * u + 1], acc[j][4 * u + 2], acc[j][4 * u + 3]};
  }
  if (MODE != WD_PARTIAL && lane < RPW) row_scale[wave * RPW + lane] = my_scale;
  __syncthreads();

  if (MODE == WD_GATED) {
    // 16 threads a row: four gate columns and their four up columns each
    const int c = 4 * (threadIdx.x & 15);
    const int n = blockIdx.x * o.own + c;
    const int n_hi = ((int)blockIdx.x + 1) * o.own < o.N ? ((int)blockIdx.x + 1) * o.own : o.N;
    OutT* const out = (OutT*)o.out;
#pragma unroll
    for (int p = 0; p < MT; ++p) {
      const int m = p * 32 + (threadIdx.x >> 4);
      if (m >= M || n >= n_hi) continue;
      const f32x4 gate = *reinterpret_cast<const f32x4*>(tile + m * WD_TILE_LD + c);
      const f32x4 up = *reinterpret_cast<const f32x4*>(tile + m * WD_TILE_LD + WD_ROWS / 2 + c);
      const float rs = row_scale[m];
      f32x4 res;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float v = gate[e] * rs, u = up[e] * rs;
        if (o.bias != nullptr && n + e < n_hi) {
          v += wide_bias(o, n + e);
          u += wide_bias(o, o.tile2_offset + n + e);
        }
        res[e] = sk_gated(v, u, o.act);
      }
      if (o.vec && n + 3 < n_hi) {
        store4(out + (size_t)m * o.ldo + n, res);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + e < n_hi) out[(size_t)m * o.ldo + n + e] = from_f32<OutT>(res[e]);
      }
    }
  } else {
    // 32 threads a row: four columns each
    const int c = 4 * (threadIdx.x & 31);
    const int n = blockIdx.x * o.own + c;
    const int n_lim = ((int)blockIdx.x + 1) * o.own < rows ? ((int)blockIdx.x + 1) * o.own : rows;
#pragma unroll
    for (int p = 0; p < 2 * MT; ++p) {
      const int m = p * 16 + (threadIdx.x >> 5);
      if (m >= M || n >= n_lim) continue;
      f32x4 v = *reinterpret_cast<const f32x4*>(tile + m * WD_TILE_LD + c);
      if (MODE == WD_PLAIN) {
        const float rs = row_scale[m];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          v[e] *= rs;
          if (o.bias != nullptr && n + e < n_lim) v[e] += wide_bias(o, n + e);
          v[e] = sk_plain(v[e], o.act.kind);
        }
        OutT* const out = (OutT*)o.out;
        if (o.vec && n + 3 < n_lim) {
          store4(out + (size_t)m * o.ldo + n, v);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (n + e < n_lim) out[(size_t)m * o.ldo + n + e] = from_f32<OutT>(v[e]);
        }
      } else {
        float* const dst = part + ((size_t)blockIdx.y * M + m) * rows + n;
        if (o.vec && n + 3 < n_lim) {
          store4(dst, v);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (n + e < n_lim) dst[e] = v[e];
        }
      }
    }
  }
}

// One wave per row m and 64 columns: adds the slices and finishes the element as the epilogue says.
template <int EPI, typename OutT, typename BiasT>
__global__ void __launch_bounds__(256)
    wide_finish_kernel(const float* __restrict__ part, int slices, int rows, const BiasT* __restrict__ bias,
                       OutT* __restrict__ out, long ldo, int M, int N, int tile2_offset, OutAct act, RowScale scale,
                       RopeEpilogue rope, ResidEpilogue res) {
  const int wave = threadIdx.x / WAVE, lane = threadIdx.x & (WAVE - 1);
  const int m = blockIdx.y * 4 + wave;
  const int n = blockIdx.x * WAVE + lane;
  if (m >= M) return;  // whole waves
  const bool live = n < N;
  const int nn = live ? n : 0;  // a lane past the end reads column 0 and stores nothing

  // Every load that does not wait for another one's result is asked for here, at once and not behind a branch:
  // the first slices, the partial sums of the rows' norm, the row's position and sequence, the stream and the next
  // norm's weight.  One after the other they were six to eight round trips to memory for a kernel that moves a
  // few megabytes.  What is out of range is read from a valid address and set aside where it is used.
  constexpr int FIRST = 8, PRE = 4;
  const size_t stride = (size_t)M * rows;
  const float* const pv = part + (size_t)m * rows + nn;
  const float* const pu = pv + tile2_offset;
  float av[FIRST], au[FIRST], pre[PRE];  // au: the up half of a gated product, unused otherwise
#pragma unroll
  for (int s = 0; s < FIRST; ++s) {
    const size_t at = (size_t)(s < slices ? s : 0) * stride;
    av[s] = pv[at];
    if (EPI == EPI_GATED) au[s] = pu[at];
  }
  if (scale.partials != nullptr) {  // uniform
#pragma unroll
    for (int j = 0; j < PRE; ++j) {
      const int i = lane + j * WAVE;
      pre[j] = scale.partials[(size_t)m * scale.count + (i < scale.count ? i : 0)];
    }
  }
  int pos = 0, seq = -1;
  if (EPI == EPI_ROPE) pos = rope.positions[m], seq = rope.seq_of_token[m];
  float stream_in = 0.f, nw = 1.f, bias_v = 0.f, bias_u = 0.f;
  if (EPI == EPI_RESID) {
    stream_in = res.resid[(size_t)m * res.ldr + nn];
    if (res.norm_w != nullptr) nw = res.norm_w_f32 ? ((const float*)res.norm_w)[nn] : to_f32(((const bf16*)res.norm_w)[nn]);
  }
  if (bias) {
    bias_v = to_f32(bias[nn]);
    if (EPI == EPI_GATED) bias_u = to_f32(bias[tile2_offset + nn]);
  }

  // The slices are added in their order, whatever the launch looks like.
  auto add_slices = [&](const float* p, const float (&first)[FIRST]) {
    float sum = 0.f;
#pragma unroll
    for (int s = 0; s < FIRST; ++s)
      if (s < slices) sum += first[s];
    int s = FIRST;
    for (; s + 4 <= slices; s += 4) {
      const float a0 = p[(size_t)s * stride], a1 = p[(size_t)(s + 1) * stride], a2 = p[(size_t)(s + 2) * stride],
                  a3 = p[(size_t)(s + 3) * stride];
      sum = (((sum + a0) + a1) + a2) + a3;
    }
    for (; s < slices; ++s) sum += p[(size_t)s * stride];
    return sum;
  };
  float v = add_slices(pv, av), u = 0.f;
  if (EPI == EPI_GATED) u = add_slices(pu, au);
  float row_scale = 1.f;
  if (scale.partials != nullptr) {
    float sum = 0.f;
#pragma unroll
    for (int j = 0; j < PRE; ++j) sum += lane + j * WAVE < scale.count ? pre[j] : 0.f;
    for (int i = lane + PRE * WAVE; i < scale.count; i += WAVE) sum += scale.partials[(size_t)m * scale.count + i];
    row_scale = rsqrtf(wave_sum(sum) * scale.inv_width + scale.eps);
  }
  v *= row_scale;
  u *= row_scale;

  if (EPI == EPI_GATED) {
    if (!live) return;
    out[(size_t)m * ldo + n] = from_f32<OutT>(sk_gated(v + bias_v, u + bias_u, act));
  } else if (EPI == EPI_ROPE) {
    v += bias_v;
    const float partner = __shfl_xor(v, 1, WAVE);  // the other element of the rotary pair (N is even)
    if (!live) return;
    const int D = rope.head_dim;
    const int hh = n / D, d = n - hh * D;
    if (hh < rope.nheads + rope.kvheads && rope.cos_t != nullptr && d < rope.rot_dim) {
      const int tpos = pos < 0 ? 0 : (pos < rope.max_pos ? pos : rope.max_pos - 1);  // the host has checked the range
      const float c = rope.cos_t[(size_t)tpos * (rope.rot_dim / 2) + d / 2];
      const float sn = rope.sin_t[(size_t)tpos * (rope.rot_dim / 2) + d / 2];
      v = (d & 1) ? sn * partner + c * v : c * v - sn * partner;
    }
    if (hh < rope.nheads) {
      out[(size_t)m * ldo + n] = from_f32<OutT>(v);
    } else if (seq >= 0 && rope.k_cache != nullptr) {
      const int entry = rope.block_table[(size_t)seq * rope.table_stride + pos / PAGE_TOKENS];
      const size_t page = readable_page(entry);
      const size_t page_elems = (size_t)rope.kvheads * PAGE_TOKENS * D;
      const int in_page = pos % PAGE_TOKENS;
      if (entry < 0) {
        // no page for this token: nothing is written
      } else if (hh < rope.nheads + rope.kvheads) {
        const int kh = hh - rope.nheads;
        rope.k_cache[page * page_elems + ((size_t)kh * PAGE_TOKENS + in_page) * D + d] = (bf16)v;
      } else {
        const int kh = hh - rope.nheads - rope.kvheads;
        rope.v_cache[page * page_elems + ((size_t)kh * D + d) * PAGE_TOKENS + in_page] = (bf16)v;
      }
    }
  } else if (EPI == EPI_RESID) {
    float stream = 0.f;
    if (live) {
      stream = stream_in + (v + bias_v);
      res.resid[(size_t)m * res.ldr + n] = stream;
      out[(size_t)m * ldo + n] = from_f32<OutT>(stream * nw);
    }
    float sq = stream * stream;  // sums over the groups of 16 neighbouring columns
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) sq += __shfl_xor(sq, off, WAVE);
    if ((lane & 15) == 0 && n / 16 < res.tiles) res.partials[(size_t)m * res.tiles + n / 16] = sq;
  } else {
    if (!live) return;
    out[(size_t)m * ldo + n] = from_f32<OutT>(sk_plain(v + bias_v, act.kind));
  }
}

// How a product is cut: weight rows a block owns, and slices of K.
struct WidePlan {
  int own, slices;
};

static bool wide_finishes_itself(int epi) { return epi == EPI_PLAIN || epi == EPI_GATED; }

// A K of up to four groups of WD_GROUP is summed as the kernel for 17 to 32 rows sums it (gemm.hip, a group to each of its
// waves): every group by itself, then the groups in their order.  One slice does that in registers (FOLD), one slice a group
// leaves it to the second kernel, and no other cut is taken.  So the products' sums are the same bits for any 17 to 192 rows, and a
// batch that shrinks below 33 rows goes on with them.  (From WD_MANY weight rows on that kernel takes no product of 17 rows or more,
// and one cut for any number of rows does it.)  With a longer K the cut, and with it the order, goes with the number of rows.
// Four groups: up to there one of those two cuts is the fastest or within a tenth of it; from six on those in between are a
// fifth faster.
#define WD_MANY 16384
static bool wide_keeps_groups(int K) { return ceil_div(K, WD_GROUP) <= 4; }

// The cut with the least estimated time.  The blocks run in rounds over the compute units; a round's time is its steps and a
// start; the partial sums of slices are written and read once, by a kernel of its own unless the product kernel finishes its
// one slice itself (with two tiles of x its blocks then take some 3 us longer than their steps say: 14336 weight rows of
// K = 4096 in one slice and in two at 33, 48 and 64 rows 34.2, 32.1, 32.3 us against 25.8, 27.2, 29.1, 7168 of K = 2048 at 64 rows 18.3
// against 15.6).  A step takes what its rows take to arrive (measured with all units at work: 28 bytes a nanosecond of
// weights for each; rows of x come out of the caches at about three times that) but never less than the operands' way from LDS
// to the matrix units (measured 0.4, 0.7 and 1.0 us for a step of one or two, three or four, five or six tiles of x).
static WidePlan wide_plan(int epi, int M, int rows, int K) {
  const int ngroups = ceil_div(K, WD_GROUP), mt = ceil_div(M, 32);
  const double busy = 0.1 + 0.3 * ((mt + 1) / 2);
  // A short K and blocks of 64 weight rows that make one round: as many slices as the round holds.  Measured at 33, 64, 128 and
  // 192 rows, in microseconds (blocks of 128 rows and a slice a group in brackets): 2048 weight rows of K = 512 6.2, 6.5, 8.1, 9.8
  // (6.7, 7.5, 9.8, 12.2), 3072 of 768 7.2, 7.7, 9.8, 12.2 (7.6, 9.3, 13.1, 17.1), 2048 of 1024 6.5, 6.9, 8.8, 11.0 (7.4, 9.0, 12.3,
  // 15.9), 16384 of 256 6.2, 6.7, 8.8, 10.9 (10.1, 13.5, 20.7, 25.9).  Blocks of 32 rows take up to a tenth longer.
  static_assert(WD_MANY <= WD_COMPUTE_UNITS * WD_ROWS / 2, "blocks of 64 rows make one round");
  const int most = WD_COMPUTE_UNITS / ceil_div(rows, WD_ROWS / 2);
  if (ngroups <= 8 && rows <= WD_MANY && (most > 1 || wide_keeps_groups(K))) {
    return {WD_ROWS / 2, most >= ngroups ? ngroups : wide_keeps_groups(K) ? 1 : most};
  }
  if (wide_keeps_groups(K)) {  // one slice, and the fewest rows a block that do not add a round
    const int rounds = ceil_div(ceil_div(rows, WD_ROWS), WD_COMPUTE_UNITS);
    return {ceil_div(ceil_div(rows, WD_COMPUTE_UNITS * rounds), 4) * 4, 1};
  }
  WidePlan best{WD_ROWS, 1};
  double best_cost = -1;
  for (int slices = 1; slices <= ngroups && slices <= 64; ++slices) {
    const int fewest = ceil_div(ceil_div(rows, WD_ROWS) * slices, WD_COMPUTE_UNITS);
    for (int rounds = fewest; rounds <= fewest + 1; ++rounds) {
      // the fewest rows a block with which the blocks make no more rounds than that
      const int blocks = WD_COMPUTE_UNITS * rounds / slices;
      if (blocks == 0) continue;
      int own = ceil_div(ceil_div(rows, blocks), 4) * 4;
      own = own < 32 ? 32 : own;
      if (own > WD_ROWS) continue;
      const double step = (own + 0.35 * 32 * mt) * (TL_BK * 2 / 28000.);
      double cost = rounds * (ceil_div(ngroups, slices) * (WD_GROUP / TL_BK) * (step > busy ? step : busy) + 3.);
      if (slices > 1 || !wide_finishes_itself(epi))
        cost += 5. + (double)slices * M * rows * 8 / 4e6;
      else if (mt == 2)
        cost += 3.;
      if (best_cost < 0 || cost < best_cost) best = {own, slices}, best_cost = cost;
    }
  }
  return best;
}

// Enough for any epilogue of this shape.
long wide_workspace_bytes(int M, int rows, int K) {
  return (long)wide_plan(EPI_RESID, M, rows, K).slices * M * rows * (long)sizeof(float);
}

template <int EPI>
static void launch_finish(const float* part, int slices, int rows, const void* bias, int bias_dtype, void* out,
                          int out_dtype, long ldo, int M, int N, int tile2_offset, OutAct act, RowScale scale,
                          RopeEpilogue rope, ResidEpilogue res, hipStream_t stream) {
  dim3 grid(ceil_div(N, WAVE), ceil_div(M, 4));
  const bool fb = bias != nullptr && bias_dtype == FMS_F32;
#define FMS_WF(O, B)                                                                                             \
  wide_finish_kernel<EPI, O, B><<<grid, 256, 0, stream>>>(part, slices, rows, (const B*)bias, (O*)out, ldo, M, N, \
                                                          tile2_offset, act, scale, rope, res)
  if (out_dtype == FMS_BF16) {
    if (fb)
      FMS_WF(bf16, float);
    else
      FMS_WF(bf16, bf16);
  } else if (EPI != EPI_ROPE && EPI != EPI_RESID) {
    if (fb)
      FMS_WF(float, float);
    else
      FMS_WF(float, bf16);
  }
#undef FMS_WF
}

template <int MODE, typename OutT>
static void launch_wide(dim3 grid, const void* x, long ldx, const void* w, float* part, int M, int rows, int K,
                        int per_slice, const WideOut& o, hipStream_t stream) {
  const bool fold = per_slice > 1 && rows <= WD_MANY && wide_keeps_groups(K);
#define FMS_WK(MT)                                                                                                          \
  if (fold)                                                                                                                 \
    wide_kernel<MT, MODE, OutT, true><<<grid, 512, 0, stream>>>((const bf16*)x, ldx, (const bf16*)w, part, M, rows, K, per_slice, o); \
  else                                                                                                                      \
    wide_kernel<MT, MODE, OutT, false><<<grid, 512, 0, stream>>>((const bf16*)x, ldx, (const bf16*)w, part, M, rows, K, per_slice, o)
  switch (ceil_div(M, 32)) {
    case 1: FMS_WK(1); break;
    case 2: FMS_WK(2); break;
    case 3: FMS_WK(3); break;
    case 4: FMS_WK(4); break;
    case 5: FMS_WK(5); break;
    default: FMS_WK(6); break;
  }
#undef FMS_WK
}

static bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

// N: columns of the output (for the gated product the hidden size; W then has tile2_offset + N rows).
int wide_product(int epi, const void* x, long ldx, const void* w, const void* bias, int bias_dtype, void* out,
                 int out_dtype, long ldo, int M, int N, int K, int tile2_offset, OutAct act, RowScale scale,
                 RopeEpilogue rope, ResidEpilogue res, void* workspace, long workspace_bytes, hipStream_t stream) {
  const int rows = epi == EPI_GATED ? tile2_offset + N : N;
  FMS_REQUIRE(M > 16 && M <= WD_MAX_ROWS, "wide product: %d rows (17..%d)", M, WD_MAX_ROWS);
  const int ngroups = ceil_div(K, WD_GROUP);
  const WidePlan plan = wide_plan(epi, M, rows, K);
  const int per_slice = ceil_div(ngroups, plan.slices);
  const int slices = ceil_div(ngroups, per_slice);  // no slice without a step (the kernel divides by its steps)
  const bool itself = slices == 1 && wide_finishes_itself(epi);
  WideOut o{out, ldo, bias, bias != nullptr && bias_dtype == FMS_F32, N, tile2_offset, act, plan.own,
            aligned16(x) && aligned16(w), 0, scale};

  if (itself) {
    const long elem = out_dtype == FMS_BF16 ? 2 : 4;
    o.vec = ((uintptr_t)out % (4 * elem)) == 0 && ldo % 4 == 0;
    if (epi == EPI_GATED) {
      o.own = ceil_div(plan.own, 8) * 4;  // of each half
      dim3 grid(ceil_div(N, o.own), 1);
      if (out_dtype == FMS_BF16)
        launch_wide<WD_GATED, bf16>(grid, x, ldx, w, nullptr, M, rows, K, per_slice, o, stream);
      else
        launch_wide<WD_GATED, float>(grid, x, ldx, w, nullptr, M, rows, K, per_slice, o, stream);
    } else {
      dim3 grid(ceil_div(N, o.own), 1);
      if (out_dtype == FMS_BF16)
        launch_wide<WD_PLAIN, bf16>(grid, x, ldx, w, nullptr, M, rows, K, per_slice, o, stream);
      else
        launch_wide<WD_PLAIN, float>(grid, x, ldx, w, nullptr, M, rows, K, per_slice, o, stream);
    }
    FMS_LAUNCH_CHECK("wide product");
    return 0;
  }

  const long needed = (long)slices * M * rows * (long)sizeof(float);
  FMS_REQUIRE(workspace != nullptr && workspace_bytes >= needed, "wide product: workspace of %ld bytes, %ld needed",
              workspace_bytes, needed);
  dim3 grid(ceil_div(rows, o.own), slices);
  FMS_REQUIRE(grid.y <= 65535, "wide product: %d slices", slices);
  float* part = (float*)workspace;
  o.vec = aligned16(workspace) && rows % 4 == 0;
  launch_wide<WD_PARTIAL, float>(grid, x, ldx, w, part, M, rows, K, per_slice, o, stream);
  FMS_LAUNCH_CHECK("wide product");
  switch (epi) {
    case EPI_PLAIN:
      launch_finish<EPI_PLAIN>(part, slices, rows, bias, bias_dtype, out, out_dtype, ldo, M, N, 0, act, scale, rope, res, stream);
      break;
    case EPI_GATED:
      launch_finish<EPI_GATED>(part, slices, rows, bias, bias_dtype, out, out_dtype, ldo, M, N, tile2_offset, act, scale,
                               rope, res, stream);
      break;
    case EPI_ROPE:
      launch_finish<EPI_ROPE>(part, slices, rows, bias, bias_dtype, out, out_dtype, ldo, M, N, 0, act, scale, rope, res, stream);
      break;
    default:
      launch_finish<EPI_RESID>(part, slices, rows, bias, bias_dtype, out, out_dtype, ldo, M, N, 0, act, scale, rope, res, stream);
  }
  FMS_LAUNCH_CHECK("wide product finish");
  return 0;
}
