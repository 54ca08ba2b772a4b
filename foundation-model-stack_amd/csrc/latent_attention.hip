// Attention over a latent cache: every token leaves one row [latent (R) | rotated shared key part (P)] in the
// cache, and all query heads read that one row.  With per-head matrices Uk [D, R] (keys) and Uv [V, R] (values)
//   score(t, j, h) = (q_plain . Uk_h c_j + q_rot . k_rot_j) * scale = ((Uk_h^T q_plain) . c_j + q_rot . k_rot_j) * scale
//   out(t, h)      = Uv_h sum_j p_j c_j
// so the kernels never expand keys or values: the query goes into the latent space once per token and head, attention
// runs as one shared "kv head" with keys of R + P and values of R elements (the first R of the same row), and the
// result leaves the latent space once per token and head.  Whole prompts, portions and single tokens run the same way.
//
// The softmax may have a sink: a learned logit per head that counts once in the denominator and has no value.  It is
// the state in which the running maximum and sum start.
//
//   latent_kv_write:      RMS norm of the latent, rotation of the shared key part, row written into its page
//   latent_q_rotate:      the rotated part of every head's query into its place behind the latent part
//   headwise_linear:      y[t, h, :] = W_h x[t, h, :] (optionally times sigmoid(gate[t, h])), FMA or MFMA
//   headwise_split:       the same for few tokens, the waves of a block sharing K
//   latent_attn_generic:  float32 arithmetic on any storage type; one block per (head, token)
//   latent_attn_mfma:     bfloat16, MFMA 16x16x32; a wave owns 16 heads of one token (+ merge of partial results)
//   latent_attn_decode:   the same for single tokens with a latent of 512, whole rows of the cache straight into LDS
//   latent_attn_prompt:   the same for prompts with a latent of 512, keys and latent straight into LDS
//
// Cache layout: rows [page][token in page][R + P]; for the MFMA kernel also the latent transposed, [page][R][token in
// page], so that both products read their contraction index contiguously, straight from global memory.
#include "common.h"
#include "fmsamd.h"
#include "tile_product.h"
#include "tile_product_lds.h"

// --------------------------------------------------------------------------
// cache write
// --------------------------------------------------------------------------
template <typename CT>
__global__ void __launch_bounds__(256)
    latent_kv_write_kernel(const float* __restrict__ down, long ld, int col0, int rank, int rot, const void* __restrict__ w,
                           int w_dtype, float eps, const int* __restrict__ positions, const int* __restrict__ seq_of_token,
                           const int* __restrict__ block_table, int table_stride, const float* __restrict__ cos_t,
                           const float* __restrict__ sin_t, CT* __restrict__ cache, CT* __restrict__ vt_cache) {
  __shared__ float scratch[17];
  const int t = blockIdx.x;
  const int seq = seq_of_token[t];
  if (seq < 0) return;
  const int pos = positions[t];
  const int page = block_table[(size_t)seq * table_stride + pos / PAGE_TOKENS];
  if (page < 0) return;
  const float* x = down + (size_t)t * ld + col0;
  CT* row = cache + ((size_t)page * PAGE_TOKENS + pos % PAGE_TOKENS) * (rank + rot);
  float sq = 0.f;
  for (int i = threadIdx.x; i < rank; i += blockDim.x) sq = fmaf(x[i], x[i], sq);
  const float rs = rsqrtf(block_sum(sq, scratch) / (float)rank + eps);
  for (int i = threadIdx.x; i < rank; i += blockDim.x) {
    const float wi = w == nullptr ? 1.f : (w_dtype == FMS_F32 ? ((const float*)w)[i] : (float)((const bf16*)w)[i]);
    const CT c = from_f32<CT>(x[i] * rs * wi);
    row[i] = c;
    // the latent once more with the tokens of a page side by side, [page][rank][token]: the layout from which the
    // second product of the MFMA kernel loads its operand without a transposition
    if (vt_cache) vt_cache[((size_t)page * rank + i) * PAGE_TOKENS + pos % PAGE_TOKENS] = c;
  }
  const int half = rot / 2;
  for (int i = threadIdx.x; i < half; i += blockDim.x) {
    const float c = cos_t[(size_t)pos * half + i], s = sin_t[(size_t)pos * half + i];
    const float u = x[rank + 2 * i], v = x[rank + 2 * i + 1];
    row[rank + 2 * i] = from_f32<CT>(u * c - v * s);
    row[rank + 2 * i + 1] = from_f32<CT>(v * c + u * s);
  }
}

extern "C" int fmsamd_latent_kv_write(const float* down, long ld, int col0, int rank, int rot, const void* norm_weight,
                                      int weight_dtype, float eps, const int* positions, const int* seq_of_token,
                                      const int* block_table, int table_stride, const float* cos_t, const float* sin_t,
                                      int max_pos, void* cache, void* vt_cache, int cache_dtype, int n_tokens,
                                      hipStream_t stream) {
  if (n_tokens == 0) return 0;
  FMS_REQUIRE(n_tokens > 0 && rank > 0 && rot >= 0 && rot % 2 == 0 && col0 >= 0 && ld >= col0 + rank + rot,
              "latent_kv_write: bad sizes T=%d rank=%d rot=%d col0=%d ld=%ld", n_tokens, rank, rot, col0, ld);
  FMS_REQUIRE(rot == 0 || (cos_t != nullptr && sin_t != nullptr && max_pos > 0), "latent_kv_write: a rotation needs its tables");
  if (cache_dtype == FMS_F32)
    latent_kv_write_kernel<float><<<n_tokens, 256, 0, stream>>>(down, ld, col0, rank, rot, norm_weight, weight_dtype, eps,
                                                                positions, seq_of_token, block_table, table_stride, cos_t,
                                                                sin_t, (float*)cache, (float*)vt_cache);
  else if (cache_dtype == FMS_BF16)
    latent_kv_write_kernel<bf16><<<n_tokens, 256, 0, stream>>>(down, ld, col0, rank, rot, norm_weight, weight_dtype, eps,
                                                               positions, seq_of_token, block_table, table_stride, cos_t,
                                                               sin_t, (bf16*)cache, (bf16*)vt_cache);
  else
    FMS_REQUIRE(false, "latent_kv_write: unknown dtype %d", cache_dtype);
  FMS_LAUNCH_CHECK("latent_kv_write");
  return 0;
}

// --------------------------------------------------------------------------
// queries: q [T, H, D + P] -> qa[t, h, R : R + P] = rotate(q[t, h, D : D + P])
// --------------------------------------------------------------------------
template <typename T>
__global__ void __launch_bounds__(256)
    latent_q_rotate_kernel(const T* __restrict__ q, long ldq, int nheads, int dim, int rot, T* __restrict__ qa, long ldqa,
                           int rank, const int* __restrict__ positions, const float* __restrict__ cos_t,
                           const float* __restrict__ sin_t) {
  const int t = blockIdx.x;
  const int pos = positions[t];
  const int half = rot / 2;
  for (int i = threadIdx.x; i < nheads * half; i += blockDim.x) {
    const int h = i / half, p = i % half;
    const T* src = q + (size_t)t * ldq + (size_t)h * (dim + rot) + dim + 2 * p;
    T* dst = qa + (size_t)t * ldqa + (size_t)h * (rank + rot) + rank + 2 * p;
    const float c = cos_t[(size_t)pos * half + p], s = sin_t[(size_t)pos * half + p];
    const float u = to_f32(src[0]), v = to_f32(src[1]);
    dst[0] = from_f32<T>(u * c - v * s);
    dst[1] = from_f32<T>(v * c + u * s);
  }
}

extern "C" int fmsamd_latent_q_rotate(const void* q, long ldq, int dtype, int nheads, int dim, int rot, void* qa, long ldqa,
                                      int rank, const int* positions, const float* cos_t, const float* sin_t, int max_pos,
                                      int n_tokens, hipStream_t stream) {
  if (n_tokens == 0 || rot == 0) return 0;
  FMS_REQUIRE(n_tokens > 0 && nheads > 0 && dim >= 0 && rot > 0 && rot % 2 == 0 && rank > 0, "latent_q_rotate: bad sizes");
  FMS_REQUIRE(ldq >= (long)nheads * (dim + rot) && ldqa >= (long)nheads * (rank + rot), "latent_q_rotate: rows too short");
  FMS_REQUIRE(cos_t != nullptr && sin_t != nullptr && max_pos > 0, "latent_q_rotate: a rotation needs its tables");
  if (dtype == FMS_F32)
    latent_q_rotate_kernel<float><<<n_tokens, 256, 0, stream>>>((const float*)q, ldq, nheads, dim, rot, (float*)qa, ldqa, rank,
                                                                positions, cos_t, sin_t);
  else if (dtype == FMS_BF16)
    latent_q_rotate_kernel<bf16><<<n_tokens, 256, 0, stream>>>((const bf16*)q, ldq, nheads, dim, rot, (bf16*)qa, ldqa, rank,
                                                               positions, cos_t, sin_t);
  else
    FMS_REQUIRE(false, "latent_q_rotate: unknown dtype %d", dtype);
  FMS_LAUNCH_CHECK("latent_q_rotate");
  return 0;
}

// --------------------------------------------------------------------------
// y[t, h, n] = sum_k x[t, h, k] W[h, n, k]  (* sigmoid(gate[t, h]))
// --------------------------------------------------------------------------
struct HeadwiseArgs {
  const void* x;
  long ldx, xs;  // row stride, head stride of x (elements)
  const void* w;  // [H, N, K]
  void* y;
  long ldy, ys;
  const float* gate;  // logits [T, ldg] or null
  long ldg;
  int T, H, N, K;
};

template <typename T>
__global__ void __launch_bounds__(TILE_THREADS) headwise_fma_kernel(HeadwiseArgs a) {
  const int t0 = blockIdx.x * TILE_ROWS, h = blockIdx.y, n0 = blockIdx.z * TILE_FMA_COLS;
  const T* x = (const T*)a.x + (size_t)h * a.xs;
  const T* w = (const T*)a.w + (size_t)h * a.N * a.K;
  float acc[4];
  tile_product_fma<T>([&](int m) { return t0 + m < a.T ? x + (size_t)(t0 + m) * a.ldx : (const T*)nullptr; },
                      [&](int n) { return n0 + n < a.N ? w + (size_t)(n0 + n) * a.K : (const T*)nullptr; }, a.K, acc);
  const int n = n0 + threadIdx.x % 64;
  if (n >= a.N) return;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int t = t0 + (threadIdx.x / 64) * 4 + i;
    if (t < a.T) {
      float v = acc[i];
      if (a.gate) v *= 1.f / (1.f + expf(-a.gate[(size_t)t * a.ldg + h]));
      ((T*)a.y)[(size_t)t * a.ldy + (size_t)h * a.ys + n] = from_f32<T>(v);
    }
  }
}

__global__ void __launch_bounds__(TILE_THREADS) headwise_mfma_kernel(HeadwiseArgs a) {
  const int t0 = blockIdx.x * TILE_ROWS, h = blockIdx.y, n0 = blockIdx.z * TILE_MFMA_COLS;
  const bf16* x = (const bf16*)a.x + (size_t)h * a.xs;
  const bf16* w = (const bf16*)a.w + (size_t)h * a.N * a.K;
  f32x4 acc[TILE_MFMA_WAVE_TILES];
  tile_product_mfma([&](int m) { return t0 + m < a.T ? x + (size_t)(t0 + m) * a.ldx : (const bf16*)nullptr; },
                    [&](int n) { return n0 + n < a.N ? w + (size_t)(n0 + n) * a.K : (const bf16*)nullptr; }, a.K, acc);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int t = t0 + (lane >> 4) * 4 + i;
    if (t >= a.T) continue;
    const float g = a.gate ? 1.f / (1.f + expf(-a.gate[(size_t)t * a.ldg + h])) : 1.f;
#pragma unroll
    for (int tl = 0; tl < TILE_MFMA_WAVE_TILES; ++tl) {
      const int n = n0 + wave * (16 * TILE_MFMA_WAVE_TILES) + tl * 16 + (lane & 15);
      if (n < a.N) ((bf16*)a.y)[(size_t)t * a.ldy + (size_t)h * a.ys + n] = (bf16)(acc[tl][i] * g);
    }
  }
}

// The same for few tokens: 16 tokens by 32 elements a block, whose four waves take every fourth of K's steps and meet in LDS.  Four times the blocks,
// and one round of loads instead of several after each other.  Us, the kernel above and this one, 16 heads: 512 into 128, 8 tokens 7.6 and 3.5, 32 8.3
// and 3.9, 192 (192 blocks above) 8.6 and 6.8; 128 into 512, 8 tokens 4.2 and 2.7, 32 4.4 and 3.4, 128 (512) 6.1 and 6.0; 64 into 128, 32 tokens
// 3.7 and 2.8; 32 heads of 512 into 128, 128 tokens (256) 10.4 and 8.6, 192 (384) 16.4 and 16.3.
#define HEADWISE_SPLIT_COLS 32
__global__ void __launch_bounds__(256) headwise_split_kernel(HeadwiseArgs a) {
  constexpr int NT = HEADWISE_SPLIT_COLS / 16, AHEAD = 4;
  __shared__ __attribute__((aligned(16))) float parts[4][NT][256];  // lane l's four results of a tile at 4 l
  const int t0 = blockIdx.x * TILE_ROWS, h = blockIdx.y, n0 = blockIdx.z * HEADWISE_SPLIT_COLS;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, kq = (lane >> 4) * 8;
  // a row that is not there is the first one: its results are not stored
  const bf16* const x = (const bf16*)a.x + (size_t)h * a.xs + (size_t)(t0 + r < a.T ? t0 + r : t0) * a.ldx;
  const bf16* w[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) w[t] = (const bf16*)a.w + ((size_t)h * a.N + (n0 + t * 16 + r < a.N ? n0 + t * 16 + r : n0)) * a.K;
  f32x4 acc[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  const bf16x8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
  for (int k0 = wave * 32; k0 < a.K; k0 += 128 * AHEAD) {
    bf16x8 xv[AHEAD], wv[AHEAD][NT];
#pragma unroll
    for (int s = 0; s < AHEAD; ++s) {
      const int k = k0 + 128 * s + kq;
      xv[s] = k < a.K ? *reinterpret_cast<const bf16x8*>(x + k) : zero;
#pragma unroll
      for (int t = 0; t < NT; ++t) wv[s][t] = k < a.K ? *reinterpret_cast<const bf16x8*>(w[t] + k) : zero;
    }
#pragma unroll
    for (int s = 0; s < AHEAD; ++s)
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xv[s], wv[s][t], acc[t], 0, 0, 0);
  }
#pragma unroll
  for (int t = 0; t < NT; ++t) *reinterpret_cast<f32x4*>(&parts[wave][t][lane * 4]) = acc[t];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < NT; ++i) {  // neighbouring threads: neighbouring elements of a token
    const int at = i * 256 + threadIdx.x, row = at / HEADWISE_SPLIT_COLS, c = at % HEADWISE_SPLIT_COLS, t = t0 + row, n = n0 + c;
    if (t >= a.T || n >= a.N) continue;
    const int from = (row / 4 * 16 + c % 16) * 4 + row % 4;
    float v = 0.f;
#pragma unroll
    for (int p = 0; p < 4; ++p) v += parts[p][c / 16][from];
    if (a.gate) v *= 1.f / (1.f + expf(-a.gate[(size_t)t * a.ldg + h]));
    ((bf16*)a.y)[(size_t)t * a.ldy + (size_t)h * a.ys + n] = (bf16)v;
  }
}

// The same for steps of many tokens, through LDS (tile_product_lds.h): tiles of 128 tokens by 128 elements, two blocks a compute
// unit.  K is short (a head's size or the latent's), so a block is mostly its first loads and its stores.  2048 tokens, 16 heads
// of 128 into a latent of 512 and back: 24.8 us on average (29.7 in tiles of 64 tokens whose operands came straight from memory).
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) headwise_lds_kernel(HeadwiseArgs a) {
  typedef TileLds<2, 2, 2, 2, 2> S;
  __shared__ __attribute__((aligned(16))) bf16 lds[S::LDS_ELEMENTS];
  const int n0 = blockIdx.x * S::BN, h = blockIdx.y, t0 = blockIdx.z * S::BM;
  const bf16* x = (const bf16*)a.x + (size_t)h * a.xs;
  const bf16* w = (const bf16*)a.w + (size_t)h * a.N * a.K;
  f32x16 acc[2][2];
  tile_product_lds<2, 2, 2, 2, 2>([&](int m) { return x + (size_t)(t0 + m < a.T ? t0 + m : t0) * a.ldx; },
                                  [&](int n) { return w + (size_t)(n0 + n < a.N ? n0 + n : 0) * a.K; }, a.K, lds, acc);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int t = t0 + ((wave >> 1) * 2 + i) * 32 + 8 * (e / 4) + 4 * (lane >> 5) + e % 4;
      if (t >= a.T) continue;
      const float g = a.gate ? 1.f / (1.f + expf(-a.gate[(size_t)t * a.ldg + h])) : 1.f;
      bf16* y = (bf16*)a.y + (size_t)t * a.ldy + (size_t)h * a.ys;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int n = n0 + ((wave & 1) * 2 + j) * 32 + (lane & 31);
        if (n < a.N) y[n] = (bf16)(acc[i][j][e] * g);
      }
    }
  }
}

#define HEADWISE_COMPUTE_UNITS 256
#define HEADWISE_SPLIT_K 64        // (two steps)
#define HEADWISE_SPLIT_BLOCKS 384  // of the kernel without the split

extern "C" int fmsamd_headwise_linear(const void* x, long ldx, long x_head_stride, const void* w, void* y, long ldy,
                                      long y_head_stride, const float* gate, long ldg, int dtype, int n_tokens, int nheads,
                                      int N, int K, hipStream_t stream) {
  if (n_tokens == 0) return 0;
  FMS_REQUIRE(n_tokens > 0 && nheads > 0 && nheads <= 65535 && N > 0 && K > 0, "headwise_linear: bad sizes T=%d H=%d N=%d K=%d",
              n_tokens, nheads, N, K);
  FMS_REQUIRE(ldx >= (nheads - 1) * x_head_stride + K && ldy >= (nheads - 1) * y_head_stride + N,
              "headwise_linear: rows too short for %d heads", nheads);
  HeadwiseArgs a{x, ldx, x_head_stride, w, y, ldy, y_head_stride, gate, ldg, n_tokens, nheads, N, K};
  const int row_tiles = ceil_div(n_tokens, TILE_ROWS);
  if (dtype == FMS_F32) {
    headwise_fma_kernel<float><<<dim3(row_tiles, nheads, ceil_div(N, TILE_FMA_COLS)), TILE_THREADS, 0, stream>>>(a);
  } else if (dtype == FMS_BF16) {
    const bool aligned = K % 8 == 0 && ldx % 8 == 0 && x_head_stride % 8 == 0 && ((uintptr_t)x % 16) == 0 && ((uintptr_t)w % 16) == 0;
    const dim3 grid(ceil_div(N, 128), nheads, ceil_div(n_tokens, 128));
    // The kernel through LDS takes 7 to 10 us however little it has to do: it is for at least a full tile of tokens, more blocks of
    // the other kernel than there are compute units, and enough products.  Measured for both, us (16 tokens a block first): 16 heads of
    // 128 into 512, 128 tokens 6.4, 8.0, 200 (2.1e8 products) 9.0, 8.2; 32 of 128 into 128, 256 tokens 6.1, 7.9, 512 9.1, 8.2; 4 of 64
    // into 2048, 256 tokens 6.6, 7.6, 384 (2.0e8) 8.7, 8.1; 16 of 512 into 128, 256 tokens (256 blocks) 8.7, 10.4, 384 13.9, 10.6.
    const bool full = n_tokens >= 128 && (long)row_tiles * nheads * ceil_div(N, TILE_MFMA_COLS) > HEADWISE_COMPUTE_UNITS &&
                      (double)n_tokens * nheads * N * K >= 2e8;
    if (aligned && K >= TL_BK && full && grid.z <= 65535)  // (and tiles that fit a launch)
      headwise_lds_kernel<<<grid, 256, 0, stream>>>(a);
    else if (aligned && K >= HEADWISE_SPLIT_K && (long)row_tiles * nheads * ceil_div(N, TILE_MFMA_COLS) <= HEADWISE_SPLIT_BLOCKS &&
             ceil_div(N, HEADWISE_SPLIT_COLS) <= 65535)
      headwise_split_kernel<<<dim3(row_tiles, nheads, ceil_div(N, HEADWISE_SPLIT_COLS)), 256, 0, stream>>>(a);
    else if (aligned)
      headwise_mfma_kernel<<<dim3(row_tiles, nheads, ceil_div(N, TILE_MFMA_COLS)), TILE_THREADS, 0, stream>>>(a);
    else
      headwise_fma_kernel<bf16><<<dim3(row_tiles, nheads, ceil_div(N, TILE_FMA_COLS)), TILE_THREADS, 0, stream>>>(a);
  } else {
    FMS_REQUIRE(false, "headwise_linear: unknown dtype %d", dtype);
  }
  FMS_LAUNCH_CHECK("headwise_linear");
  return 0;
}

// --------------------------------------------------------------------------
// generic attention: one block per (head, token), keys 256 at a time
// --------------------------------------------------------------------------
#define LAT_THREADS 256
#define LAT_MAX_RANK 1024  // 4 output elements a thread

template <typename T>
__global__ void __launch_bounds__(LAT_THREADS)
    latent_attn_generic_kernel(const T* __restrict__ qa, long ldq, T* __restrict__ out, long ldo,
                               const int* __restrict__ positions, const int* __restrict__ seq_of_token,
                               const int* __restrict__ block_table, int table_stride, const T* __restrict__ cache,
                               const float* __restrict__ sink, int rank, int rot, float scale, int window) {
  extern __shared__ float qs[];  // rank + rot
  __shared__ float ps[LAT_THREADS];
  __shared__ float scratch[17];
  const int h = blockIdx.x, t = blockIdx.y;
  const int width = rank + rot;
  const int seq = seq_of_token[t];
  T* o = out + (size_t)t * ldo + (size_t)h * rank;
  if (seq < 0) {
    for (int d = threadIdx.x; d < rank; d += blockDim.x) o[d] = from_f32<T>(0.f);
    return;
  }
  const int pos = positions[t];
  const int lo = window > 0 ? (pos - window + 1 > 0 ? pos - window + 1 : 0) : 0;
  const int* bt = block_table + (size_t)seq * table_stride;
  const T* qrow = qa + (size_t)t * ldq + (size_t)h * width;
  for (int d = threadIdx.x; d < width; d += blockDim.x) qs[d] = to_f32(qrow[d]);
  __syncthreads();

  // the sink is where the softmax starts: a logit that is already in the denominator, with no value
  float m_run = sink ? sink[h] : -1e30f, l_run = sink ? 1.f : 0.f;
  float acc[4] = {0.f, 0.f, 0.f, 0.f};
  const int first = lo - lo % PAGE_TOKENS;  // chunks begin at a page's first token
  for (int base = first; base <= pos; base += LAT_THREADS) {
    const int j = base + threadIdx.x;
    float s = -INFINITY;
    if (j >= lo && j <= pos) {
      const T* krow = cache + (readable_page(bt[j / PAGE_TOKENS]) * PAGE_TOKENS + j % PAGE_TOKENS) * width;
      float dot = 0.f;
      for (int d = 0; d < width; ++d) dot = fmaf(qs[d], to_f32(krow[d]), dot);
      s = dot * scale;
    }
    const float m_new = fmaxf(m_run, block_max(s, scratch));
    const float p = (j >= lo && j <= pos) ? expf(s - m_new) : 0.f;
    const float alpha = expf(m_run - m_new);
    ps[threadIdx.x] = p;
    const float psum = block_sum(p, scratch);  // has the barriers that publish ps
    l_run = l_run * alpha + psum;
    m_run = m_new;
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] *= alpha;
    const int n = pos - base + 1 < LAT_THREADS ? pos - base + 1 : LAT_THREADS;
    for (int pg = 0; pg * PAGE_TOKENS < n; ++pg) {
      const T* prow = cache + readable_page(bt[base / PAGE_TOKENS + pg]) * PAGE_TOKENS * width;
      const int cnt = n - pg * PAGE_TOKENS < PAGE_TOKENS ? n - pg * PAGE_TOKENS : PAGE_TOKENS;
      for (int i = 0; i < cnt; ++i) {
        const float pi = ps[pg * PAGE_TOKENS + i];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int d = threadIdx.x + e * LAT_THREADS;
          if (d < rank) acc[e] = fmaf(pi, to_f32(prow[(size_t)i * width + d]), acc[e]);
        }
      }
    }
    __syncthreads();  // ps is overwritten by the next chunk
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int d = threadIdx.x + e * LAT_THREADS;
    if (d < rank) o[d] = from_f32<T>(l_run > 0.f ? acc[e] / l_run : 0.f);
  }
}

extern "C" int fmsamd_latent_attn_generic(const void* qa, long ldq, void* out, long ldo, int dtype, const int* positions,
                                          const int* seq_of_token, const int* block_table, int table_stride,
                                          const void* cache, const float* sink, int n_tokens, int nheads, int rank, int rot,
                                          float scale, int window, hipStream_t stream) {
  if (n_tokens == 0) return 0;
  FMS_REQUIRE(n_tokens > 0 && n_tokens <= 65535 && nheads > 0, "latent_attn_generic: %d tokens, %d heads (at most 65535 tokens a launch)",
              n_tokens, nheads);
  FMS_REQUIRE(rank > 0 && rank <= LAT_MAX_RANK && rot >= 0 && rank + rot <= 2048, "latent_attn_generic: latent size %d (at most %d), rotated size %d",
              rank, LAT_MAX_RANK, rot);
  FMS_REQUIRE(ldq >= (long)nheads * (rank + rot) && ldo >= (long)nheads * rank, "latent_attn_generic: rows too short");
  FMS_REQUIRE(window >= 0, "latent_attn_generic: window %d", window);
  const dim3 grid(nheads, n_tokens);
  const size_t lds = (size_t)(rank + rot) * sizeof(float);
  if (dtype == FMS_F32)
    latent_attn_generic_kernel<float><<<grid, LAT_THREADS, lds, stream>>>((const float*)qa, ldq, (float*)out, ldo, positions,
                                                                          seq_of_token, block_table, table_stride,
                                                                          (const float*)cache, sink, rank, rot, scale, window);
  else if (dtype == FMS_BF16)
    latent_attn_generic_kernel<bf16><<<grid, LAT_THREADS, lds, stream>>>((const bf16*)qa, ldq, (bf16*)out, ldo, positions,
                                                                         seq_of_token, block_table, table_stride,
                                                                         (const bf16*)cache, sink, rank, rot, scale, window);
  else
    FMS_REQUIRE(false, "latent_attn_generic: unknown dtype %d", dtype);
  FMS_LAUNCH_CHECK("latent_attn_generic");
  return 0;
}


// --------------------------------------------------------------------------
// bfloat16 MFMA kernel.  A wave owns one token and 16 of its heads (the columns of its tiles) and walks over tiles of
// 32 keys.  S^T = K Q^T (rows: keys, columns: heads) leaves the probabilities in the accumulator in the operand
// layout of O^T = C^T P^T, so nothing goes through LDS.  The 32 keys of a tile are dealt to the two score tiles so
// that a lane's eight probabilities are eight consecutive keys: tile a has the keys 8g + i, tile b the keys
// 8g + 4 + i (g, i < 4).
//
// Two ways to share the work of a block's four waves:
//   * prompts: each wave another (token, head group); every wave walks all keys of its token (the waves of a block
//     read the same rows, which the caches serve);
//   * single tokens: a block's waves deal out a run of key tiles of one (token, head group) in turn and meet in LDS; the
//     blocks that share it leave (maximum, sum, unnormalised result) each in a workspace, and a second kernel merges them.
// The sink starts the maximum of every part and is counted in the sum of part 0 only.
// --------------------------------------------------------------------------
#define LAT_EMPTY -1e30f
#define LAT_NO_KEYS -1.f  // the sum of a part without keys: a real one is no negative number

// The state of a wave's 16 columns, and one tile of 32 keys worked into it.  load_k(which, c) gives this lane's eight
// elements c * 32 + grp * 8 .. of its row of score tile a (which 0) or b (1); load_v(dt) its eight keys grp * 8 .. of
// latent element dt * 16 + col.  Loads are asked for in groups (KG steps of K, VG tiles of the latent) before the
// first of a group is multiplied: with the accumulators of a large latent a wave has a SIMD to itself, and the loads
// it keeps in flight are all that hides the memory's latency.
template <int RT, int WC>
struct LatentState {
  f32x4 acc[RT];
  float m, l;
};

// EXACT: the latent has exactly RT * 16 elements and a row exactly WC * 32, so no product of the loops below has
// to be asked whether it exists (each such question is a branch around a matrix instruction).
// AHEAD: the tile's keys and the first VG tiles of its latent are asked for at once, the next VG once the keys have been
// multiplied, and so on VG at a time behind the products: not a round trip to memory for every group (KG is the whole of K).
template <int RT, int WC, int KG, int VG, bool EXACT, bool AHEAD = false, typename LoadQ, typename LoadK, typename LoadV>
__device__ __forceinline__ void latent_tile(LatentState<RT, WC>& st, LoadQ load_q, LoadK load_k, LoadV load_v, int base,
                                            int lo, int pos, int rank, int width, float scale, int grp) {
  f32x4 sa = {0.f, 0.f, 0.f, 0.f}, sb = {0.f, 0.f, 0.f, 0.f};
  bf16x8 ahead[2][AHEAD ? VG : 1];
  auto ask = [&](int set, int d0) {
#pragma unroll
    for (int dt = 0; dt < VG; ++dt)
      if (d0 + dt < RT && (EXACT || (d0 + dt) * 16 < rank)) ahead[set][AHEAD ? dt : 0] = load_v(d0 + dt);
  };
#pragma unroll
  for (int c0 = 0; c0 < WC; c0 += KG) {
    bf16x8 ka[KG], kb[KG];
#pragma unroll
    for (int c = 0; c < KG; ++c) {
      if (c0 + c < WC && (EXACT || (c0 + c) * 32 < width)) ka[c] = load_k(0, c0 + c), kb[c] = load_k(1, c0 + c);
    }
    if constexpr (AHEAD) {
      static_assert(KG >= WC, "one group of keys");
      ask(0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int c = 0; c < KG; ++c) {
      if (c0 + c < WC && (EXACT || (c0 + c) * 32 < width)) {
        const bf16x8 q = load_q(c0 + c);
        sa = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ka[c], q, sa, 0, 0, 0);
        sb = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kb[c], q, sb, 0, 0, 0);
      }
    }
  }
  if constexpr (AHEAD && VG < RT) {
    __builtin_amdgcn_sched_barrier(0);
    ask(1, VG);
    __builtin_amdgcn_sched_barrier(0);
  }
  // this lane's scores: keys base + 8 grp + i (sa) and base + 8 grp + 4 + i (sb) of its column
  float s[8];
  float top = -INFINITY;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int ja = base + 8 * grp + i, jb = ja + 4;
    s[i] = (ja >= lo && ja <= pos) ? sa[i] * scale : -INFINITY;
    s[4 + i] = (jb >= lo && jb <= pos) ? sb[i] * scale : -INFINITY;
    top = fmaxf(top, fmaxf(s[i], s[4 + i]));
  }
  top = fmaxf(top, __shfl_xor(top, 16, WAVE));
  top = fmaxf(top, __shfl_xor(top, 32, WAVE));
  const float m_new = fmaxf(st.m, top);
  const float alpha = __expf(st.m - m_new);
  float psum = 0.f;
  bf16x8 pmat;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float p = __expf(s[i] - m_new);  // exp(-inf) = 0 for the keys that are not seen
    psum += p;
    pmat[i] = (bf16)p;
  }
  st.l = st.l * alpha + psum;
  st.m = m_new;
  // Once a column's maximum has settled, alpha is one: the accumulators (which live in the matrix unit's registers
  // and have to be moved out and back to be scaled) are left alone unless some column's maximum rose.
  const bool rescale = __any(alpha != 1.f);
#pragma unroll
  for (int d0 = 0; d0 < RT; d0 += VG) {
    bf16x8 v[VG];
#pragma unroll
    for (int dt = 0; dt < VG; ++dt) {
      if (d0 + dt < RT && (EXACT || (d0 + dt) * 16 < rank)) {
        if constexpr (AHEAD) v[dt] = ahead[d0 / VG & 1][dt];
        else v[dt] = load_v(d0 + dt);
      }
    }
#pragma unroll
    for (int dt = 0; dt < VG; ++dt) {
      if (d0 + dt < RT && (EXACT || (d0 + dt) * 16 < rank)) {
        if (rescale) {
#pragma unroll
          for (int i = 0; i < 4; ++i) st.acc[d0 + dt][i] *= alpha;
        }
        st.acc[d0 + dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v[dt], pmat, st.acc[d0 + dt], 0, 0, 0);
      }
    }
    if constexpr (AHEAD) {
      if (d0 + 2 * VG < RT) ask(d0 / VG & 1, d0 + 2 * VG);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
}

// What a wave that has all keys of its tile leaves: the normalised result.
template <int RT, int WC, bool EXACT>
__device__ __forceinline__ void latent_finish(LatentState<RT, WC>& st, bf16* __restrict__ out, long ldo, int t, int head, int nheads,
                                              int rank, int grp) {
  st.l += __shfl_xor(st.l, 16, WAVE);
  st.l += __shfl_xor(st.l, 32, WAVE);
  if (head >= nheads) return;
  // acc[dt][i] is element d = dt * 16 + grp * 4 + i of this lane's column
  const float inv = st.l > 0.f ? 1.f / st.l : 0.f;
  bf16* o = out + (size_t)t * ldo + (size_t)head * rank;
#pragma unroll
  for (int dt = 0; dt < RT; ++dt) {
    if (EXACT || dt * 16 < rank) {
      bf16x4 r = {(bf16)(st.acc[dt][0] * inv), (bf16)(st.acc[dt][1] * inv), (bf16)(st.acc[dt][2] * inv), (bf16)(st.acc[dt][3] * inv)};
      *reinterpret_cast<bf16x4*>(o + dt * 16 + grp * 4) = r;
    }
  }
}

// What a block of single tokens leaves, whose four waves had a share of the keys each: they meet in LDS (`lds`: 4 x 16 rows of
// RT * 16 + 4 floats, in the place of the queries), and the block leaves one part: maximum, sum and unnormalised result, or with
// no other part the result itself.  (A part a wave was 34 MB to write and to read again for 32 tokens of 16 heads.)  `used`: the
// waves that had any keys, the first ones.
template <int RT, int WC, bool EXACT>
__device__ __forceinline__ void latent_meet(LatentState<RT, WC>& st, float* __restrict__ lds, bf16* __restrict__ out, long ldo,
                                            float* __restrict__ ws, int t, int head0, int nheads, int rank, int n_parts, int part,
                                            int used) {
  constexpr int ROW = RT * 16 + 4;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, col = lane & 15, grp = lane >> 4;
  st.l += __shfl_xor(st.l, 16, WAVE);
  st.l += __shfl_xor(st.l, 32, WAVE);
  __syncthreads();  // the queries have been read
  float* row = lds + (wave * 16 + col) * ROW;
  if (wave < used) {
#pragma unroll
    for (int dt = 0; dt < RT; ++dt)
      if (EXACT || dt * 16 < rank) *reinterpret_cast<f32x4*>(row + dt * 16 + grp * 4) = st.acc[dt];
    if (grp == 0) row[RT * 16] = st.m, row[RT * 16 + 1] = st.l;
  }
  __syncthreads();
  // a wave takes the same quarter of every column
#pragma unroll
  for (int n = 0; n < RT / 4; ++n) {
    const int at = n * 64 + lane, c = at / RT, d = (wave * RT + at % RT) * 4;
    if (head0 + c >= nheads || (!EXACT && d >= rank)) continue;
    float m[4], top = LAT_EMPTY, l = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) m[w] = w < used ? lds[(w * 16 + c) * ROW + RT * 16] : LAT_EMPTY, top = fmaxf(top, m[w]);
    f32x4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      if (w >= used) break;
      const float e = __expf(m[w] - top);
      l = fmaf(lds[(w * 16 + c) * ROW + RT * 16 + 1], e, l);
      sum += *reinterpret_cast<const f32x4*>(lds + (w * 16 + c) * ROW + d) * e;
    }
    if (n_parts == 1) {
      const float inv = l > 0.f ? 1.f / l : 0.f;
      const bf16x4 r = {(bf16)(sum[0] * inv), (bf16)(sum[1] * inv), (bf16)(sum[2] * inv), (bf16)(sum[3] * inv)};
      *reinterpret_cast<bf16x4*>(out + (size_t)t * ldo + (size_t)(head0 + c) * rank + d) = r;
    } else {
      float* o = ws + (((size_t)t * nheads + head0 + c) * n_parts + part) * (rank + 4);
      *reinterpret_cast<f32x4*>(o + 4 + d) = sum;
      if (d == 0) o[0] = top, o[1] = l;
    }
  }
}

// LDS: the four waves of a block (four consecutive tiles of one sequence: neighbouring tokens, or the head groups of
// one token) share every tile of keys through LDS, so a tile comes from the caches once a block instead of once a
// wave; a block whose tiles lie in different sequences, and every block of a decode step, loads straight from
// global memory.
template <int RT, int WC, bool LDS, bool EXACT>
__global__ void __launch_bounds__(256)
    latent_attn_mfma_kernel(const bf16* __restrict__ qa, long ldq, bf16* __restrict__ out, long ldo, float* __restrict__ ws,
                            const int* __restrict__ positions, const int* __restrict__ seq_of_token,
                            const int* __restrict__ block_table, int table_stride, const bf16* __restrict__ cache,
                            const bf16* __restrict__ vt_cache, const float* __restrict__ sink, int n_tokens, int nheads,
                            int rank, int width, float scale, int window, int tiles_per_token, int n_parts) {
  extern __shared__ __attribute__((aligned(16))) bf16 lds[];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int col = lane & 15, grp = lane >> 4;
  const int n_tiles = n_tokens * tiles_per_token;
  // prompts: four tiles a block; single tokens (!LDS): one, whose keys up to n_parts blocks share, and their waves
  const int tile = LDS ? blockIdx.x * 4 + wave : blockIdx.x, block_part = LDS ? 0 : blockIdx.y;
  // do the block's four tiles share their keys?  (every wave works that out for itself, and all agree)
  bool together = false;
  int seq = -1, pos = -1, t = 0;
  if (tile < n_tiles) {
    t = tile / tiles_per_token;
    seq = uniform_load(seq_of_token + t);
    pos = seq >= 0 ? uniform_load(positions + t) : -1;
  }
  int first_pos = 0x7fffffff, last_pos = -1;
  if (LDS) {
    together = true;
    int common = -2;
    for (int w = 0; w < 4; ++w) {
      const int tl = blockIdx.x * 4 + w;
      if (tl >= n_tiles) continue;
      const int tt = tl / tiles_per_token;
      const int sq = uniform_load(seq_of_token + tt);
      if (sq < 0) continue;
      if (common == -2) common = sq;
      together = together && sq == common;
      const int p = uniform_load(positions + tt);
      first_pos = p < first_pos ? p : first_pos;
      last_pos = p > last_pos ? p : last_pos;
    }
    together = together && common >= 0;
  }
  const int head = (tile % tiles_per_token) * 16 + col;
  const bool valid = tile < n_tiles && seq >= 0 && head < nheads;
  if (!(LDS && together)) {
    if (tile >= n_tiles) return;
    if (seq < 0) {
      if (n_parts == 1 && head < nheads) {
        for (int d = grp; d < rank; d += 4) out[(size_t)t * ldo + (size_t)head * rank + d] = (bf16)0.f;
      }
      return;
    }
  }
  const int lo = window > 0 ? (pos - window + 1 > 0 ? pos - window + 1 : 0) : 0;

  // single tokens: the block's keys are tiles first .. end - 1, `share` of them as far as there are.  The cut goes by this token's
  // own context and the number of parts, so that what the other rows of the step hold changes no bit.  (Shares that spread the
  // tiles of all rows over one round of blocks by the contexts as they are take 31.5 us instead of 32.2 for 32 sequences of 128 to
  // 2048 tokens, 16 heads, latent 512 + 64, and 41 instead of 47.5 for 64; where all have 2000, 40.5 instead of 34 and 63 instead of 58.)
  int first = lo / 32, end = pos / 32 + 1, used = 4;  // used: the waves that have keys to work on, the first ones
  if constexpr (!LDS) {
    const int least = (end - first + n_parts - 1) / n_parts, share = n_parts > 1 && least < 4 ? 4 : least;  // a tile a wave
    const int parts = (end - first + share - 1) / share;
    if (n_parts > 1 && block_part == 0) {  // what the merge passes by
      for (int i = parts + wave * 4 + grp; i < n_parts; i += 16)
        if (head < nheads) {
          float* w = ws + (((size_t)t * nheads + head) * n_parts + i) * (rank + 4);
          w[0] = LAT_EMPTY, w[1] = LAT_NO_KEYS;
        }
    }
    first += block_part * share;
    end = end < first + share ? end : first + share;
    used = end - first < 4 ? end - first : 4;
    if (used <= 0) return;
  }
  // The queries wait in LDS, each lane's eight elements of every step of K in a slot: in registers they would crowd out
  // the loads that have to be in flight.  A prompt's wave has its own (written and read by the same lane: no barrier), the
  // waves of a single token share them.
  const bf16x8 zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
  bf16* q_lds = lds + ((size_t)(LDS ? wave * WC * 64 : 0) + lane) * 8;
  {
    const bf16* qrow = qa + (size_t)t * ldq + (size_t)(valid ? head : 0) * width;
#pragma unroll
    for (int c = 0; c < WC; ++c) {
      if (!LDS && (c & 3) != wave) continue;
      const int k = c * 32 + grp * 8;
      *reinterpret_cast<bf16x8*>(q_lds + c * 64 * 8) = (valid && (EXACT || k < width)) ? *reinterpret_cast<const bf16x8*>(qrow + k) : zero8;
    }
  }
  if constexpr (!LDS) __syncthreads();
  auto load_q = [&](int c) { return *reinterpret_cast<const bf16x8*>(q_lds + c * 64 * 8); };
  LatentState<RT, WC> st;
#pragma unroll
  for (int dt = 0; dt < RT; ++dt) st.acc[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  st.m = (sink && valid) ? sink[head] : LAT_EMPTY;
  st.l = (sink && valid && (LDS || (block_part == 0 && wave == 0)) && grp == 0) ? 1.f : 0.f;
  const int key_a = 8 * (col >> 2) + (col & 3);  // the key of this lane's row in score tile a; tile b: + 4

  if (LDS && together) {
    // all four waves walk the keys that any of them sees; a wave's own mask hides what it must not see
    const int ks = width + 8, vs = 32 + 8;  // row strides in LDS (elements): 16 bytes of padding against bank conflicts
    bf16* k_lds = lds + 4 * WC * 64 * 8;  // behind the four waves' queries
    bf16* v_lds = k_lds + 32 * ks;
    const int first_lo = window > 0 ? (first_pos - window + 1 > 0 ? first_pos - window + 1 : 0) : 0;
    const int common_seq = uniform_load(seq_of_token + (blockIdx.x * 4 < n_tiles ? (blockIdx.x * 4) / tiles_per_token : 0));
    int any_seq = common_seq;
    if (any_seq < 0) any_seq = seq;  // the block's first tile may be a padding row
    for (int w = 0; w < 4 && any_seq < 0; ++w) {
      const int tl = blockIdx.x * 4 + w;
      if (tl < n_tiles) any_seq = uniform_load(seq_of_token + tl / tiles_per_token);
    }
    const int* bt = block_table + (size_t)any_seq * table_stride;
    const int chunks_k = width / 8;  // 16-byte pieces in a key row
    // A thread's pieces of a tile: KP 16-byte pieces of the key rows, VP of the transposed latent.  The next tile's
    // pieces are asked for before this tile is worked on and wait in registers until every wave is done with it.
    constexpr int KP = (32 * WC * 4 + 255) / 256, VP = (RT * 16 * 4 + 255) / 256;
    bf16x8 kpre[KP], vpre[VP];
    // where this thread's pieces lie in a tile of the cache and in LDS: the same for every tile (the divisions are
    // done once; -1: this thread has no such piece)
    int k_from[KP], k_to[KP], v_from[VP], v_to[VP];
#pragma unroll
    for (int n = 0; n < KP; ++n) {
      const int i = threadIdx.x + n * 256;
      const bool has = i < 32 * chunks_k;
      k_from[n] = has ? (i / chunks_k) * width + (i % chunks_k) * 8 : -1;
      k_to[n] = has ? (i / chunks_k) * ks + (i % chunks_k) * 8 : -1;
    }
#pragma unroll
    for (int n = 0; n < VP; ++n) {
      const int i = threadIdx.x + n * 256;
      const bool has = i < rank * 4;
      v_from[n] = has ? (i >> 2) * PAGE_TOKENS + (i & 3) * 8 : -1;
      v_to[n] = has ? (i >> 2) * vs + (i & 3) * 8 : -1;
    }
    auto fetch = [&](int base) {
      const size_t page = readable_page(uniform_load(bt + base / PAGE_TOKENS));
      const int in_page = base % PAGE_TOKENS;
      const bf16* kp = cache + (page * PAGE_TOKENS + in_page) * width;
      const bf16* vp = vt_cache + page * rank * PAGE_TOKENS + in_page;
#pragma unroll
      for (int n = 0; n < KP; ++n) {
        if (k_from[n] >= 0) kpre[n] = *reinterpret_cast<const bf16x8*>(kp + k_from[n]);
      }
#pragma unroll
      for (int n = 0; n < VP; ++n) {
        if (v_from[n] >= 0) vpre[n] = *reinterpret_cast<const bf16x8*>(vp + v_from[n]);
      }
    };
    const int first_base = (first_lo / 32) * 32;
    if (first_base <= last_pos) fetch(first_base);
    for (int base = first_base; base <= last_pos; base += 32) {
      __syncthreads();  // the tile before this one has been read by every wave
#pragma unroll
      for (int n = 0; n < KP; ++n) {
        if (k_to[n] >= 0) *reinterpret_cast<bf16x8*>(k_lds + k_to[n]) = kpre[n];
      }
#pragma unroll
      for (int n = 0; n < VP; ++n) {
        if (v_to[n] >= 0) *reinterpret_cast<bf16x8*>(v_lds + v_to[n]) = vpre[n];
      }
      __syncthreads();
      if (base + 32 <= last_pos) fetch(base + 32);
      // (a condition that all lanes of the wave share: matrix instructions take their operands from every lane)
      if (tile < n_tiles && seq >= 0 && base <= pos) {
        latent_tile<RT, WC, (WC <= 10 ? WC : 6), (RT <= 16 ? RT : 8), EXACT>(
            st, load_q,
            [&](int which, int c) {
              return (EXACT || c * 32 + grp * 8 < width) ? *reinterpret_cast<const bf16x8*>(k_lds + (key_a + 4 * which) * ks + c * 32 + grp * 8) : zero8;
            },
            [&](int dt) { return *reinterpret_cast<const bf16x8*>(v_lds + (dt * 16 + col) * vs + grp * 8); }, base, lo, pos, rank, width,
            scale, grp);
      }
    }
    if (tile >= n_tiles) return;
    if (seq < 0) {
      if (head < nheads) {
        for (int d = grp; d < rank; d += 4) out[(size_t)t * ldo + (size_t)head * rank + d] = (bf16)0.f;
      }
      return;
    }
  } else {
    const int* bt = block_table + (size_t)seq * table_stride;
    for (int kt = first + (LDS ? 0 : wave); kt < end; kt += LDS ? 1 : 4) {
      const int base = kt * 32;
      const size_t page = readable_page(uniform_load(bt + base / PAGE_TOKENS));
      const int in_page = base % PAGE_TOKENS;
      const bf16* ka = cache + (page * PAGE_TOKENS + in_page + key_a) * width + grp * 8;
      const bf16* vt = vt_cache + (page * rank + col) * PAGE_TOKENS + in_page + grp * 8;
      // straight from global memory (guarded products of the largest sizes, and blocks of a prompt whose tiles lie in several
      // sequences, have no registers for loads that far ahead)
      constexpr bool AHEAD = !LDS && RT <= 16;
      latent_tile<RT, WC, (WC > 10 ? 9 : WC), (AHEAD && RT > 8 ? 8 : RT <= 16 ? RT : 16), EXACT, AHEAD>(
          st, load_q,
          [&](int which, int c) {
            return (EXACT || c * 32 + grp * 8 < width) ? *reinterpret_cast<const bf16x8*>(ka + which * 4 * (size_t)width + c * 32) : zero8;
          },
          [&](int dt) { return *reinterpret_cast<const bf16x8*>(vt + (size_t)dt * 16 * PAGE_TOKENS); }, base, lo, pos, rank, width, scale,
          grp);
    }
  }
  if constexpr (LDS) latent_finish<RT, WC, EXACT>(st, out, ldo, t, head, nheads, rank, grp);
  else latent_meet<RT, WC, EXACT>(st, reinterpret_cast<float*>(lds), out, ldo, ws, t, tile % tiles_per_token * 16, nheads, rank, n_parts, block_part, used);
}

// --------------------------------------------------------------------------
// bfloat16 prompts with a latent of RT * 16 elements in rows of WC * 32, the arithmetic of the kernel above.  A
// wave owns one tile (a token and 16 of its heads), its queries and results in registers, a SIMD to itself; the four
// tiles of a block share every 32 keys (rows and transposed latent) through LDS, in two buffers filled straight from memory
// while the other one is worked on, and operands are read from LDS some products ahead.
//
// Bound by the LDS reads of the operands (68 KB a wave and 32 keys for a latent of 512) and the chain through a tile's products and
// softmax, which a wave alone on its SIMD cannot hide.  One prompt of 2048 tokens, 16 heads, latent 512 + 64: 138 us; with the keys
// through registers and the shortest contexts first (the kernel above) 355, with results scaled whenever a maximum moved 212,
// with that inside the loop over the keys 182.
// A block whose tiles belong to several sequences takes the sequences one after the other: each wave works while its own
// tile's is there.  So a token has the same bits whatever else is in the step.  16 heads: 333, 1 and 90 tokens behind 1000 cached
// ones 172 us, nine prompts of 17 tokens 12.3 (355 and 27 with such blocks left to a second launch, of the kernel above; that
// kernel alone 277 and 17.2); 16 sequences of one token behind 500, four to a block, 110 (131).
// --------------------------------------------------------------------------
#define LAT_SLACK 8.f
#define LAT_GROUP 4  // tiles of a block

template <int RT, int WC>
__global__ void __launch_bounds__(256, 1)
    latent_attn_prompt_kernel(const bf16* __restrict__ qa, long ldq, bf16* __restrict__ out, long ldo, const int* __restrict__ positions,
                              const int* __restrict__ seq_of_token, const int* __restrict__ block_table, int table_stride,
                              const bf16* __restrict__ cache, const bf16* __restrict__ vt_cache, const float* __restrict__ sink,
                              int n_tokens, int nheads, float scale, int window, int tiles_per_token) {
  constexpr int RANK = RT * 16, WIDTH = WC * 32;
  constexpr int K_BYTES = 32 * WIDTH * 2, V_BYTES = RANK * 64, STAGE = K_BYTES + V_BYTES;
  constexpr int K_LOADS = K_BYTES / 4096, V_LOADS = V_BYTES / 4096;  // of 1 KB, a wave
  constexpr int PIECES = WIDTH / 8;                                  // of 16 bytes in a key's row
  static_assert(K_BYTES % 4096 == 0 && V_BYTES % 4096 == 0 && PIECES % 8 == 0, "whole loads, whole groups of pieces");
  extern __shared__ __attribute__((aligned(16))) bf16 lds[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, grp = lane >> 4;
  const int n_tiles = n_tokens * tiles_per_token;
  const int group = gridDim.x - 1 - blockIdx.x;  // the longest contexts first
  const int first_tile = group * LAT_GROUP, last_tile = first_tile + LAT_GROUP < n_tiles ? first_tile + LAT_GROUP - 1 : n_tiles - 1;
  int seqs[LAT_GROUP], places[LAT_GROUP];  // of the tiles; seqs -1: a padding row, or no tile
#pragma unroll
  for (int i = 0; i < LAT_GROUP; ++i) {
    const int u = (first_tile + i <= last_tile ? first_tile + i : last_tile) / tiles_per_token;
    seqs[i] = uniform_load(seq_of_token + u), places[i] = uniform_load(positions + u);
    if (first_tile + i > last_tile) seqs[i] = -1;
  }
  const int tile = first_tile + wave;
  const bool there = tile <= last_tile;
  const int t = (there ? tile : last_tile) / tiles_per_token, head = (tile % tiles_per_token) * 16 + col;
  const bool valid = there && head < nheads;
  int own_seq = -1, pos = -1;
#pragma unroll
  for (int i = 0; i < LAT_GROUP; ++i)
    if (i == wave) own_seq = seqs[i], pos = places[i];
  const int lo = window > 0 && pos - window + 1 > 0 ? pos - window + 1 : 0;

  bf16x8 q[WC];
  {
    const bf16* qrow = qa + (size_t)t * ldq + (size_t)(head < nheads ? head : 0) * WIDTH + grp * 8;
#pragma unroll
    for (int c = 0; c < WC; ++c) q[c] = *reinterpret_cast<const bf16x8*>(qrow + c * 32);
  }

  // what this lane loads: LDS holds a tile's pieces in the order of the rows; which piece of its group of eight (of a latent
  // element's four) a lane asks for is swizzled with the key (the element), so that operand reads cover all banks
  auto key_swizzle = [](int key) { return (key & 3) | ((key >> 1) & 4); };
  unsigned k_from[K_LOADS];
#pragma unroll
  for (int n = 0; n < K_LOADS; ++n) {
    const int at = (wave * K_LOADS + n) * 64 + lane, key = at / PIECES, p = at % PIECES;
    k_from[n] = (key * PIECES + (p ^ key_swizzle(key))) * 16;
  }
  const int v_row = wave * V_LOADS * 16 + (lane >> 2);
  const unsigned v_from = v_row * (PAGE_TOKENS * 2) + ((lane & 3) ^ ((lane >> 3) & 3)) * 16;  // rows 16 apart swizzle alike
  const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) bf16*)lds;
  auto fetch = [&](const int* bt, int base, int buffer) {
    const size_t page = readable_page(uniform_load(bt + base / PAGE_TOKENS));
    const int in_page = base % PAGE_TOKENS;
    const char* kp = (const char*)(cache + (page * PAGE_TOKENS + in_page) * WIDTH);
    const char* vp = (const char*)(vt_cache + page * RANK * PAGE_TOKENS + in_page);
    const unsigned to = lds0 + buffer * STAGE;
#pragma unroll
    for (int n = 0; n < K_LOADS; ++n) load_to_lds(kp, k_from[n], to + (wave * K_LOADS + n) * 1024);
#pragma unroll
    for (int n = 0; n < V_LOADS; ++n) load_to_lds(vp + n * 16 * PAGE_TOKENS * 2, v_from, to + K_BYTES + (wave * V_LOADS + n) * 1024);
  };

  // operand reads: this lane's key in score tile a (tile b: + 4), its latent element of every 16.  Steps of K two apart differ
  // by 128 bytes, which leaves the swizzle as it is.
  const int key_a = 8 * (col >> 2) + (col & 3);
  int k_at[2][2], v_at;  // [tile][step of K % 2]
#pragma unroll
  for (int w = 0; w < 2; ++w)
#pragma unroll
    for (int c = 0; c < 2; ++c) k_at[w][c] = (key_a + 4 * w) * WIDTH * 2 + ((4 * c + grp) ^ key_swizzle(key_a + 4 * w)) * 16;
  v_at = K_BYTES + col * 64 + (grp ^ ((col >> 1) & 3)) * 16;

  f32x4 acc[RT];
#pragma unroll
  for (int d = 0; d < RT; ++d) acc[d] = f32x4{0.f, 0.f, 0.f, 0.f};
  // the sink is where the softmax starts
  float m = sink && valid ? sink[head] : LAT_EMPTY, l = sink && valid && grp == 0 ? 1.f : 0.f;

  constexpr int KG = 3, VG = 4;  // steps of K, and tiles of the latent, that are read before the ones in front are multiplied
  bf16x8 ka[2][KG], kb[2][KG], v[2][VG];
  float s[8];
  // the scores of the buffer's 32 keys: s[i] is key base + 8 grp + i of this lane's column
  auto scores = [&](const char* kv, int base) {
    f32x4 sa = {0.f, 0.f, 0.f, 0.f}, sb = {0.f, 0.f, 0.f, 0.f};
    auto read_k = [&](int set, int c0) {
#pragma unroll
      for (int c = 0; c < KG; ++c)
        if (c0 + c < WC) {
          ka[set][c] = *reinterpret_cast<const bf16x8*>(kv + k_at[0][(c0 + c) & 1] + ((c0 + c) >> 1) * 128);
          kb[set][c] = *reinterpret_cast<const bf16x8*>(kv + k_at[1][(c0 + c) & 1] + ((c0 + c) >> 1) * 128);
        }
    };
    read_k(0, 0);
#pragma unroll
    for (int c0 = 0; c0 < WC; c0 += KG) {
      const int set = (c0 / KG) & 1;
      if (c0 + KG < WC) read_k(set ^ 1, c0 + KG);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int c = 0; c < KG; ++c)
        if (c0 + c < WC) {
          sa = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ka[set][c], q[c0 + c], sa, 0, 0, 0);
          sb = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kb[set][c], q[c0 + c], sb, 0, 0, 0);
        }
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) s[i] = sa[i] * scale, s[4 + i] = sb[i] * scale;
    if (base + 31 > pos || base < lo) {  // the same in all lanes
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int key = base + 8 * grp + i;
        s[i] = key >= lo && key <= pos ? s[i] : -INFINITY;
      }
    }
    float top = fmaxf(fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3])), fmaxf(fmaxf(s[4], s[5]), fmaxf(s[6], s[7])));
    top = fmaxf(top, __shfl_xor(top, 16, WAVE));
    return fmaxf(top, __shfl_xor(top, 32, WAVE));
  };
  // their probabilities and values into the sums
  auto values = [&](const char* kv) {
    auto read_v = [&](int set, int d0) {
#pragma unroll
      for (int d = 0; d < VG; ++d) v[set][d] = *reinterpret_cast<const bf16x8*>(kv + v_at + (d0 + d) * 16 * 64);
    };
    read_v(0, 0);
    float psum = 0.f;
    bf16x8 pmat;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float p = __expf(s[i] - m);  // exp(-inf) = 0 for the keys that are not seen
      psum += p;
      pmat[i] = (bf16)p;
    }
    l += psum;
#pragma unroll
    for (int d0 = 0; d0 < RT; d0 += VG) {
      const int set = (d0 / VG) & 1;
      if (d0 + VG < RT) read_v(set ^ 1, d0 + VG);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int d = 0; d < VG; ++d) acc[d0 + d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v[set][d], pmat, acc[d0 + d], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  // The reference m that probabilities are taken against follows the maximum only where that has left it LAT_SLACK behind: sums
  // and results are float32, and a bfloat16 probability is as exact at e^LAT_SLACK as at 1.  The results live in the matrix
  // unit's registers and have to be moved out and back to be scaled: that stands outside the loop over the keys, or the
  // compiler moves them for every tile (the waves of a block meet at the same barriers wherever they stand in the code).
  float top = LAT_EMPTY;
#pragma unroll 1
  for (int turn = 0; turn < LAT_GROUP; ++turn) {
    int seq = -1;  // of tile `turn`; its turn if no tile before it has the same
    bool again = false;
    int first_pos = 0x7fffffff, last_pos = -1;  // of the sequence's tokens in the block
#pragma unroll
    for (int i = 0; i < LAT_GROUP; ++i)
      if (i == turn) seq = seqs[i];
#pragma unroll
    for (int i = 0; i < LAT_GROUP; ++i)
      if (seqs[i] == seq) {
        again = again || i < turn;
        first_pos = places[i] < first_pos ? places[i] : first_pos, last_pos = places[i] > last_pos ? places[i] : last_pos;
      }
    if (seq < 0 || again) continue;
    const bool works = own_seq == seq;
    const int* bt = block_table + (size_t)seq * table_stride;
    const int first_lo = window > 0 && first_pos - window + 1 > 0 ? first_pos - window + 1 : 0;
    const int first_base = first_lo / 32 * 32;
    if (first_base <= last_pos) fetch(bt, first_base, 0);  // (no load may be on its way to LDS when the block ends)
    int base = first_base, buffer = 0;
    for (;;) {
      bool behind = false;
      for (; base <= last_pos; base += 32, buffer ^= 1) {
        if (base + 32 <= last_pos) {
          fetch(bt, base + 32, buffer ^ 1);
          tile_wait<K_LOADS + V_LOADS>();
        } else {
          tile_wait<0>();
        }
        if (works && base <= pos) {  // the same in all lanes of the wave
          const char* kv = (const char*)lds + buffer * STAGE;
          top = scores(kv, base);
          behind = __any(top > m + LAT_SLACK);
          if (behind) break;
          values(kv);
        }
        block_sync_lds();  // everybody has read the buffer
      }
      if (!behind) break;
      const float m_new = top > m + LAT_SLACK ? top : m;
      const float alpha = __expf(m - m_new);
      l *= alpha;
      m = m_new;
#pragma unroll
      for (int d = 0; d < RT; ++d)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[d][i] *= alpha;
      values((const char*)lds + buffer * STAGE);
      block_sync_lds();
      base += 32, buffer ^= 1;
    }
  }
  if (!there) return;
  LatentState<RT, WC> st;
#pragma unroll
  for (int d = 0; d < RT; ++d) st.acc[d] = acc[d];
  st.m = m, st.l = l;
  latent_finish<RT, WC, true>(st, out, ldo, t, head, nheads, RANK, grp);
}

// --------------------------------------------------------------------------
// bfloat16 single tokens with a latent of 512 (RT * 16 elements in rows of WC * 32): the parts, shares and arithmetic of the kernel above, bit
// by bit.  A wave brings its tile of 32 keys straight into its own place in LDS, as whole rows, and reads both operands there: the keys as they
// lie, the values transposed by the read (ds_read_b64_tr_b16), so that the latent comes from memory once and the transposed copy not at all.
// Bound by the rows' bytes (64 sequences of 2000 tokens: 147 MB in 34 us without the merge's 6) and, for few, by the chain of lookups, first loads and
// meeting.  Us with the merge, 16 heads, latent 512 + 64, the kernel above (keys and transposed latent through registers, 64 bytes of a row at a
// time) and this one: 32 sequences of 128 to 2048 tokens 33.0 and 26.1, 64 of them 48.2 and 33.9, 64 of 2000 59.0 and 39.9, 8 of 2000 22.2
// and 17.0, one of 100 19.0 and 14.2.  Operands asked for in other groups: the same within 3 %, whole rows of keys and 16 tiles of the latent
// ahead 36.1 (registers).
// The pieces of 16 bytes of a row are XOR-swizzled with the row on the address side of the loads, so that the reads of the 16 rows of an operand
// cover all banks: a row of 1152 bytes begins half way round them after the row before, one of 1024 where that does.
// --------------------------------------------------------------------------
template <int RT, int WC>
__global__ void __launch_bounds__(256, 1)
    latent_attn_decode_kernel(const bf16* __restrict__ qa, long ldq, bf16* __restrict__ out, long ldo, float* __restrict__ ws,
                              const int* __restrict__ positions, const int* __restrict__ seq_of_token, const int* __restrict__ block_table,
                              int table_stride, const bf16* __restrict__ cache, const float* __restrict__ sink, int nheads, float scale,
                              int window, int tiles_per_token, int n_parts) {
  constexpr int RANK = RT * 16, WIDTH = WC * 32, ROW = WIDTH * 2, TILE = 32 * ROW, LOADS = TILE / 1024;
  static_assert(ROW == 1152 || ROW == 1024, "the swizzles");
  extern __shared__ __attribute__((aligned(1024))) bf16 lds[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, grp = lane >> 4;
  const int t = blockIdx.x / tiles_per_token, head0 = blockIdx.x % tiles_per_token * 16, head = head0 + col, block_part = blockIdx.y;
  const bool valid = head < nheads;
  const int seq = uniform_load(seq_of_token + t);
  if (seq < 0) {
    if (n_parts == 1 && valid)
      for (int d = grp; d < RANK; d += 4) out[(size_t)t * ldo + (size_t)head * RANK + d] = (bf16)0.f;
    return;
  }
  const int pos = uniform_load(positions + t), lo = window > 0 ? (pos - window + 1 > 0 ? pos - window + 1 : 0) : 0;
  int first = lo / 32, end = pos / 32 + 1;
  const int least = (end - first + n_parts - 1) / n_parts, share = n_parts > 1 && least < 4 ? 4 : least;  // a tile a wave
  const int parts = (end - first + share - 1) / share;
  if (n_parts > 1 && block_part == 0) {  // what the merge passes by
    for (int i = parts + wave * 4 + grp; i < n_parts; i += 16)
      if (valid) {
        float* w = ws + (((size_t)t * nheads + head) * n_parts + i) * (RANK + 4);
        w[0] = LAT_EMPTY, w[1] = LAT_NO_KEYS;
      }
  }
  first += block_part * share;
  end = end < first + share ? end : first + share;
  const int used = end - first < 4 ? end - first : 4;
  if (used <= 0) return;

  bf16x8 q[WC];
  const bf16x8 zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
  const bf16* const qrow = qa + (size_t)t * ldq + (size_t)(valid ? head : 0) * WIDTH + grp * 8;
#pragma unroll
  for (int c = 0; c < WC; ++c) q[c] = valid ? *reinterpret_cast<const bf16x8*>(qrow + c * 32) : zero8;

  // where a lane's 16 bytes of a load come from: the loads fill LDS in the order of the lanes, 72 (64) of them a row
  constexpr int PIECES = ROW / 16, BASES = ROW == 1152 ? 9 : 1;  // nine loads are eight rows of 1152 bytes
  unsigned from[BASES];
#pragma unroll
  for (int j = 0; j < BASES; ++j) {
    const int at = j * 64 + lane, row = at / PIECES, piece = at % PIECES;
    from[j] = row * ROW + (ROW == 1152 ? piece ^ (row >> 1 & 1) : piece) * 16;
  }
  const unsigned place = (unsigned)(uintptr_t)(__attribute__((address_space(3))) bf16*)lds + wave * TILE;
  // rows 8 g + i and 8 g + 4 + i (i < 4) have the same swizzle: of 1152 bytes bit 1 of i and the two of g, of 1024 the two of i and of g
  auto swizzle = [](int g, int i) { return ROW == 1152 ? (i >> 1 & 1) | g << 1 : (i & 3) | g << 2; };
  const char* const mine = reinterpret_cast<const char*>(lds) + wave * TILE;
  const char* const key_row = mine + (8 * (col >> 2) + (col & 3)) * ROW;
  const int key_swizzle = swizzle(col >> 2, col & 3);
  // a transposing read: sixteen lanes ask for four keys, each a quarter of 16 elements, and lane l gets element l of the four
  const unsigned value_row = place + (8 * grp + (col >> 2)) * ROW + (col & 1) * 8;
  const int value_swizzle = swizzle(grp, col >> 2);

  LatentState<RT, WC> st;
#pragma unroll
  for (int dt = 0; dt < RT; ++dt) st.acc[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  st.m = (sink && valid) ? sink[head] : LAT_EMPTY;
  st.l = (sink && valid && block_part == 0 && wave == 0 && grp == 0) ? 1.f : 0.f;
  const int* const bt = block_table + (size_t)seq * table_stride;
  for (int kt = first + wave; kt < end; kt += 4) {
    const int base = kt * 32;
    const char* const rows = (const char*)(cache + (readable_page(uniform_load(bt + base / PAGE_TOKENS)) * PAGE_TOKENS + base % PAGE_TOKENS) * WIDTH);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the tile before this one has been read
#pragma unroll
    for (int j = 0; j < LOADS; ++j) {
      const int g = ROW == 1152 ? j / 9 : (j & 3) | (j >> 3) << 2;
      load_to_lds(rows + (ROW == 1152 ? j / 9 * 9216 : j * 1024), from[ROW == 1152 ? j % 9 : 0] ^ (g << (ROW == 1152 ? 5 : 4)), place + j * 1024);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    typedef __attribute__((address_space(3))) bf16x4 LdsRow;
    latent_tile<RT, WC, 6, 8, true>(
        st, [&](int c) { return q[c]; },
        [&](int which, int c) { return *reinterpret_cast<const bf16x8*>(key_row + which * 4 * ROW + ((c * 4 + grp) ^ key_swizzle) * 16); },
        [&](int dt) {
          const unsigned at = value_row + (((dt * 2 + (col >> 1 & 1)) ^ value_swizzle) * 16);
          const bf16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((LdsRow*)(uintptr_t)at);
          const bf16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((LdsRow*)(uintptr_t)(at + 4 * ROW));
          return __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
        },
        base, lo, pos, RANK, WIDTH, scale, grp);
  }
  latent_meet<RT, WC, true>(st, reinterpret_cast<float*>(lds), out, ldo, ws, t, head0, nheads, RANK, n_parts, block_part, used);
}

// out[t, h, :] = sum_i acc_i exp(m_i - M) / sum_i l_i exp(m_i - M) over the parts i.  The parts' maxima and sums are
// loaded side by side (a thread a part) and their weights left in LDS: no chain of dependent loads.
#define LAT_MAX_PARTS 64
__global__ void __launch_bounds__(256)
    latent_attn_merge_kernel(const float* __restrict__ ws, bf16* __restrict__ out, long ldo, const int* __restrict__ seq_of_token,
                             int nheads, int rank, int n_parts) {
  __shared__ float weight[LAT_MAX_PARTS];
  __shared__ float inv_total;
  __shared__ int n_used;  // the parts that have keys: the first ones
  const int h = blockIdx.x, t = blockIdx.y;
  bf16* o = out + (size_t)t * ldo + (size_t)h * rank;
  if (uniform_load(seq_of_token + t) < 0) {
    for (int d = threadIdx.x; d < rank; d += blockDim.x) o[d] = (bf16)0.f;
    return;
  }
  const float* w = ws + ((size_t)t * nheads + h) * n_parts * (rank + 4);
  // Two waits on memory, one after the other, bound this kernel, so a thread's elements of the first parts are asked for beside the parts'
  // weights (a part without keys is there, but nobody uses it).  Attention and merge of 32 tokens with 128 to 2048 keys, 16 heads: 26.2 us
  // without, 23.7 with; where a token has more parts than EARLY the rest follows as before (1 token of 2000 keys 15.2 either way).
  constexpr int EARLY = 8, MINE = 2;
  float early[MINE][EARLY];
#pragma unroll
  for (int m = 0; m < MINE; ++m) {
    const int d = threadIdx.x + m * blockDim.x;
#pragma unroll
    for (int i = 0; i < EARLY; ++i) early[m][i] = d < rank && i < n_parts ? w[(size_t)i * (rank + 4) + 4 + d] : 0.f;
  }
  if (threadIdx.x < WAVE) {  // the first wave weighs the parts
    float top;
    const int i = threadIdx.x;  // n_parts <= 64: a part a lane
    const float m = i < n_parts ? w[(size_t)i * (rank + 4)] : LAT_EMPTY, l = i < n_parts ? w[(size_t)i * (rank + 4) + 1] : 0.f;
    const bool counts = i < n_parts && l != LAT_NO_KEYS;  // also where every score is no number: the maximum passes those by
    top = wave_max(m);
    const float e = __expf(m - top);
    if (i < n_parts) weight[i] = e;
    const float total = wave_sum(counts ? l * e : 0.f);
    const unsigned long long mask = __ballot(counts);
    if (i == 0) inv_total = total > 0.f ? 1.f / total : 0.f, n_used = mask == 0 ? 0 : 64 - __clzll(mask);
  }
  __syncthreads();
  const float inv = inv_total;
  const int used = n_used;
#pragma unroll
  for (int m = 0; m < MINE; ++m) {  // at most two elements a thread
    const int d = threadIdx.x + m * blockDim.x;
    if (d >= rank) continue;
    float v = 0.f;
#pragma unroll
    for (int i = 0; i < EARLY; ++i) v = i < used ? fmaf(early[m][i], weight[i], v) : v;
#pragma unroll 8
    for (int i = EARLY; i < used; ++i) v = fmaf(w[(size_t)i * (rank + 4) + 4 + d], weight[i], v);
    o[d] = (bf16)(v * inv);
  }
}

// bytes of the workspace for n_splits blocks, a part each (0: one block per four tiles; neither that nor one block need any)
extern "C" long fmsamd_latent_attn_workspace(int n_tokens, int nheads, int rank, int n_splits) {
  return n_splits <= 1 ? 0 : (long)n_tokens * nheads * n_splits * (rank + 4) * (long)sizeof(float);
}

// 1 if the MFMA kernel takes these sizes
extern "C" int fmsamd_latent_attn_mfma_fits(int rank, int rot) {
  return rank > 0 && rank % 16 == 0 && rot >= 0 && (rank + rot) % 8 == 0 && rank <= 512 && rank + rot <= 576;
}

// n_splits 0: prompts (a wave per tile, every wave all keys); n_splits >= 1: single tokens (n_splits blocks of four
// waves deal a tile's keys out; workspace as fmsamd_latent_attn_workspace says)
extern "C" int fmsamd_latent_attn_mfma(const void* qa, long ldq, void* out, long ldo, void* workspace, long workspace_bytes,
                                       const int* positions, const int* seq_of_token, const int* block_table,
                                       int table_stride, const void* cache, const void* vt_cache, const float* sink,
                                       int n_tokens, int nheads, int rank, int rot, float scale, int window, int n_splits,
                                       hipStream_t stream) {
  if (n_tokens == 0) return 0;
  const int width = rank + rot;
  FMS_REQUIRE(n_tokens > 0 && nheads > 0 && fmsamd_latent_attn_mfma_fits(rank, rot), "latent_attn_mfma: sizes T=%d H=%d rank=%d rot=%d do not fit",
              n_tokens, nheads, rank, rot);
  FMS_REQUIRE(ldq >= (long)nheads * width && ldq % 8 == 0 && ldo >= (long)nheads * rank && ldo % 4 == 0 && ((uintptr_t)qa % 16) == 0,
              "latent_attn_mfma: rows too short or not aligned");
  FMS_REQUIRE(cache != nullptr && vt_cache != nullptr && window >= 0 && n_splits >= 0 && n_splits <= LAT_MAX_PARTS, "latent_attn_mfma: bad arguments (at most 64 splits)");
  const int tiles_per_token = ceil_div(nheads, 16);
  const long tiles = (long)n_tokens * tiles_per_token;
  const int n_parts = n_splits == 0 ? 1 : n_splits;
  FMS_REQUIRE(n_splits <= 1 || (workspace != nullptr && workspace_bytes >= fmsamd_latent_attn_workspace(n_tokens, nheads, rank, n_splits)),
              "latent_attn_mfma: the workspace is too small");
  const dim3 grid(n_splits == 0 ? ceil_div(tiles, 4) : (unsigned)tiles, n_splits == 0 ? 1 : n_splits);
  FMS_REQUIRE(tiles <= 0x7fffffffL, "latent_attn_mfma: too many tiles for one launch");
  // LDS: every wave's queries; for prompts also a tile of 32 key rows and the same keys' latent, transposed, which the
  // waves of a block share
#define LAUNCH_LATENT(RT, WC, EXACT)                                                                                               \
  const size_t q_lds = (size_t)4 * WC * 64 * 8 * sizeof(bf16); /* the four waves' queries of a prompt */                           \
  const size_t lds = q_lds + (size_t)(32 * (width + 8) + rank * 40) * sizeof(bf16);                                                \
  static bool allowed = false; /* more than 64 KB of LDS a block has to be asked for, once a kernel */                             \
  if (!allowed) {                                                                                                                  \
    hipError_t e1 = hipFuncSetAttribute((const void*)latent_attn_mfma_kernel<RT, WC, true, EXACT>,                                 \
                                        hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);                                   \
    hipError_t e2 = hipFuncSetAttribute((const void*)latent_attn_mfma_kernel<RT, WC, false, EXACT>,                                \
                                        hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);                                   \
    FMS_REQUIRE(e1 == hipSuccess && e2 == hipSuccess, "latent_attn_mfma: the kernel's LDS could not be sized: %s",                 \
                hipGetErrorString(e1 != hipSuccess ? e1 : e2));                                                                    \
    allowed = true;                                                                                                                \
  }                                                                                                                                \
  const size_t meet = (size_t)4 * 16 * (RT * 16 + 4) * sizeof(float); /* where the waves of a single token meet */                 \
  FMS_REQUIRE(lds <= 160 * 1024 && meet <= 160 * 1024, "latent_attn_mfma: %zu bytes of LDS", lds);                                 \
  if (n_splits == 0)                                                                                                               \
    latent_attn_mfma_kernel<RT, WC, true, EXACT><<<grid, 256, lds, stream>>>(                                                      \
        (const bf16*)qa, ldq, (bf16*)out, ldo, (float*)workspace, positions, seq_of_token, block_table, table_stride,              \
        (const bf16*)cache, (const bf16*)vt_cache, sink, n_tokens, nheads, rank, width, scale, window, tiles_per_token, n_parts);  \
  else                                                                                                                             \
    latent_attn_mfma_kernel<RT, WC, false, EXACT><<<grid, 256, meet > q_lds / 4 ? meet : q_lds / 4, stream>>>(                                                   \
        (const bf16*)qa, ldq, (bf16*)out, ldo, (float*)workspace, positions, seq_of_token, block_table, table_stride,              \
        (const bf16*)cache, (const bf16*)vt_cache, sink, n_tokens, nheads, rank, width, scale, window, tiles_per_token, n_parts)
  // prompts with a latent of 512 (the rows go straight to LDS, which wants 16-byte addresses)
  const bool prompt_kernel =
      n_splits == 0 && rank == 512 && (width == 576 || width == 512) && (uintptr_t)cache % 16 == 0 && (uintptr_t)vt_cache % 16 == 0;
  if (prompt_kernel) {
    const int groups = ceil_div(tiles, LAT_GROUP);
#define LAUNCH_PROMPT(RT, WC)                                                                                                      \
  const size_t bytes = 2 * (size_t)(32 * WC * 32 * 2 + RT * 16 * 64); /* two buffers of keys and latent */                         \
  static bool allowed = false;                                                                                                     \
  if (!allowed) {                                                                                                                  \
    const hipError_t e = hipFuncSetAttribute((const void*)latent_attn_prompt_kernel<RT, WC>,                                       \
                                             hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);                              \
    FMS_REQUIRE(e == hipSuccess, "latent_attn_mfma: the kernel's LDS could not be sized: %s", hipGetErrorString(e));               \
    allowed = true;                                                                                                                \
  }                                                                                                                                \
  latent_attn_prompt_kernel<RT, WC><<<groups, 256, bytes, stream>>>((const bf16*)qa, ldq, (bf16*)out, ldo, positions, seq_of_token, \
                                                                    block_table, table_stride, (const bf16*)cache,                 \
                                                                    (const bf16*)vt_cache, sink, n_tokens, nheads, scale, window,   \
                                                                    tiles_per_token)
    if (width == 576) {
      LAUNCH_PROMPT(32, 18);
    } else {
      LAUNCH_PROMPT(32, 16);
    }
#undef LAUNCH_PROMPT
    FMS_LAUNCH_CHECK("latent_attn_prompt");
    return 0;
  }
  // single tokens with a latent of 512 (likewise)
  const bool decode_kernel = n_splits > 0 && rank == 512 && (width == 576 || width == 512) && (uintptr_t)cache % 16 == 0;
  if (decode_kernel) {
#define LAUNCH_DECODE(RT, WC)                                                                                                      \
  constexpr int tiles_bytes = 4 * 32 * WC * 64, meet_bytes = 4 * 16 * (RT * 16 + 4) * (int)sizeof(float);                          \
  constexpr int bytes = tiles_bytes > meet_bytes ? tiles_bytes : meet_bytes;                                                       \
  static const hipError_t sized = hipFuncSetAttribute((const void*)latent_attn_decode_kernel<RT, WC>,                              \
                                                      hipFuncAttributeMaxDynamicSharedMemorySize, bytes);                          \
  FMS_REQUIRE(sized == hipSuccess, "latent_attn_mfma: the kernel's LDS could not be sized: %s", hipGetErrorString(sized));         \
  latent_attn_decode_kernel<RT, WC><<<grid, 256, bytes, stream>>>((const bf16*)qa, ldq, (bf16*)out, ldo, (float*)workspace, positions, \
                                                                  seq_of_token, block_table, table_stride, (const bf16*)cache, sink, nheads, \
                                                                  scale, window, tiles_per_token, n_parts)
    if (width == 576) {
      LAUNCH_DECODE(32, 18);
    } else {
      LAUNCH_DECODE(32, 16);
    }
#undef LAUNCH_DECODE
  } else
  // the smaller latents without a rotated part run without a question around any product; everything else in the smallest
  // configuration that holds it (also a latent of 512 whose cache does not start at a 16-byte address)
  if (rank == 256 && width == 256) {
    LAUNCH_LATENT(16, 8, true);
  } else if (rank == 128 && width == 128) {
    LAUNCH_LATENT(8, 4, true);
  } else if (rank <= 128 && width <= 192) {
    LAUNCH_LATENT(8, 6, false);
  } else if (rank <= 256 && width <= 320) {
    LAUNCH_LATENT(16, 10, false);
  } else {
    LAUNCH_LATENT(32, 18, false);
  }
#undef LAUNCH_LATENT
  FMS_LAUNCH_CHECK("latent_attn_mfma");
  if (n_parts > 1) {
    latent_attn_merge_kernel<<<dim3(nheads, n_tokens), rank > 128 ? 256 : 64, 0, stream>>>((const float*)workspace, (bf16*)out, ldo, seq_of_token, nheads,
                                                                         rank, n_parts);
    FMS_LAUNCH_CHECK("latent_attn_merge");
  }
  return 0;
}
