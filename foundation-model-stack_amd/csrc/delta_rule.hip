// The gated delta rule: a recurrent mixer whose state is a matrix S [key channels, value channels] per head.
//
//   S <- g * S           g: one decay per head, or one per head and key channel (it scales rows of S)
//   u  = beta (v - S^T k)
//   S <- S + k u^T
//   o  = S^T q           the read-out sees the token's own write
//
// Three kernels run a step of any number of tokens per sequence, all in float32:
//   delta_prepare:  the short causal convolution over time of the q, k and v channels (inputs before the step come
//                   from the sequence's state, zeros before its start), silu, unit vectors per q and k head, q's scale,
//                   beta = sigmoid, g = exp(-exp(A_log) softplus(a + dt_bias)).
//   conv_state:     the last (taps - 1) inputs of every sequence go into its state (a decode step's delta_prepare does that itself).
//   delta_rule:     the recurrence.  Columns of S never mix (each value channel is a recurrence of its own), so a wave
//                   owns a few columns of one head of one sequence: 16 (or 32) lanes share a column, each with a run of
//                   its rows in registers.  The wave walks over the sequence's tokens; q, k and g of a run of tokens are
//                   staged in LDS for all its lanes (the next run's are asked for before this one is worked on).  With
//                   kg = g k and qg = g q, both inner products of a token read the state as the token found it,
//                   u = beta (v - S^T kg),  o = S^T qg + (k . q) u,  and are summed over the column's lanes together, in
//                   the vector unit; then S <- g S + k u^T.  (A decay per head leaves the sums: g S^T k.)
//   gated_head_norm: o / rms(o) * weight * act(gate) per head, rounded once to the activation type.
//
// The state is kept transposed, [slot][head][value channel][key channel], so that a lane's rows are contiguous.
#include "common.h"
#include "fmsamd.h"
#include "short_conv.h"

#define DELTA_MAX_TAPS CONV_MAX_TAPS

__device__ __forceinline__ float sigmoid_f32(float z) { return 1.f / (1.f + expf(-z)); }

// Blocks of 1024 threads for steps of few tokens (short prompts, and callers that do not say where sequences start: a block per token
// and nothing else to hide a load's latency behind: the fewer passes a thread makes, the fewer round trips to memory follow one another).
template <typename W>
__global__ void __launch_bounds__(1024)
    delta_prepare_kernel(const float* __restrict__ proj, long ld, int col_b, const float* __restrict__ a, long lda, int col_a,
                         const W* __restrict__ conv_w, int taps, const float* __restrict__ a_log,
                         const float* __restrict__ dt_bias, const float* __restrict__ conv_state,
                         const int* __restrict__ seq_of_token, const int* __restrict__ slot_ids, float* __restrict__ qkv,
                         float* __restrict__ beta, float* __restrict__ decay, float* __restrict__ kq, int H, int G, int D, int Dv,
                         int per_channel, float q_scale) {
  extern __shared__ float y[];  // the C convolved channels of this token
  const int t = blockIdx.x;
  const int seq = seq_of_token[t];
  if (seq < 0) return;
  const int slot = slot_ids[seq];
  const int C = 2 * G * D + H * Dv;
  const int have = tokens_before(seq_of_token, t, seq, taps);
  const float* state = conv_state + (size_t)slot * (taps - 1) * C;
  // two channels a thread and pass, all their taps asked for before any is used
  for (int c0 = threadIdx.x; c0 < C; c0 += 2 * blockDim.x) {
    float x[2][DELTA_MAX_TAPS], w[2][DELTA_MAX_TAPS];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int c = c0 + e * blockDim.x;
#pragma unroll
      for (int j = 0; j < DELTA_MAX_TAPS; ++j) {
        const int d = taps - 1 - j;  // how far back this tap reaches
        x[e][j] = w[e][j] = 0.f;
        if (j < taps && c < C) {
          x[e][j] = d <= have ? proj[(size_t)(t - d) * ld + c] : state[(size_t)(taps - 1 + have - d) * C + c];
          w[e][j] = to_f32(conv_w[(size_t)c * taps + j]);
        }
      }
    }
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int c = c0 + e * blockDim.x;
      float acc = 0.f;
#pragma unroll
      for (int j = 0; j < DELTA_MAX_TAPS; ++j) acc = fmaf(w[e][j], x[e][j], acc);
      if (c < C) y[c] = acc / (1.f + expf(-acc));
    }
  }
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nwaves = blockDim.x >> 6;
  for (int head = wave; head < 2 * G; head += nwaves) {
    float* v = y + (size_t)head * D;
    float s = 0.f;
    for (int i = lane; i < D; i += WAVE) s = fmaf(v[i], v[i], s);
    s = wave_sum(s);
    const float inv = (head < G ? q_scale : 1.f) / sqrtf(s + 1e-6f);
    for (int i = lane; i < D; i += WAVE) v[i] *= inv;
  }
  __syncthreads();
  for (int head = wave; head < G; head += nwaves) {  // k . q of the finished vectors, which the recurrence's read-out needs
    float s = 0.f;
    for (int i = lane; i < D; i += WAVE) s = fmaf(y[(size_t)head * D + i], y[(size_t)(G + head) * D + i], s);
    s = wave_sum(s);
    if (lane == 0) kq[(size_t)t * G + head] = s;
  }
  for (int c = threadIdx.x; c < C; c += blockDim.x) qkv[(size_t)t * C + c] = y[c];
  for (int h = threadIdx.x; h < H; h += blockDim.x) beta[(size_t)t * H + h] = sigmoid_f32(proj[(size_t)t * ld + col_b + h]);
  const int per_head = per_channel ? D : 1;
  for (int i = threadIdx.x; i < H * per_head; i += blockDim.x) {
    const float z = a[(size_t)t * lda + col_a + i] + dt_bias[i];
    decay[(size_t)t * H * per_head + i] = expf(-expf(a_log[i / per_head]) * softplus_f32(z));
  }
}

// The same for prompts: a block takes 16 tokens and the channels of a q head and its k head, 256 value channels, or 256 decays (and
// the betas).  A thread has a channel of all 16 tokens and asks for its inputs at once, each of them once (the kernel above
// reads an input once for every tap, in eight passes of a block that has one token and all channels, and is bound by their
// round trips: 2277 tokens of 4096 channels 63 us, 41 here; with a decay per channel 78 and 47; the line between them stands at
// fmsamd_delta_prepare).
#define PREP_TOKENS 16
template <typename W>
__global__ void __launch_bounds__(256)
    delta_prepare_tokens_kernel(const float* __restrict__ proj, long ld, int col_b, const float* __restrict__ a, long lda, int col_a,
                                const W* __restrict__ conv_w, int taps, const float* __restrict__ a_log,
                                const float* __restrict__ dt_bias, const float* __restrict__ conv_state,
                                const int* __restrict__ seq_of_token, const int* __restrict__ slot_ids, float* __restrict__ qkv,
                                float* __restrict__ beta, float* __restrict__ decay, float* __restrict__ kq, int n_tokens, int H, int G,
                                int D, int Dv, int per_channel, float q_scale) {
  extern __shared__ float y[];  // q and k of the block's tokens: [16][2 D + 4]
  __shared__ int sq[PREP_TOKENS + DELTA_MAX_TAPS - 1];  // sequences, from the first token's earliest predecessor on
  __shared__ float inv[2][PREP_TOKENS];
  const int tb = blockIdx.x * PREP_TOKENS, tid = threadIdx.x, n = n_tokens - tb < PREP_TOKENS ? n_tokens - tb : PREP_TOKENS;
  const int C = 2 * G * D + H * Dv, v_units = (H * Dv + 255) / 256;
  int unit = blockIdx.y;
  if (tid < PREP_TOKENS + DELTA_MAX_TAPS - 1) {
    const int t = tb + tid - (DELTA_MAX_TAPS - 1);
    sq[tid] = t >= 0 && t < n_tokens ? seq_of_token[t] : -2;
  }
  __syncthreads();
  const int* own = sq + DELTA_MAX_TAPS - 1;  // own[i]: of token tb + i

  if (unit >= G + v_units) {  // decays and betas
    const int per = per_channel ? D : 1, c = (unit - G - v_units) * 256 + tid;
    for (int i = 0; i < n; ++i) {
      if (own[i] < 0) continue;
      const size_t t = tb + i;
      if (unit == G + v_units)
        for (int h = tid; h < H; h += 256) beta[t * H + h] = sigmoid_f32(proj[t * ld + col_b + h]);
      if (c < H * per) decay[t * H * per + c] = expf(-expf(a_log[c / per]) * softplus_f32(a[t * lda + col_a + c] + dt_bias[c]));
    }
    return;
  }

  bool one = true;  // all tokens and their predecessors are of one sequence
  for (int i = 1 - taps; i < PREP_TOKENS; ++i) one = one && own[i] == own[0];
  one = one && own[0] >= 0;
  auto convolve = [&](int c, float (&out)[PREP_TOKENS]) {
    float w[DELTA_MAX_TAPS];
#pragma unroll
    for (int j = 0; j < DELTA_MAX_TAPS; ++j) w[j] = j < taps ? to_f32(conv_w[(size_t)c * taps + j]) : 0.f;
    if (one) {
      float x[PREP_TOKENS + DELTA_MAX_TAPS - 1];  // x[r]: token tb + r - (taps - 1)
      const float* row = proj + (size_t)(tb - (taps - 1)) * ld + c;
#pragma unroll
      for (int r = 0; r < PREP_TOKENS + DELTA_MAX_TAPS - 1; ++r) x[r] = r < PREP_TOKENS + taps - 1 ? row[(size_t)r * ld] : 0.f;
#pragma unroll
      for (int i = 0; i < PREP_TOKENS; ++i) {
        float acc = 0.f;
#pragma unroll
        for (int j = 0; j < DELTA_MAX_TAPS; ++j) acc = j < taps ? fmaf(w[j], x[i + j], acc) : acc;
        out[i] = acc;
      }
    } else {
#pragma unroll
      for (int i = 0; i < PREP_TOKENS; ++i) {
        out[i] = 0.f;
        const int seq = own[i];
        if (seq < 0) continue;  // uniform
        int have = 0;           // predecessors in the step
        while (have < taps - 1 && own[i - have - 1] == seq) ++have;
        const float* state = conv_state + (size_t)slot_ids[seq] * (taps - 1) * C;
        float acc = 0.f;
#pragma unroll
        for (int j = 0; j < DELTA_MAX_TAPS; ++j) {
          const int d = taps - 1 - j;
          if (j < taps) acc = fmaf(w[j], d <= have ? proj[(size_t)(tb + i - d) * ld + c] : state[(size_t)(taps - 1 + have - d) * C + c], acc);
        }
        out[i] = acc;
      }
    }
#pragma unroll
    for (int i = 0; i < PREP_TOKENS; ++i) out[i] = out[i] / (1.f + expf(-out[i]));
  };

  float out[PREP_TOKENS];
  if (unit >= G) {  // values
    const int c = (unit - G) * 256 + tid;
    if (c >= H * Dv) return;
    convolve(2 * G * D + c, out);
#pragma unroll
    for (int i = 0; i < PREP_TOKENS; ++i)
      if (own[i] >= 0) qkv[(size_t)(tb + i) * C + 2 * G * D + c] = out[i];
    return;
  }
  const int stride = 2 * D + 4;
  for (int c = tid; c < 2 * D; c += 256) {
    convolve((c < D ? 0 : G * D - D) + unit * D + c, out);
#pragma unroll
    for (int i = 0; i < PREP_TOKENS; ++i) y[i * stride + c] = out[i];
  }
  __syncthreads();
  {
    const int i = tid / 16, part = tid % 16;  // 16 lanes a token
    const float *q = y + i * stride, *k = q + D;
    float qq = 0.f, kk = 0.f, dot = 0.f;
    for (int d = part; d < D; d += 16) qq = fmaf(q[d], q[d], qq), kk = fmaf(k[d], k[d], kk);
    const float iq = q_scale / sqrtf(row16_sum(qq) + 1e-6f), ik = 1.f / sqrtf(row16_sum(kk) + 1e-6f);
    for (int d = part; d < D; d += 16) dot = fmaf(q[d] * iq, k[d] * ik, dot);  // k . q of the finished vectors
    dot = row16_sum(dot);
    if (part == 0) {
      inv[0][i] = iq, inv[1][i] = ik;
      if (own[i] >= 0) kq[(size_t)(tb + i) * G + unit] = dot;
    }
  }
  __syncthreads();
  for (int c = tid; c < 2 * D; c += 256) {
    const int col = (c < D ? 0 : G * D - D) + unit * D + c;
    for (int i = 0; i < n; ++i)
      if (own[i] >= 0) qkv[(size_t)(tb + i) * C + col] = y[i * stride + c] * inv[c < D ? 0 : 1][i];
  }
}

// The same for a decode step, which also moves the convolution's state on: a block takes a sequence and the channels of a q head and
// its k head, blockDim value channels, or as many decays (and the betas).  A channel's window of inputs belongs to one thread, which
// reads it from the state, walks the sequence's tokens (one in a decode step) and writes it back, so no second kernel has to follow
// the last reader.  What bounds such a step is the chain of round trips of a block and the launches, not the bytes: a block of all
// channels takes them in passes.  8 sequences of 4096 channels (16 value heads of 128): 12.1 us and 4.5 us for the state behind it,
// 4.9 us here.
template <typename W>
__global__ void __launch_bounds__(512)
    delta_prepare_seqs_kernel(const float* __restrict__ proj, long ld, int col_b, const float* __restrict__ a, long lda, int col_a,
                              const W* __restrict__ conv_w, int taps, const float* __restrict__ a_log,
                              const float* __restrict__ dt_bias, float* __restrict__ conv_state, const int* __restrict__ seq_starts,
                              const int* __restrict__ seq_of_token, const int* __restrict__ slot_ids, float* __restrict__ qkv,
                              float* __restrict__ beta, float* __restrict__ decay, float* __restrict__ kq, int H, int G, int D, int Dv,
                              int per_channel, float q_scale) {
  extern __shared__ float y[];  // q and k of a token
  __shared__ float inv[2];
  const int b = blockIdx.x, tid = threadIdx.x, threads = blockDim.x;
  const int C = 2 * G * D + H * Dv, v_units = (H * Dv + threads - 1) / threads;
  const int unit = blockIdx.y;
  const int t0 = seq_starts[b], t1 = seq_starts[b + 1];
  const int slot_b = slot_ids[b];
  if (t0 >= t1) return;

  if (unit >= G + v_units) {  // decays and betas
    const int per = per_channel ? D : 1, c = (unit - G - v_units) * threads + tid;
    for (int t = t0; t < t1; ++t) {
      if (seq_of_token[t] < 0) continue;
      if (unit == G + v_units)
        for (int h = tid; h < H; h += threads) beta[(size_t)t * H + h] = sigmoid_f32(proj[(size_t)t * ld + col_b + h]);
      if (c < H * per)
        decay[(size_t)t * H * per + c] = expf(-expf(a_log[c / per]) * softplus_f32(a[(size_t)t * lda + col_a + c] + dt_bias[c]));
    }
    return;
  }

  const bool values = unit >= G;
  int c = -1;  // this thread's channel
  if (values) {
    const int v = (unit - G) * threads + tid;
    if (v < H * Dv) c = 2 * G * D + v;
  } else if (tid < 2 * D) {
    c = (tid < D ? 0 : G * D - D) + unit * D + tid;
  }
  const bool live = c >= 0;
  float w[DELTA_MAX_TAPS], x[DELTA_MAX_TAPS] = {};  // x: the inputs a token's taps meet, the token's own last
#pragma unroll
  for (int j = 0; j < DELTA_MAX_TAPS; ++j) w[j] = j < taps && live ? to_f32(conv_w[(size_t)c * taps + j]) : 0.f;
  float* state = nullptr;
  int before = -1;  // the last token's sequence
  auto leave = [&]() {  // the last inputs of a sequence, into its state
#pragma unroll
    for (int j = 1; j < DELTA_MAX_TAPS; ++j)
      if (j < taps && live) state[(size_t)(j - 1) * C + c] = x[j];
  };
  for (int t = t0; t < t1; ++t) {
    const float fresh = live ? proj[(size_t)t * ld + c] : 0.f;
    const int seq = seq_of_token[t];
    const bool first = seq != before;
    if (first && before >= 0) leave();  // a range may end in padding, or in another sequence's token
    before = seq;
    if (seq < 0) continue;
    if (first) {
      state = conv_state + (size_t)(seq == b ? slot_b : slot_ids[seq]) * (taps - 1) * C;
#pragma unroll
      for (int j = 0; j < DELTA_MAX_TAPS - 1; ++j) x[j] = j < taps - 1 && live ? state[(size_t)j * C + c] : 0.f;
    } else {
#pragma unroll
      for (int j = 0; j < DELTA_MAX_TAPS - 1; ++j) x[j] = x[j + 1];
    }
    float acc = 0.f;
#pragma unroll
    for (int j = 0; j < DELTA_MAX_TAPS; ++j) {
      x[j] = j == taps - 1 ? fresh : x[j];
      acc = fmaf(w[j], x[j], acc);
    }
    const float out = acc / (1.f + expf(-acc));
    if (values) {
      if (live) qkv[(size_t)t * C + c] = out;
      continue;
    }
    if (live) y[tid] = out;
    __syncthreads();
    const int lane = tid & 63, wave = tid >> 6;
    if (wave < 2) {  // of the q head, of the k head
      const float* v = y + wave * D;
      float s = 0.f;
      for (int i = lane; i < D; i += WAVE) s = fmaf(v[i], v[i], s);
      s = wave_sum(s);
      if (lane == 0) inv[wave] = (wave == 0 ? q_scale : 1.f) / sqrtf(s + 1e-6f);
    }
    __syncthreads();
    const float iq = inv[0], ik = inv[1];
    if (live) qkv[(size_t)t * C + c] = out * (tid < D ? iq : ik);
    if (wave == 0) {  // k . q of the finished vectors
      float s = 0.f;
      for (int i = lane; i < D; i += WAVE) s = fmaf(y[i] * iq, y[D + i] * ik, s);
      s = wave_sum(s);
      if (lane == 0) kq[(size_t)t * G + unit] = s;
    }
    if (t + 1 < t1) __syncthreads();  // y and inv are read
  }
  if (before >= 0) leave();
}

// --------------------------------------------------------------------------
// the recurrence
// --------------------------------------------------------------------------
#define DELTA_WAVES 4                       // waves of a block: they share the staged tokens
#define DELTA_THREADS (DELTA_WAVES * WAVE)

struct DeltaArgs {
  const float* qkv;    // [T, C]: q [G*D] | k [G*D] | v [H*Dv]
  const float* beta;   // [T, H]
  const float* decay;  // [T, H] or [T, H*D]
  const float* kq;     // [T, G]: k . q
  float* state;        // [slots][H][Dv][D]
  float* out;          // [T, H*Dv]
  const int* seq_starts;
  const int* seq_of_token;
  const int* slot_ids;
  int H, G, D, Dv, per_channel;
};

// The sums of two numbers over the PARTS lanes that share a column: a row of 16 lanes, or two rows.  With two rows the first
// step swaps the odd rows of u with the even rows of q, so that one row then sums u and its neighbour q, and a last swap of the
// result with itself gives both rows both sums: half the steps of two
// sums one after the other.  The recurrence issues about forty vector instructions a token and is bound by them: sequences of
// 900 and 1400 tokens, 16 heads of 128 by 128, 304 us instead of 321.
template <int PARTS>
__device__ __forceinline__ void row_sums(float& u, float& q) {
  if constexpr (PARTS == 32) {
    const auto halves = __builtin_amdgcn_permlane16_swap(__float_as_uint(u), __float_as_uint(q), false, false);
    const float both = row16_sum(__uint_as_float(halves[0]) + __uint_as_float(halves[1]));
    const auto rows = __builtin_amdgcn_permlane16_swap(__float_as_uint(both), __float_as_uint(both), false, false);  // rows [0, 0, 2, 2] and [1, 1, 3, 3]
    u = __uint_as_float(rows[0]), q = __uint_as_float(rows[1]);
  } else {
    u = row16_sum(u), q = row16_sum(q);
  }
}

// PARTS: lanes that share a column of S (16, or 32 where a step has few sequences and heads: twice the blocks, half the
// work a token and lane).  R: rows of S per lane (D <= PARTS R).  TC: tokens staged at a time.  A block's four waves own
// 256 / PARTS columns of one head and share the staged tokens (staging costs instructions, and four waves split them).
// The next run's q, k and g are asked for from global memory before this run is worked on and wait in registers meanwhile.
template <int PARTS, int R, int TC, bool PER_CHANNEL>
__global__ void __launch_bounds__(DELTA_THREADS) delta_rule_kernel(DeltaArgs a) {
  constexpr int DELTA_COLS = DELTA_THREADS / PARTS;  // columns of S the block owns
  constexpr int DELTA_PARTS = PARTS;
  constexpr int DP = R * DELTA_PARTS;          // padded key size
  constexpr int NI = TC * DP / DELTA_THREADS;  // staged elements a thread
  static_assert(TC * DP % DELTA_THREADS == 0 && TC * DELTA_COLS <= DELTA_THREADS, "the staging loops assume this");
  // With a decay per channel: qg = g q, kg = g k, k and g.  With one decay per head the factor leaves the inner products
  // (S^T (g k) = g S^T k): q and k alone are staged, and g as one number a token; half the LDS traffic.
  constexpr int CH = PER_CHANNEL ? TC : 1;
  __shared__ __attribute__((aligned(16))) float qg[TC][DP];
  __shared__ __attribute__((aligned(16))) float kg[CH][DP];
  __shared__ __attribute__((aligned(16))) float kk[TC][DP];
  __shared__ __attribute__((aligned(16))) float gg[CH][DP];
  __shared__ float vv[TC][DELTA_COLS];
  __shared__ float gs[TC];
  __shared__ float bb[TC];
  __shared__ float kqs[TC];
  __shared__ float oo[TC][DELTA_COLS];

  const int b = blockIdx.x, h = blockIdx.y;
  const int t0 = uniform_load(a.seq_starts + b), t1 = uniform_load(a.seq_starts + b + 1), slot = uniform_load(a.slot_ids + b);
  if (t0 >= t1 || uniform_load(a.seq_of_token + t0) < 0) return;
  const int lane = threadIdx.x;  // of the block
  const int part = lane % DELTA_PARTS, col = lane / DELTA_PARTS;
  const int j = blockIdx.z * DELTA_COLS + col;  // this lane's column of S
  const int H = a.H, G = a.G, D = a.D, Dv = a.Dv;
  const int C = 2 * G * D + H * Dv;
  const int kh = h / (H / G);
  const bool live = j < Dv;

  float S[R];
  float* srow = a.state + (((size_t)slot * H + h) * Dv + (live ? j : 0)) * D + part * R;
  // A lane's rows lie next to each other: 16 bytes at a time where a column is whole.  A decode step moves little else: 16 heads of 128 by 128, us, four
  // bytes at a time (a lane's neighbour 32 bytes on) and so, 1 sequence 4.5 and 3.5, 8 11.0 and 5.5, 32 36.5 and 14.8; 64 of 32 heads 120 and 51 (5.3
  // TB/s); 8 of 8 heads of 256 by 256 28.4 and 10.3.
  const bool pieces = R % 4 == 0 && D == R * PARTS && ((uintptr_t)a.state & 15) == 0;  // uniform
  if (pieces) {
#pragma unroll
    for (int r = 0; r < R; r += 4) {
      const f32x4 v = live ? *reinterpret_cast<const f32x4*>(srow + r) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < 4 && r + i < R; ++i) S[r + i] = v[i];
    }
  } else {
#pragma unroll
    for (int r = 0; r < R; ++r) S[r] = (live && part * R + r < D) ? srow[r] : 0.f;
  }

  // what a lane fetches of a run: NI (q, k, g) triples, one value, and beta and k . q of one token
  float pq[NI], pk[NI], pg[PER_CHANNEL ? NI : 1], pv = 0.f, pb = 0.f, pkq = 0.f, pgs = 1.f;
  const int vt = lane / DELTA_COLS, vc = lane % DELTA_COLS;  // the (token, column) whose value and output this lane moves
  const int vj = blockIdx.z * DELTA_COLS + vc;
  auto fetch = [&](int tb) {
#pragma unroll
    for (int it = 0; it < NI; ++it) {
      const int idx = it * DELTA_THREADS + lane;
      const int tt = idx / DP, i = idx % DP;
      const int t = tb + tt;
      // past the run's last token (and past the key channels) a token that changes nothing: k = 0, g = 1
      pq[it] = pk[it] = 0.f;
      if constexpr (PER_CHANNEL) pg[it] = 1.f;
      if (t < t1 && i < D) {
        const float* row = a.qkv + (size_t)t * C;
        pq[it] = row[kh * D + i];
        pk[it] = row[G * D + kh * D + i];
        if constexpr (PER_CHANNEL) pg[it] = a.decay[((size_t)t * H + h) * D + i];
      }
    }
    pgs = 1.f;
    pb = 0.f;
    pv = (vt < TC && tb + vt < t1 && vj < Dv) ? a.qkv[(size_t)(tb + vt) * C + 2 * G * D + h * Dv + vj] : 0.f;
    if (lane < TC && tb + lane < t1) {
      pb = a.beta[(size_t)(tb + lane) * H + h];
      pkq = a.kq[(size_t)(tb + lane) * G + kh];
      if constexpr (!PER_CHANNEL) pgs = a.decay[(size_t)(tb + lane) * H + h];
    }
  };
  fetch(t0);

  for (int tb = t0; tb < t1; tb += TC) {
    const int n = t1 - tb < TC ? t1 - tb : TC;
#pragma unroll
    for (int it = 0; it < NI; ++it) {
      const int idx = it * DELTA_THREADS + lane;
      const int tt = idx / DP, i = idx % DP;
      kk[tt][i] = pk[it];
      if constexpr (PER_CHANNEL) {
        qg[tt][i] = pq[it] * pg[it];
        kg[tt][i] = pk[it] * pg[it];
        gg[tt][i] = pg[it];
      } else {
        qg[tt][i] = pq[it];
      }
    }
    if (vt < TC) vv[vt][vc] = pv;
    if (lane < TC) bb[lane] = pb, kqs[lane] = pkq, gs[lane] = pgs;
    block_sync_lds();
    if (tb + TC < t1) fetch(tb + TC);  // under way while this run is worked on

    // a token's operands are read from LDS into registers while the token before it is worked on (two sets, in turn)
    struct Operands {
      float kg[PER_CHANNEL ? R : 1], qg[R], kk[R], gg[PER_CHANNEL ? R : 1], g, beta, v, kq;
    };
    auto load = [&](Operands& x, int tt) {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        x.qg[r] = qg[tt][part * R + r];
        x.kk[r] = kk[tt][part * R + r];
        if constexpr (PER_CHANNEL) {
          x.kg[r] = kg[tt][part * R + r];
          x.gg[r] = gg[tt][part * R + r];
        }
      }
      x.g = gs[tt];
      x.beta = bb[tt];
      x.v = vv[tt][col];
      x.kq = kqs[tt];
    };
    auto work = [&](const Operands& x, int tt) {
      float du0 = 0.f, du1 = 0.f, dq0 = 0.f, dq1 = 0.f;
#pragma unroll
      for (int r = 0; r < R; r += 2) {
        du0 = fmaf(S[r], PER_CHANNEL ? x.kg[PER_CHANNEL ? r : 0] : x.kk[r], du0);
        dq0 = fmaf(S[r], x.qg[r], dq0);
        du1 = fmaf(S[r + 1], PER_CHANNEL ? x.kg[PER_CHANNEL ? r + 1 : 0] : x.kk[r + 1], du1);
        dq1 = fmaf(S[r + 1], x.qg[r + 1], dq1);
      }
      float du = du0 + du1, dq = dq0 + dq1;
      row_sums<PARTS>(du, dq);
      if constexpr (!PER_CHANNEL) du *= x.g, dq *= x.g;  // the head's decay, taken out of the sums
      const float u = x.beta * (x.v - du);
#pragma unroll
      for (int r = 0; r < R; ++r) S[r] = fmaf(x.kk[r], u, (PER_CHANNEL ? x.gg[PER_CHANNEL ? r : 0] : x.g) * S[r]);
      if (part == 0) oo[tt][col] = fmaf(x.kq, u, dq);
    };
    // Tokens go in pairs, and a run of an odd number works on one staged token that changes nothing (beta = 0, k = 0,
    // g = 1; its output is not copied out): the loop's body then has no branch around its loads, and the compiler can
    // let a token's work wait for its own operands only, not for the ones just asked for.
    Operands xa, xb;
    load(xa, 0);
    const int n2 = TC > 1 ? (n + 1) & ~1 : 1;
    for (int tt = 0; tt < n2; tt += 2) {
      load(xb, tt + 1 < TC ? tt + 1 : tt);
      work(xa, tt);
      if constexpr (TC > 1) {
        load(xa, tt + 2 < TC ? tt + 2 : tt);
        work(xb, tt + 1);
      }
    }
    block_sync_lds();
    if (vt < n && vj < Dv) a.out[(size_t)(tb + vt) * H * Dv + h * Dv + vj] = oo[vt][vc];
    block_sync_lds();  // the run's reads are done before the next one is written
  }
  if (live && pieces) {
    if constexpr (R % 4 == 0) {
#pragma unroll
      for (int r = 0; r < R; r += 4) *reinterpret_cast<f32x4*>(srow + r) = f32x4{S[r], S[r + 1], S[r + 2], S[r + 3]};
    }
  } else if (live) {
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (part * R + r < D) srow[r] = S[r];
  }
}

// out[t, h, j] = o / rms_j(o) * weight[j] * act(gate[t, h, j]) * out_scale; one wave per (token, head).  Padding rows become zeros:
// a product over all rows follows, which a fill kernel in front of it cost 4.7 us of a decode layer.
template <typename T, typename W>
__global__ void __launch_bounds__(256)
    gated_head_norm_kernel(const float* __restrict__ o, const float* __restrict__ gate, long ldg, const W* __restrict__ weight,
                           float eps, int act, float out_scale, T* __restrict__ out, long ldo, const int* __restrict__ seq_of_token,
                           int n_tokens, int H, int Dv) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const long pair = (long)blockIdx.x * 4 + wave;
  if (pair >= (long)n_tokens * H) return;
  const int t = (int)(pair / H), h = (int)(pair % H);
  if (seq_of_token[t] < 0) {
    for (int j = lane; j < Dv; j += WAVE) out[(size_t)t * ldo + (size_t)h * Dv + j] = from_f32<T>(0.f);
    return;
  }
  const float* row = o + ((size_t)t * H + h) * Dv;
  float s = 0.f;
  for (int j = lane; j < Dv; j += WAVE) s = fmaf(row[j], row[j], s);
  s = wave_sum(s);
  const float inv = 1.f / sqrtf(s / (float)Dv + eps);
  for (int j = lane; j < Dv; j += WAVE) {
    const float g = fms_activate(gate[(size_t)t * ldg + (size_t)h * Dv + j], act);
    out[(size_t)t * ldo + (size_t)h * Dv + j] = from_f32<T>(row[j] * inv * to_f32(weight[j]) * g * out_scale);
  }
}

// The same for heads of 64, 128 or 256 and aligned rows: a lane has four neighbours, a wave 256 columns.  Bound by its bytes.  2277 tokens of 16 heads of 128: 13 us where the kernel above takes 21; of 32 of 64: 14 and 28.
template <typename T, typename W, int LANES>
__global__ void __launch_bounds__(256)
    gated_head_norm4_kernel(const float* __restrict__ o, const float* __restrict__ gate, long ldg, const W* __restrict__ weight,
                            float eps, int act, float out_scale, T* __restrict__ out, long ldo, const int* __restrict__ seq_of_token,
                            int n_tokens, int H) {
  constexpr int DV = 4 * LANES, PER = WAVE / LANES;
  typedef T T4 __attribute__((ext_vector_type(4)));
  const int lane = threadIdx.x & 63, j = lane % LANES * 4;
  const long pair = ((long)blockIdx.x * 4 + (threadIdx.x >> 6)) * PER + lane / LANES;
  if (pair >= (long)n_tokens * H) return;
  const int t = (int)(pair / H), h = (int)(pair % H);
  T* const to = out + (size_t)t * ldo + (size_t)h * DV + j;
  if (seq_of_token[t] < 0) {
    *(T4*)to = T4{};
    return;
  }
  const f32x4 v = *(const f32x4*)(o + (size_t)pair * DV + j), g = *(const f32x4*)(gate + (size_t)t * ldg + (size_t)h * DV + j);
  float s = fmaf(v[0], v[0], fmaf(v[1], v[1], fmaf(v[2], v[2], v[3] * v[3])));
#pragma unroll
  for (int off = LANES / 2; off > 0; off >>= 1) s += __shfl_xor(s, off, WAVE);
  const float inv = 1.f / sqrtf(s / (float)DV + eps);
  T4 r;
#pragma unroll
  for (int e = 0; e < 4; ++e) r[e] = from_f32<T>(v[e] * inv * to_f32(weight[j + e]) * fms_activate(g[e], act) * out_scale);
  *(T4*)to = r;
}

// --------------------------------------------------------------------------
extern "C" int fmsamd_delta_prepare(const float* proj, long ld, int col_b, const float* a, long lda, int col_a, const void* conv_w,
                                    int conv_dtype, int taps, const float* a_log, const float* dt_bias, float* conv_state,
                                    const int* seq_of_token, const int* slot_ids, float* qkv, float* beta, float* decay,
                                    float* kq, int n_tokens, int heads, int kv_heads, int dim, int vdim, int per_channel,
                                    float q_scale, const int* seq_starts, int n_seqs, int single_tokens, hipStream_t stream) {
  if (n_tokens == 0) return 0;
  FMS_REQUIRE(n_tokens > 0 && heads > 0 && kv_heads > 0 && heads % kv_heads == 0 && dim > 0 && vdim > 0,
              "delta_prepare: bad sizes heads=%d kv_heads=%d dim=%d vdim=%d", heads, kv_heads, dim, vdim);
  FMS_REQUIRE(taps >= 1 && taps <= DELTA_MAX_TAPS, "delta_prepare: %d taps (1 to %d)", taps, DELTA_MAX_TAPS);
  const long C = 2L * kv_heads * dim + (long)heads * vdim;
  FMS_REQUIRE(ld >= C && col_b >= 0 && col_b + heads <= ld, "delta_prepare: rows of %ld for %ld channels", ld, C);
  FMS_REQUIRE(C * 4 <= 64 * 1024, "delta_prepare: %ld channels do not fit one block's LDS", C);
  FMS_REQUIRE(col_a >= 0 && col_a + heads * (per_channel ? dim : 1) <= lda, "delta_prepare: the decay's columns leave its rows");
  FMS_REQUIRE(seq_starts == nullptr || n_seqs > 0, "delta_prepare: no sequences");
  const size_t lds = (size_t)C * sizeof(float);
  const int threads = n_tokens <= 64 ? 1024 : 256;
  // 16 tokens a block where that is less work than it is a longer way: some 21 us for loads, sums and gates one after the other, whatever
  // the sizes, and then half the time a token.  The other kernel's way is its passes over the columns.  Microseconds of the other kernel
  // and of this one (with conv_state behind them):
  //   8192 columns: 65 tokens 32 and 21.7, 2277 121 and 59;  6144 (4096 channels with a decay per channel): 65 22.3 and 21.4, 2277 70 and 48;
  //   4096: 65 to 256 tokens 19 to 20 and 21 to 22, 512 24.5 and 22.9, 2277 56.3 and 42.6;
  //   3072: 512 19.6 and 22.5, 2277 46.0 and 39.2;  2048: 2277 35.3 and 33.6, 3000 40.6 and 33.7;  1024: 2277 24.1 and 26.9, 8192 56.5 and 43.9;
  //   384: 2277 15.2 and 22.4, 8192 40 and 29.8;  heads of 256: 4096 columns, 512 tokens 23.7 and 37.2, 2277 61.5 and 57.8; 1536, 2277 27.9
  //     and 45.5, 8192 70 and 54.
  // Blocks of several sequences ask for every tap by itself: 200 sequences of 17 60 and 87 (2304 columns), 86 and 98 (4096), 102 and 109
  // (6144), 175 and 171 (8192); of 4096 columns 12 of 100 35.4 and 37.6, 8 of 130 35 and 33.4.
  const long decays = heads * (long)(per_channel ? dim : 1), columns = C + decays, work = n_tokens * columns;
  const long units = kv_heads + (heads * (long)vdim + 255) / 256 + (decays + 255) / 256;
  const bool long_seqs = n_tokens >= 128L * n_seqs;
  const bool pays = dim > 128 ? long_seqs && work >= 8000000
                              : columns >= 8192 || (long_seqs && (columns >= 6144 || work >= 5000000 || (columns >= 4096 && n_tokens >= 512)));
  const bool by_tokens = n_tokens > 64 && dim <= 256 && units <= 65535 && pays;
  // A sequence a block, and no kernel for the state behind it, where sequences bring a token each (a decode step, with or without
  // rows of padding behind its sequences, so that it is the same kernel in a captured step and in an eager one) or less on average.  More
  // tokens a sequence would follow one another in a block that the others spread over blocks.
  const int seq_threads = dim <= 128 ? 256 : 512;
  const long seq_units = kv_heads + (heads * (long)vdim + seq_threads - 1) / seq_threads + (decays + seq_threads - 1) / seq_threads;
  const bool by_seqs = seq_starts != nullptr && (single_tokens || n_tokens <= n_seqs) && dim <= 256 && seq_units <= 65535;
  const dim3 grid(ceil_div(n_tokens, PREP_TOKENS), (unsigned)units);
  const size_t token_lds = (size_t)PREP_TOKENS * (2 * dim + 4) * sizeof(float);
#define FMS_PREP(W)                                                                                                   \
  do {                                                                                                                \
    if (by_seqs)                                                                                                      \
      delta_prepare_seqs_kernel<W><<<dim3(n_seqs, (unsigned)seq_units), seq_threads, 2 * dim * sizeof(float), stream>>>( \
          proj, ld, col_b, a, lda, col_a, (const W*)conv_w, taps, a_log, dt_bias, conv_state, seq_starts, seq_of_token, slot_ids, qkv, \
          beta, decay, kq, heads, kv_heads, dim, vdim, per_channel, q_scale);                                         \
    else if (by_tokens)                                                                                               \
      delta_prepare_tokens_kernel<W><<<grid, 256, token_lds, stream>>>(proj, ld, col_b, a, lda, col_a, (const W*)conv_w, taps, a_log, \
                                                                       dt_bias, conv_state, seq_of_token, slot_ids, qkv, beta, decay, \
                                                                       kq, n_tokens, heads, kv_heads, dim, vdim, per_channel, q_scale); \
    else                                                                                                              \
      delta_prepare_kernel<W><<<n_tokens, threads, lds, stream>>>(proj, ld, col_b, a, lda, col_a, (const W*)conv_w, taps, a_log, \
                                                                  dt_bias, conv_state, seq_of_token, slot_ids, qkv, beta, decay, \
                                                                  kq, heads, kv_heads, dim, vdim, per_channel, q_scale); \
  } while (0)
  if (conv_dtype == FMS_F32) FMS_PREP(float);
  else if (conv_dtype == FMS_BF16) FMS_PREP(bf16);
  else FMS_REQUIRE(false, "delta_prepare: unknown dtype %d", conv_dtype);
#undef FMS_PREP
  FMS_LAUNCH_CHECK("delta_prepare");
  if (taps > 1 && !by_seqs) {
    move_conv_state(proj, ld, taps, conv_state, seq_of_token, slot_ids, n_tokens, (int)C, threads, seq_starts, n_seqs, stream);
    FMS_LAUNCH_CHECK("conv_state");
  }
  return 0;
}

extern "C" int fmsamd_delta_rule(const float* qkv, const float* beta, const float* decay, const float* kq, float* state,
                                 float* out, const int* seq_starts, const int* seq_of_token, const int* slot_ids, int n_seqs, int heads,
                                 int kv_heads, int dim, int vdim, int per_channel, int single_tokens, hipStream_t stream) {
  if (n_seqs == 0) return 0;
  FMS_REQUIRE(n_seqs > 0 && heads > 0 && kv_heads > 0 && heads % kv_heads == 0 && dim > 0 && vdim > 0,
              "delta_rule: bad sizes heads=%d kv_heads=%d dim=%d vdim=%d", heads, kv_heads, dim, vdim);
  FMS_REQUIRE(dim <= 256, "delta_rule: %d key channels (at most 256)", dim);
  DeltaArgs a{qkv, beta, decay, kq, state, out, seq_starts, seq_of_token, slot_ids, heads, kv_heads, dim, vdim, per_channel};
  // Few sequences and heads (a prompt alone): 32 lanes a column instead of 16, so that the step has twice the blocks and a
  // token costs every wave half the work; with many blocks anyway, 16 lanes (fewer reduction steps a token).
  const bool wide = !single_tokens && dim > 32 && (long)n_seqs * heads * ceil_div(vdim, 16) <= 512;
  const int cols = DELTA_THREADS / (wide ? 32 : 16);
  FMS_REQUIRE(heads <= 65535 && ceil_div(vdim, cols) <= 65535, "delta_rule: too many heads or value channels for one launch");
  const dim3 grid(n_seqs, heads, ceil_div(vdim, cols));
#define FMS_DR(P, R, TC)                                                                        \
  do {                                                                                          \
    if (per_channel) delta_rule_kernel<P, R, TC, true><<<grid, DELTA_THREADS, 0, stream>>>(a);  \
    else delta_rule_kernel<P, R, TC, false><<<grid, DELTA_THREADS, 0, stream>>>(a);             \
  } while (0)
  // single_tokens: every sequence brings one token (a decode step).  Staging room for one pass of the block's threads
  // is then enough, and a block that small leaves the compute unit's LDS to many more blocks.
  if (single_tokens) {
    if (dim <= 32) FMS_DR(16, 2, 8);
    else if (dim <= 64) FMS_DR(16, 4, 4);
    else if (dim <= 128) FMS_DR(16, 8, 2);
    else FMS_DR(16, 16, 1);
  } else if (wide) {
    if (dim <= 64) FMS_DR(32, 2, 16);
    else if (dim <= 128) FMS_DR(32, 4, 16);
    else FMS_DR(32, 8, 8);
  } else if (dim <= 32) FMS_DR(16, 2, 16);
  else if (dim <= 64) FMS_DR(16, 4, 16);
  else if (dim <= 128) FMS_DR(16, 8, 16);
  else FMS_DR(16, 16, 8);
#undef FMS_DR
  FMS_LAUNCH_CHECK("delta_rule");
  return 0;
}

extern "C" int fmsamd_gated_head_norm(const float* o, const float* gate, long ldg, const void* weight, int weight_dtype, float eps,
                                      int act, float out_scale, void* out, int out_dtype, long ldo, const int* seq_of_token,
                                      int n_tokens, int heads, int vdim, hipStream_t stream) {
  if (n_tokens == 0) return 0;
  FMS_REQUIRE(n_tokens > 0 && heads > 0 && vdim > 0 && ldg >= (long)heads * vdim && ldo >= (long)heads * vdim,
              "gated_head_norm: bad sizes heads=%d vdim=%d", heads, vdim);
  FMS_REQUIRE(act >= 0 && act <= FMS_ACT_LAST, "gated_head_norm: unknown activation %d", act);
  const size_t out_piece = out_dtype == FMS_F32 ? 16 : 8;
  const bool fours = (vdim == 64 || vdim == 128 || vdim == 256) && ldg % 4 == 0 && ldo % 4 == 0 && ((uintptr_t)o | (uintptr_t)gate) % 16 == 0 &&
                     (uintptr_t)out % out_piece == 0;
  const int blocks = ceil_div((long)n_tokens * heads, fours ? 1024 / vdim : 4);
#define FMS_GHN4(T, W, LANES)                                                                                                  \
  gated_head_norm4_kernel<T, W, LANES><<<blocks, 256, 0, stream>>>(o, gate, ldg, (const W*)weight, eps, act, out_scale, (T*)out, ldo, \
                                                                   seq_of_token, n_tokens, heads)
#define FMS_GHN(T, W)                                                                                                          \
  do {                                                                                                                         \
    if (fours && vdim == 64)                                                                                                   \
      FMS_GHN4(T, W, 16);                                                                                                      \
    else if (fours && vdim == 128)                                                                                             \
      FMS_GHN4(T, W, 32);                                                                                                      \
    else if (fours)                                                                                                            \
      FMS_GHN4(T, W, 64);                                                                                                      \
    else                                                                                                                       \
      gated_head_norm_kernel<T, W><<<blocks, 256, 0, stream>>>(o, gate, ldg, (const W*)weight, eps, act, out_scale, (T*)out, ldo, \
                                                               seq_of_token, n_tokens, heads, vdim);                           \
  } while (0)
  if (out_dtype == FMS_F32 && weight_dtype == FMS_F32) FMS_GHN(float, float);
  else if (out_dtype == FMS_BF16 && weight_dtype == FMS_F32) FMS_GHN(bf16, float);
  else if (out_dtype == FMS_BF16 && weight_dtype == FMS_BF16) FMS_GHN(bf16, bf16);
  else if (out_dtype == FMS_F32 && weight_dtype == FMS_BF16) FMS_GHN(float, bf16);
  else FMS_REQUIRE(false, "gated_head_norm: unknown dtypes %d, %d", out_dtype, weight_dtype);
#undef FMS_GHN
#undef FMS_GHN4
  FMS_LAUNCH_CHECK("gated_head_norm");
  return 0;
}
