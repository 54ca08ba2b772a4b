// The gated delta rule of delta_rule.hip for prompts, in runs of 16 tokens on the matrix unit.
//
//   S <- g * S;  u = beta (v - S^T k);  S <- S + k u^T;  o = S^T q          (S: [key channels, value channels] of a head)
//
// Within a run that starts from the state S0, with G_i the product of the decays up to token i (per head or per key
// channel) and R_ij = G_i / G_j that of the decays behind token j:
//
//   (I + A) U = diag(beta) (V - (G * K) S0),      A_ij = beta_i sum_d k_id k_jd R_ijd   for j < i
//   U = Y - W S0            with (I + A) Y = diag(beta) V and (I + A) W = diag(beta) (G * K)
//   O = (G * Q) S0 + P U    with P_ij = sum_d q_id k_jd R_ijd                           for j <= i
//   S = G_15 * S0 + sum_j (R_15,j * k_j) u_j^T
//
// Two kernels.  delta_runs_prepare: everything that does not need the state (Y, W, G * Q, P, R_15 * K), a block per run and
// head, so all runs at once; sums, decays and the triangular solve in 64 bits, every result rounded once to float32.
// delta_runs: the chain over a sequence's runs, a block per (sequence, head, 16 value channels): W S0, (G * Q) S0 and P U in
// float32, u and the update of S in 64 bits, S itself rounded to float32 once a run.  A wave keeps a
// quarter of S's rows in registers as 16x16x4 products take and leave them (register e of a lane is row 4 (lane / 16) + e: product
// e of a tile takes exactly these rows as its four; the 64-bit product leaves row 4 e + lane / 16 there, so that R_15 * K has its
// rows in that order).  What it
// multiplies is asked for two runs ahead, straight into registers, in the order in which the first kernel left it (the loads
// stand among the products: all of them at a run's start cost 0.16 us a run).
// Row r of a run's 16-row tiles is token 4 (r % 4) + r / 4: product e of a sum over the tokens then takes tokens 4 e to 4 e + 3,
// so that sums grow from the oldest token (the one that the decays have made smallest) to the newest.
//
// Sequences of 777 and 1500 tokens, 16 heads of 128 by 128: 132 us (138 with a decay per key channel), of which the first kernel
// takes 39 (44), where the kernel that goes token by token takes 305 (350), bound by some 45 vector instructions a token.  The first
// kernel is near what its 77 MB of results and 40 MB of inputs take; a run of the chain is 1 us, of which its 25 products a wave are
// 0.45 and the rest is the way of the partial sums through LDS and what a compute unit takes in.
// Errors against 64 bits (300 tokens, heads of 128 by 128), this kernel and the other one: outputs 5.5e-8 and 6.6e-8 for decays
// around 0.5, 6.9e-8 and 9.8e-8 around 0.86, 1.2e-7 and 3.2e-7 around 0.999; the state 3.8e-8 and 5.1e-8, 4.2e-8 and 7.5e-8,
// 1.0e-7 and 3.7e-7; where keys are alike, outputs 5.8e-8 and 6.7e-8, 8.9e-8 and 1.0e-7, 1.3e-7 and 3.9e-7, the state 4.0e-8 and
// 5.1e-8, 6.2e-8 and 8.0e-8, 1.2e-7 and 4.9e-7.  (With the update in float32 a run is 0.16 us shorter, and the state is up to a fifth
// further off than token by token where decays are fast: a sum of 16 products then rounds more often than the decays forget.)
#include "common.h"
#include "fmsamd.h"

#include <type_traits>

typedef double f64x4 __attribute__((ext_vector_type(4)));

#define RUN 16               // tokens of a run
#define RUNS_THREADS 256     // threads of a block of either kernel

// What delta_runs_prepare leaves of one run of one head, in floats:
//   W, G * Q, R_15 * K: [D / 16 tiles][64 lanes][4], lane l of tile t holding for e < 4
//       (G * Q)[row l % 16][16 t + 4 (l / 16) + e] and W likewise, (R_15 * K)[token 4 e + l / 16][16 t + row_token(l % 16)]
//   Y: [Dv / 16 tiles][64][4], lane l holding Y[token 4 e + l / 16][16 t + l % 16]
//   P without its diagonal: [4][64], P[row l % 16][token 4 e + l / 16] at e, l; then the diagonal, by tokens
//   G_15: [D]
__host__ __device__ static inline size_t run_floats(int D, int Dv) { return (size_t)RUN * (3 * D + Dv + RUN + 1) + D; }
__device__ __forceinline__ int row_token(int r) { return 4 * (r % 4) + r / 4; }  // and a token's row

// Run c of sequence b is place starts[b] / 16 + b + c: sequences of any length never meet, and n tokens in s sequences
// take at most n / 16 + s places.
// Long steps go in pieces, so that the workspace stays bounded: a piece is the runs whose first token is one of p0 .. p1 (multiples
// of 16), which are places from p0 / 16 on, (p1 - p0) / 16 + s at most.  The state passes from piece to piece through memory, as it
// is: the pieces change no bit.  A piece should hold as many sequences as the chip has blocks for (four with 16 heads of 128 by 128):
// in pieces of 128, 256, 384 and 512 MB and as one, 8 sequences of 1000 tokens take 417, 368 and 322 us (266 MB is one), 4 of 4000 1713,
// 1065, 1001, 667 and 616, 16 of 2000 2255, 1629, 1540, 1504 and 1970, one of 16000 1209, 1221, 1200, 1209 and 1197.
#define RUNS_WORKSPACE (512L << 20)  // bytes: 15600 tokens of 16 heads of 128 by 128

struct RunsArgs {
  const float* qkv;    // [T, C]: q [G*D] | k [G*D] | v [H*Dv]
  const float* beta;   // [T, H]
  const float* decay;  // [T, H] or [T, H*D]
  float* state;        // [slots][H][Dv][D]
  float* out;          // [T, H*Dv]
  float* runs;         // [places][H][run_floats]
  const int* seq_starts;
  const int* seq_of_token;
  const int* slot_ids;
  int n_seqs, H, G, D, Dv;
  int p0, p1;          // the piece
};

// Products of decays may underflow to nothing; a quotient of two of them is formed from decays of at least this (16 of
// them stay above 64 bits' smallest number).  What a smaller decay lets through is at most this much of a term of size one.
#define LEAST_DECAY 1e-18

// A block: 256 threads.  A thread first holds a channel of q and k of all 16 tokens, then a pair of tokens of A and P, then a
// column of W or Y, which it solves in registers: 120 fused multiply-adds, A from LDS, every lane the same address.  (The
// columns of A above its diagonal are never read, so that a token that is no number reaches only those behind it.)
template <bool PER_CHANNEL>
__global__ void __launch_bounds__(RUNS_THREADS, PER_CHANNEL ? 3 : 4) delta_runs_prepare_kernel(RunsArgs a) {
  extern __shared__ __attribute__((aligned(16))) char shared[];
  using KEY = typename std::conditional<PER_CHANNEL, double, float>::type;  // scaled by products of decays: 64 bits
  const int D = a.D, Dv = a.Dv, H = a.H, G = a.G;
  const int KS = D + 4;                         // stride of the staged rows
  double* A = (double*)shared;                  // [16][16]
  double* gp = A + RUN * RUN;                   // [16] one decay per head: its products up to each token
  float* gs = (float*)(gp + RUN);               // [16] the decays
  float* bs = gs + RUN;                         // [16] beta, 0 past the run's end
  KEY* kr = (KEY*)(bs + RUN);                   // [16][KS] k of the row's token (PER_CHANNEL: G k)
  KEY* qr = kr + RUN * KS;                      // [16][KS] q (PER_CHANNEL: G q)
  KEY* kc = PER_CHANNEL ? qr + RUN * KS : kr;   // [16][KS] k of the column's token (PER_CHANNEL: k / G)
  float* w = (float*)(qr + RUN * KS);           // [16][KS], takes the place of kc

  const int place = a.p0 / RUN + blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
  // the sequence whose places this one is among: the last with first_run <= place
  int b = 0;
  for (int lo = 0, hi = a.n_seqs; lo + 1 < hi;) {
    const int mid = (lo + hi) / 2;
    if (uniform_load(a.seq_starts + mid) / RUN + mid <= place) lo = b = mid;
    else hi = mid;
  }
  const int t0 = uniform_load(a.seq_starts + b), t1 = uniform_load(a.seq_starts + b + 1);
  const int tb = t0 + (place - t0 / RUN - b) * RUN;
  if (tb >= t1 || tb < a.p0 || tb >= a.p1 || uniform_load(a.seq_of_token + t0) < 0) return;
  const int n = t1 - tb < RUN ? t1 - tb : RUN;
  const int C = 2 * G * D + H * Dv, kh = h / (H / G);
  float* run = a.runs + ((size_t)blockIdx.x * H + h) * run_floats(D, Dv);
  float *oW = run, *oQ = oW + RUN * D, *oK = oQ + RUN * D, *oY = oK + RUN * D, *oP = oY + RUN * Dv, *oG = oP + RUN * (RUN + 1);

  // Tokens past the run's end: k = q = v = 0, beta = 0, g = 1.
  if (tid < RUN) {
    bs[tid] = tid < n ? a.beta[(size_t)(tb + tid) * H + h] : 0.f;
    if constexpr (!PER_CHANNEL) gs[tid] = tid < n ? a.decay[(size_t)(tb + tid) * H + h] : 1.f;
  }
  const float* rows = a.qkv + (size_t)tb * C;
  const float* decays = a.decay + ((size_t)tb * H + h) * D;  // PER_CHANNEL
  float v[RUN];  // the first column of values, under way from here
#pragma unroll
  for (int i = 0; i < RUN; ++i) v[i] = 0.f;
  auto fetch_values = [&](int c) {  // rows past the end are the last one's, and then nothing: no branch a token
#pragma unroll
    for (int i = 0; i < RUN; ++i) v[i] = rows[(unsigned)((i < n ? i : n - 1) * C + 2 * G * D + h * Dv + c)];
    if (n < RUN) {
#pragma unroll
      for (int i = 0; i < RUN; ++i) v[i] = i < n ? v[i] : 0.f;
    }
  };
  if (tid >= D && tid < D + Dv) fetch_values(tid - D);
  float k[RUN], q[RUN], g[RUN];
  if constexpr (!PER_CHANNEL) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < RUN; ++i) g[i] = gs[i];
    double p = 1.;
#pragma unroll
    for (int i = 0; i < RUN; ++i) {
      p *= (double)g[i];
      if (tid == 0) gp[i] = p;
    }
  }
  for (int d = tid; d < D; d += RUNS_THREADS) {
#pragma unroll
    for (int i = 0; i < RUN; ++i) {
      const int r = i < n ? i : n - 1;
      q[i] = rows[(unsigned)(r * C + kh * D + d)];
      k[i] = rows[(unsigned)(r * C + G * D + kh * D + d)];
      if constexpr (PER_CHANNEL) g[i] = decays[(unsigned)(r * H * D + d)];
    }
    if (n < RUN) {
#pragma unroll
      for (int i = 0; i < RUN; ++i) {
        q[i] = i < n ? q[i] : 0.f, k[i] = i < n ? k[i] : 0.f;
        if constexpr (PER_CHANNEL) g[i] = i < n ? g[i] : 1.f;
      }
    }
    double p = 1.;
    if constexpr (PER_CHANNEL) {
      double least = 1.;
#pragma unroll
      for (int i = 0; i < RUN; ++i) {
        p *= (double)g[i];
        least *= (double)g[i] < LEAST_DECAY ? LEAST_DECAY : (double)g[i];  // what is no number stays so
        kr[i * KS + d] = (double)k[i] * least;
        qr[i * KS + d] = (double)q[i] * least;
        kc[i * KS + d] = (double)k[i] / least;
      }
    } else {
#pragma unroll
      for (int i = 0; i < RUN; ++i) kr[i * KS + d] = k[i], qr[i * KS + d] = q[i], p *= (double)g[i];
    }
    oG[d] = (float)p;
    double after = 1.;  // the decays behind a token
    float back[RUN];
#pragma unroll
    for (int i = RUN - 1; i >= 0; --i) {
      back[i] = (float)((double)k[i] * after);
      after *= (double)g[i];
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
      *(f32x4*)(oK + (d / 16) * 256 + (j * 16 + row_token(d % 16)) * 4) = f32x4{back[j], back[4 + j], back[8 + j], back[12 + j]};
  }
  __syncthreads();
  {
    const int i = tid / RUN, j = tid % RUN;
    double sa[2] = {0., 0.}, sp[2] = {0., 0.};
    typedef KEY KEY4 __attribute__((ext_vector_type(4)));
    for (int d = 0; d < D; d += 4) {
      const KEY4 c = *(const KEY4*)(kc + j * KS + d), r = *(const KEY4*)(kr + i * KS + d), s = *(const KEY4*)(qr + i * KS + d);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        sa[e & 1] = fma((double)r[e], (double)c[e], sa[e & 1]);
        sp[e & 1] = fma((double)s[e], (double)c[e], sp[e & 1]);
      }
    }
    double ra = sa[0] + sa[1], rp = sp[0] + sp[1];
    if constexpr (!PER_CHANNEL) {
      double r = 1.;
#pragma unroll
      for (int l = 1; l < RUN; ++l) r *= l > j && l <= i ? (double)g[l] : 1.;
      ra *= r, rp *= r;
    }
    A[i * RUN + j] = (double)bs[i] * ra;
    oP[j / 4 * 64 + j % 4 * 16 + row_token(i)] = j < i ? (float)rp : 0.f;
    if (i == j) oP[RUN * RUN + i] = (float)rp;
  }
  __syncthreads();
  for (int c = tid; c < D + Dv; c += RUNS_THREADS) {
    double x[RUN];
    if (c < D) {
#pragma unroll
      for (int i = 0; i < RUN; ++i) x[i] = (double)bs[i] * (PER_CHANNEL ? 1. : gp[i]) * (double)kr[i * KS + c];
    } else {
      if (c >= RUNS_THREADS) fetch_values(c - D);
#pragma unroll
      for (int i = 0; i < RUN; ++i) x[i] = (double)bs[i] * (double)v[i];
    }
#pragma unroll
    for (int i = 1; i < RUN; ++i) {
      if (i % 2 == 1) asm volatile("" ::: "memory");  // A is read two rows at a time, not all of it into registers
#pragma unroll
      for (int l = 0; l < i; ++l) x[i] = fma(-A[i * RUN + l], x[l], x[i]);
    }
    if (c < D) {
#pragma unroll
      for (int i = 0; i < RUN; ++i) w[i * KS + c] = (float)x[i];
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        *(f32x4*)(oY + (c - D) / 16 * 256 + (j * 16 + (c - D) % 16) * 4) =
            f32x4{(float)x[j], (float)x[4 + j], (float)x[8 + j], (float)x[12 + j]};
    }
  }
  __syncthreads();
  const double gq = PER_CHANNEL ? 1. : gp[row_token(tid % 16)];
  for (int x = tid; x < 4 * D; x += RUNS_THREADS) {
    const int at = row_token(x % 16) * KS + 16 * (x / 64) + 4 * (x % 64 / 16);
    *(f32x4*)(oW + x * 4) = *(const f32x4*)(w + at);
    f32x4 s;
#pragma unroll
    for (int e = 0; e < 4; ++e) s[e] = (float)((double)qr[at + e] * gq);
    *(f32x4*)(oQ + x * 4) = s;
  }
}

// ROWS: tiles of 16 rows of S a wave keeps (D = 64 ROWS).  A run costs a wave 12 ROWS + 1 products: 2 x 4 ROWS for its
// share of W S0 and (G * Q) S0, 4 ROWS for the update, one for its quarter of P U; partial sums meet in LDS, one barrier
// a run (what a run leaves there, the run after the next overwrites).
template <int ROWS>
__global__ void __launch_bounds__(RUNS_THREADS, ROWS < 3 ? 2 : 1) delta_runs_kernel(RunsArgs a) {
  __shared__ f32x4 parts_u[2][4][WAVE], parts_o[2][4][WAVE];
  const int D = a.D, Dv = a.Dv, H = a.H;
  // The blocks of one sequence and head read the same W, G * Q and R_15 * K: blocks go round the XCDs, so with a multiple
  // of eight pairs between them they share one XCD's L2.
  const int pairs = a.n_seqs * H, stride = (pairs + 7) & ~7;
  const int pair = blockIdx.x % stride, ct = blockIdx.x / stride;
  if (pair >= pairs) return;
  const int b = pair / H, h = pair % H;
  int t0 = uniform_load(a.seq_starts + b), t1 = uniform_load(a.seq_starts + b + 1);
  if (t0 >= t1 || uniform_load(a.seq_of_token + t0) < 0) return;
  // the sequence's runs in this piece
  if (t0 >= a.p1) return;
  t1 = min(t1, t0 + (a.p1 - t0 + RUN - 1) / RUN * RUN);
  if (t0 < a.p0) t0 += (a.p0 - t0 + RUN - 1) / RUN * RUN;
  if (t0 >= t1) return;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, quad = lane >> 4;
  const int n_runs = (t1 - t0 + RUN - 1) / RUN;
  const size_t step = (size_t)H * run_floats(D, Dv);
  const float* run0 = a.runs + ((size_t)(t0 / RUN + b - a.p0 / RUN) * H + h) * run_floats(D, Dv);
  float* state = a.state + (((size_t)a.slot_ids[b] * H + h) * Dv + 16 * ct + col) * D + 16 * ROWS * wave + 4 * quad;

  f32x4 S[ROWS];
#pragma unroll
  for (int t = 0; t < ROWS; ++t) S[t] = *(const f32x4*)(state + 16 * t);

  struct Operands {
    f32x4 w[ROWS], q[ROWS], k[ROWS], g[ROWS], y;
    float p, diag;
  };
  const int frag = ROWS * wave * 256 + lane * 4;
  auto load_w = [&](Operands& x, const float* run) {
#pragma unroll
    for (int t = 0; t < ROWS; ++t) x.w[t] = *(const f32x4*)(run + frag + t * 256);
    x.y = *(const f32x4*)(run + 3 * RUN * D + ct * 256 + lane * 4);
  };
  auto load_q = [&](Operands& x, const float* run) {
#pragma unroll
    for (int t = 0; t < ROWS; ++t) x.q[t] = *(const f32x4*)(run + RUN * D + frag + t * 256);
    x.p = run[RUN * (3 * D + Dv) + wave * 64 + lane];
    x.diag = run[RUN * (3 * D + Dv + RUN) + 4 * wave + quad];
  };
  auto load_k = [&](Operands& x, const float* run) {
#pragma unroll
    for (int t = 0; t < ROWS; ++t) {
      x.k[t] = *(const f32x4*)(run + 2 * RUN * D + frag + t * 256);
      x.g[t] = *(const f32x4*)(run + RUN * (3 * D + Dv + RUN + 1) + 16 * (ROWS * wave + t) + 4 * quad);
    }
  };
  // What a run leaves goes out behind the next runs' work.  Run c - 1's share of its outputs, in `o`, gets its quarter of P U
  // behind run c's barrier and is written to LDS; run c + 1 adds the four waves' up, with what a token reads of its own write
  // (often the most of it), and rounds once.  A wave stores a quarter of the tokens.
  f32x4 o = {};
  float p1 = 0.f, mine1 = 0.f, diag1 = 0.f, mine2 = 0.f, diag2 = 0.f;  // of the last run and of the one before it
  int t2 = t0 + 4 * wave + quad - 2 * RUN;                             // the token this lane stores of the run before the last
  const size_t out_step = (size_t)RUN * H * Dv;
  float* out2 = a.out + (size_t)(t0 + 4 * wave + quad) * H * Dv + h * Dv + 16 * ct + col;  // and its place, once t2 >= t0
  auto add_written = [&]() {
    if (__any(!(fabsf(mine1) <= 3.4028235e38f))) {
      // A value that is no number must not reach the tokens before it through the zeros of P: token by token
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const float uj = __shfl(mine1, g * 16 + col, WAVE);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float pij = __shfl(p1, g * 16 + 4 * quad + e, WAVE);
          if (4 * wave + g < 4 * e + quad) o[e] = fmaf(pij, uj, o[e]);
        }
      }
    } else {
      o = __builtin_amdgcn_mfma_f32_16x16x4f32(p1, mine1, o, 0, 0, 0);
    }
  };
  auto leave = [&](const float (&part)[4]) {
    if (t2 >= t0) {
      const double sum = ((double)part[0] + (double)part[1]) + ((double)part[2] + (double)part[3]);
      if (t2 < t1) *out2 = (float)fma((double)diag2, (double)mine2, sum);
      out2 += out_step;
    }
    t2 += RUN;
  };
  auto work = [&](const Operands& x, Operands& next, const float* ahead, int c) {
    f32x4 u0 = {}, u1 = {}, o0 = {}, o1 = {};
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int t = 0; t < ROWS; ++t) {
        f32x4& u = t & 1 ? u1 : u0;
        u = __builtin_amdgcn_mfma_f32_16x16x4f32(x.w[t][e], S[t][e], u, 0, 0, 0);
      }
    load_w(next, ahead);
    __builtin_amdgcn_sched_barrier(0);
    parts_u[c & 1][wave][lane] = u0 + u1;
    f64x4 s[ROWS], k[ROWS];
#pragma unroll
    for (int t = 0; t < ROWS; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) s[t][e] = (double)x.g[t][e] * (double)S[t][e], k[t][e] = (double)x.k[t][e];
    block_sync_lds();
    const f32x4 s0 = parts_u[c & 1][0][lane], s1 = parts_u[c & 1][1][lane], s2 = parts_u[c & 1][2][lane], s3 = parts_u[c & 1][3][lane];
    float part[4];
#pragma unroll
    for (int p = 0; p < 4; ++p) part[p] = ((const float*)&parts_o[c & 1][p][lane])[wave];
    __builtin_amdgcn_sched_barrier(0);
    add_written();
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int t = 0; t < ROWS; ++t) {
        f32x4& o = t & 1 ? o1 : o0;
        o = __builtin_amdgcn_mfma_f32_16x16x4f32(x.q[t][e], S[t][e], o, 0, 0, 0);
      }
    load_q(next, ahead);
    const f32x4 ws = (s0 + s1) + (s2 + s3);
    double u[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) u[e] = (double)x.y[e] - (double)ws[e];
    __builtin_amdgcn_sched_barrier(0);
    // the update in 64 bits, from S as the decays leave it: S is rounded once a run
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int t = 0; t < ROWS; ++t) s[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(k[t][e], u[e], s[t], 0, 0, 0);
    load_k(next, ahead);
    parts_o[(c + 1) & 1][wave][lane] = o;
    leave(part);
    mine2 = mine1, diag2 = diag1;
    p1 = x.p, diag1 = x.diag;
    mine1 = (float)(wave == 0 ? u[0] : wave == 1 ? u[1] : wave == 2 ? u[2] : u[3]);
    o = o0 + o1;
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < ROWS; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) S[t][e] = (float)s[t][e];
  };
  Operands x0, x1, x2;
  const float *ahead = run0, *last = run0 + (size_t)(n_runs - 1) * step;
  auto advance = [&]() { ahead = ahead == last ? last : ahead + step; };  // no branch around loads that later runs wait for
  load_w(x0, ahead), load_q(x0, ahead), load_k(x0, ahead);
  advance();
  load_w(x1, ahead), load_q(x1, ahead), load_k(x1, ahead);
  for (int c = 0;;) {
    advance();
    work(x0, x2, ahead, c);
    if (++c == n_runs) break;
    advance();
    work(x1, x0, ahead, c);
    if (++c == n_runs) break;
    advance();
    work(x2, x1, ahead, c);
    if (++c == n_runs) break;
  }
  // the last two runs' outputs
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    float part[4];
    block_sync_lds();
#pragma unroll
    for (int p = 0; p < 4; ++p) part[p] = ((const float*)&parts_o[(n_runs + c) & 1][p][lane])[wave];
    leave(part);
    if (c == 0) {
      add_written();
      parts_o[(n_runs + 1) & 1][wave][lane] = o;
      mine2 = mine1, diag2 = diag1;
    }
  }
#pragma unroll
  for (int t = 0; t < ROWS; ++t) *(f32x4*)(state + 16 * t) = S[t];
}

// --------------------------------------------------------------------------
// The places of the whole step, or as many as RUNS_WORKSPACE holds, and then at least two a sequence and 64 (a sequence's state is
// as large as two): a piece is 1000 tokens or more.
extern "C" long fmsamd_delta_runs_workspace(int n_tokens, int n_seqs, int heads, int dim, int vdim) {
  if (n_tokens < 0 || n_seqs < 0 || heads <= 0 || dim <= 0 || vdim <= 0 || dim % 64 || dim > 256 || vdim % 16) return -1;
  const long place = heads * (long)run_floats(dim, vdim) * (long)sizeof(float), all = n_tokens / RUN + (long)n_seqs;
  const long bound = RUNS_WORKSPACE / place > 2L * n_seqs + 64 ? RUNS_WORKSPACE / place : 2L * n_seqs + 64;
  return (all < bound ? all : bound) * place;
}

extern "C" int fmsamd_delta_runs(const float* qkv, const float* beta, const float* decay, float* state, float* out, const int* seq_starts,
                                 const int* seq_of_token, const int* slot_ids, int n_tokens, int n_seqs, int heads, int kv_heads, int dim,
                                 int vdim, int per_channel, void* workspace, long workspace_bytes, hipStream_t stream) {
  if (n_seqs == 0 || n_tokens == 0) return 0;
  FMS_REQUIRE(n_seqs > 0 && n_tokens > 0 && heads > 0 && kv_heads > 0 && heads % kv_heads == 0 && dim > 0 && vdim > 0,
              "delta_runs: bad sizes heads=%d kv_heads=%d dim=%d vdim=%d", heads, kv_heads, dim, vdim);
  FMS_REQUIRE(dim % 64 == 0 && dim <= 256 && vdim % 16 == 0, "delta_runs: %d key and %d value channels (multiples of 64 up to 256, and of 16)",
              dim, vdim);
  FMS_REQUIRE(n_tokens <= 0x7fffffff - 4 * RUN, "delta_runs: too many tokens");
  const long room = workspace_bytes / (heads * (long)run_floats(dim, vdim) * (long)sizeof(float)), all = n_tokens / RUN + (long)n_seqs;
  const long blocks = (((long)n_seqs * heads + 7) & ~7L) * (vdim / 16);
  FMS_REQUIRE(heads <= 65535 && blocks <= 0x7fffffffL && all <= 0x7fffffffL, "delta_runs: too many heads or value channels for one launch");
  FMS_REQUIRE(room >= all || room > n_seqs, "delta_runs: the workspace is too small");
  FMS_REQUIRE(((uintptr_t)state | (uintptr_t)workspace) % 16 == 0, "delta_runs: the state and the workspace start at 16-byte addresses");
  RunsArgs a{qkv, beta, decay, state, out, (float*)workspace, seq_starts, seq_of_token, slot_ids, n_seqs, heads, kv_heads, dim, vdim, 0, 0};
  const size_t lds = (size_t)(RUN * RUN + RUN) * sizeof(double) + 2 * RUN * sizeof(float) +
                     (size_t)RUN * (dim + 4) * 3 * (per_channel ? sizeof(double) : sizeof(float));
  if (lds > 64 * 1024) {  // a decay per key channel from 192 channels on: more has to be asked for, once a kernel
    static const hipError_t sized = hipFuncSetAttribute(reinterpret_cast<const void*>(delta_runs_prepare_kernel<true>),
                                                        hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    FMS_REQUIRE(sized == hipSuccess && per_channel && lds <= 160 * 1024, "delta_runs: %zu bytes of LDS refused: %s", lds, hipGetErrorString(sized));
  }
  const int end = (n_tokens + RUN - 1) / RUN * RUN;
  const long piece = room >= all ? end : (room - n_seqs) * RUN;  // tokens of a piece
  for (long p0 = 0; p0 < end; p0 += piece) {
    a.p0 = (int)p0, a.p1 = (int)(p0 + piece < end ? p0 + piece : end);
    const dim3 grid((unsigned)(room >= all ? all : (a.p1 - a.p0) / RUN + n_seqs), heads);
    if (per_channel) delta_runs_prepare_kernel<true><<<grid, RUNS_THREADS, lds, stream>>>(a);
    else delta_runs_prepare_kernel<false><<<grid, RUNS_THREADS, lds, stream>>>(a);
    FMS_LAUNCH_CHECK("delta_runs_prepare");
    if (dim == 64) delta_runs_kernel<1><<<blocks, RUNS_THREADS, 0, stream>>>(a);
    else if (dim == 128) delta_runs_kernel<2><<<blocks, RUNS_THREADS, 0, stream>>>(a);
    else if (dim == 192) delta_runs_kernel<3><<<blocks, RUNS_THREADS, 0, stream>>>(a);
    else delta_runs_kernel<4><<<blocks, RUNS_THREADS, 0, stream>>>(a);
    FMS_LAUNCH_CHECK("delta_runs");
  }
  return 0;
}
