// Attention in float32 on the matrix unit's float32 products (16x16x4): a block per 16 query rows of a head and sequence, whose
// four waves take tiles of 32 keys in turn and meet in LDS.  S^T = K Q^T leaves keys 4 (lane / 16) + r
// of a lane's query in register r, which is the operand layout of O^T = V^T P for a product that takes these four keys as its
// four: nothing goes through LDS, and a lane's keys and values are 16 consecutive bytes (the steps of K are dealt the same way).
//
// A query's result has the same bits whatever rows stand beside it, in a prompt, a portion or a decode step: keys are cut at
// absolute places, and a tile that it does not see changes nothing.  So single tokens run here too, with one row of 16 in use:
// the products they waste hide behind the keys and values.
//
// Bound by what a compute unit takes in: a head's keys and values once for every 16 queries.  Microseconds, in brackets with a
// block of FMAs per token and head: 301 tokens of 32 heads of 128 25 (175), 1000 tokens 151 (1752); one token behind 8, 64, 300,
// 1000 and 4000 tokens 6.6, 6.8, 16, 41 and 161 (4.8, 6.5, 16, 47, 193); 64 single tokens behind 1000 each 388 (504).  (A branch
// that leaves out a tile's second half where it has no key is 0.6 us faster for contexts up to 16 and a quarter slower beyond.)
// 15 single tokens behind 2000 and a prompt of 64 197 (212), where a block that takes the sequences of its rows one after the other
// needs a chain of 16 contexts.  The scores are sums of four
// accumulators and the results of four waves: errors against 64 bits of 1.35e-7 and 2.6e-7 (301 tokens).
#include "common.h"
#include "fmsamd.h"

#define F32_ATTN_EMPTY -1e30f

struct AttnF32Args {
  const float* q;
  long q_stride;
  float* out;
  long out_stride;
  const int *positions, *seq_of_token, *block_table;
  int table_stride;
  const float *k_cache, *v_cache;
  int n_tokens, nheads, kvheads, window;
  float scale;
};

// NT: tiles of 16 elements of a head
template <int NT>
__global__ void __launch_bounds__(256, 2) attn_f32_kernel(AttnF32Args a) {
  constexpr int D = NT * 16, ROW = D + 4;
  __shared__ __attribute__((aligned(16))) float meet[4][16][ROW];
  __shared__ bool theirs[16];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, quad = lane >> 4;
  const int h = blockIdx.x, kh = h / (a.nheads / a.kvheads);
  const int t0 = (gridDim.y - 1 - blockIdx.y) * 16;  // the longest contexts of a prompt first
  const int n_rows = a.n_tokens - t0 < 16 ? a.n_tokens - t0 : 16;
  const bool there = col < n_rows;
  const int t = t0 + (there ? col : 0);
  const int seq = there ? a.seq_of_token[t] : -1;
  // The block's sequence: the blockIdx.z-th of those of the 16 rows (rows without one go with the first block).  Contexts of
  // several sequences side by side, not one behind the other; a block too many leaves after one round trip.
  unsigned long long left = __ballot(seq >= 0 && lane < 16);
  if (blockIdx.z > 0) {
    for (int z = 0; z < (int)blockIdx.z && left != 0; ++z)
      left &= ~__ballot(seq == __builtin_amdgcn_readlane(seq, __builtin_ctzll(left)));
    if (left == 0) return;
  }
  const int turn = left != 0 ? __builtin_amdgcn_readlane(seq, __builtin_ctzll(left)) : 0;
  const bool writes = there && (seq == turn || (seq < 0 && blockIdx.z == 0));
  const int pos = seq >= 0 ? a.positions[t] : -1;
  const int lo = a.window > 0 && pos - a.window + 1 > 0 ? pos - a.window + 1 : 0;

  f32x4 q[NT];
#pragma unroll
  for (int c = 0; c < NT; ++c) q[c] = *(const f32x4*)(a.q + (size_t)t * a.q_stride + (size_t)h * D + 16 * c + 4 * quad);
  f32x4 acc[NT];
#pragma unroll
  for (int d = 0; d < NT; ++d) acc[d] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = F32_ATTN_EMPTY, l = 0.f;

  // of the rows whose sequence is `turn`, the keys from the first to the last that any sees
  if (left != 0) {
    const bool mine = seq == turn;
    int last = mine ? pos : -1, first = mine ? lo : 0x7fffffff;
    int all_lo = mine ? lo : 0, all_pos = mine ? pos : -1;  // what every column sees (nothing, beside a row of another sequence)
#pragma unroll
    for (int off = 1; off < 16; off <<= 1) {
      last = max(last, __shfl_xor(last, off, WAVE)), first = min(first, __shfl_xor(first, off, WAVE));
      all_lo = max(all_lo, __shfl_xor(all_lo, off, WAVE)), all_pos = min(all_pos, __shfl_xor(all_pos, off, WAVE));
    }
    last = __builtin_amdgcn_readfirstlane(last), first = __builtin_amdgcn_readfirstlane(first);
    all_lo = __builtin_amdgcn_readfirstlane(all_lo), all_pos = __builtin_amdgcn_readfirstlane(all_pos);
    const int* bt = a.block_table + (size_t)turn * a.table_stride;
    const size_t page_elems = (size_t)a.kvheads * PAGE_TOKENS * D;
    // tile u goes to wave u % 4, by its place in the sequence
    for (int u = first / 32 + ((wave - first / 32) & 3); u * 32 <= last; u += 4) {
      const int base = u * 32;
      const size_t page = readable_page(uniform_load(bt + base / PAGE_TOKENS));
      const float* kp = a.k_cache + page * page_elems + ((size_t)kh * PAGE_TOKENS + base % PAGE_TOKENS + col) * D + 4 * quad;
      const float* vp = a.v_cache + page * page_elems + ((size_t)kh * D + col) * PAGE_TOKENS + base % PAGE_TOKENS + 4 * quad;
      f32x4 v[2][NT];  // under way while the scores are multiplied
#pragma unroll
      for (int k = 0; k < 2; ++k)
#pragma unroll
        for (int d = 0; d < NT; ++d) v[k][d] = *(const f32x4*)(vp + (size_t)d * 16 * PAGE_TOKENS + 16 * k);
      f32x4 s[2];
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        f32x4 part[4] = {};
#pragma unroll
        for (int c = 0; c < NT; ++c) {
          const f32x4 key = *(const f32x4*)(kp + k * 16 * D + 16 * c);
#pragma unroll
          for (int e = 0; e < 4; ++e) part[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(key[e], q[c][e], part[e], 0, 0, 0);
        }
        s[k] = ((part[0] + part[1]) + (part[2] + part[3])) * a.scale;
      }
      const bool full = base >= all_lo && base + 31 <= all_pos;
      float top = -INFINITY;
#pragma unroll
      for (int k = 0; k < 2; ++k)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int j = base + 16 * k + 4 * quad + r;
          if (!full) s[k][r] = mine && j >= lo && j <= pos ? s[k][r] : -INFINITY;
          top = fmaxf(top, s[k][r]);
        }
      top = fmaxf(top, __shfl_xor(top, 16, WAVE));
      top = fmaxf(top, __shfl_xor(top, 32, WAVE));
      const float m_new = fmaxf(m, top), alpha = expf(m - m_new);
      m = m_new;
      f32x4 p[2];
      float psum = 0.f;
#pragma unroll
      for (int k = 0; k < 2; ++k)
#pragma unroll
        for (int r = 0; r < 4; ++r) p[k][r] = expf(s[k][r] - m_new), psum += p[k][r];
      l = l * alpha + psum;
      if (__any(alpha != 1.f)) {
#pragma unroll
        for (int d = 0; d < NT; ++d) acc[d] *= alpha;
      }
      float broken = 0.f;  // a value that some column must not see, and that its weight of zero would not hide: no number then
      if (!full) {
#pragma unroll
        for (int k = 0; k < 2; ++k)
#pragma unroll
          for (int d = 0; d < NT; ++d)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const int j = base + 16 * k + 4 * quad + r;
              if (j < first || j > last) v[k][d][r] = 0.f;  // nobody's
              broken = fmaf(v[k][d][r], 0.f, broken);
            }
      }
      if (__any(broken != 0.f)) {
        for (int i = 0; i < 32; ++i) {
          const int j = base + i;
          float pj = 0.f;
#pragma unroll
          for (int k = 0; k < 2; ++k)
#pragma unroll
            for (int r = 0; r < 4; ++r)
              if (i / 16 == k && i % 4 == r) pj = __shfl(p[k][r], i % 16 / 4 * 16 + col, WAVE);
          if (!(mine && j >= lo && j <= pos)) continue;
          const float* vj = a.v_cache + page * page_elems + ((size_t)kh * D + 4 * quad) * PAGE_TOKENS + j % PAGE_TOKENS;
#pragma unroll
          for (int d = 0; d < NT; ++d)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[d][r] = fmaf(pj, vj[(16 * d + r) * PAGE_TOKENS], acc[d][r]);
        }
      } else {
#pragma unroll
        for (int k = 0; k < 2; ++k)
#pragma unroll
          for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int d = 0; d < NT; ++d) acc[d] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[k][d][r], p[k][r], acc[d], 0, 0, 0);
      }
    }
  }

  l += __shfl_xor(l, 16, WAVE);
  l += __shfl_xor(l, 32, WAVE);
#pragma unroll
  for (int d = 0; d < NT; ++d) *(f32x4*)&meet[wave][col][16 * d + 4 * quad] = acc[d];
  if (quad == 0) meet[wave][col][D] = m, meet[wave][col][D + 1] = l;
  if (wave == 0 && quad == 0) theirs[col] = writes;
  __syncthreads();
  for (int x = threadIdx.x; x < n_rows * (D / 4); x += 256) {
    const int c = x / (D / 4), d = x % (D / 4) * 4;
    if (!theirs[c]) continue;
    float top = F32_ATTN_EMPTY, sum = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) top = fmaxf(top, meet[w][c][D]);
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float f = expf(meet[w][c][D] - top);
      sum = fmaf(meet[w][c][D + 1], f, sum);
      o += *(const f32x4*)&meet[w][c][d] * f;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = sum > 0.f ? o[e] / sum : 0.f;
    *(f32x4*)(a.out + (size_t)(t0 + c) * a.out_stride + (size_t)h * D + d) = o;
  }
}

extern "C" int fmsamd_attn_f32(const float* q, long q_stride, float* out, long out_stride, const int* positions, const int* seq_of_token,
                               const int* block_table, int table_stride, const float* k_cache, const float* v_cache, int n_tokens,
                               int n_seqs, int nheads, int kvheads, int head_dim, float scale, int window, hipStream_t stream) {
  if (n_tokens == 0) return 0;
  FMS_REQUIRE(n_tokens > 0 && n_seqs >= 0 && nheads > 0 && kvheads > 0 && nheads % kvheads == 0 && window >= 0, "attn_f32: bad sizes");
  FMS_REQUIRE(head_dim > 0 && head_dim % 16 == 0 && head_dim <= 128, "attn_f32: head size %d is no multiple of 16 up to 128", head_dim);
  FMS_REQUIRE(q_stride >= (long)nheads * head_dim && out_stride >= (long)nheads * head_dim && q_stride % 4 == 0 && out_stride % 4 == 0,
              "attn_f32: rows too short or not of whole 16 bytes");
  FMS_REQUIRE((((uintptr_t)q | (uintptr_t)out | (uintptr_t)k_cache | (uintptr_t)v_cache) & 15) == 0, "attn_f32: addresses of 16 bytes");
  FMS_REQUIRE(ceil_div(n_tokens, 16) <= 65535, "attn_f32: %d tokens exceed one launch", n_tokens);
  AttnF32Args a{q, q_stride, out, out_stride, positions, seq_of_token, block_table, table_stride, k_cache, v_cache,
                n_tokens, nheads, kvheads, window, scale};
  const dim3 grid(nheads, ceil_div(n_tokens, 16), n_seqs < 1 ? 1 : n_seqs < 16 ? n_seqs : 16);
  switch (head_dim / 16) {
#define FMS_AF(NT) case NT: attn_f32_kernel<NT><<<grid, 256, 0, stream>>>(a); break
    FMS_AF(1); FMS_AF(2); FMS_AF(3); FMS_AF(4); FMS_AF(5); FMS_AF(6); FMS_AF(7); FMS_AF(8);
#undef FMS_AF
  }
  FMS_LAUNCH_CHECK("attn_f32");
  return 0;
}
