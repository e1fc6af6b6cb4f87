// Temperature / top-k sampling of the next token on the device: sample_from_logits_values and the
// temperature division of sample_next_token (src/generation.rs:26-72, :117).  One wavefront (V <= 1024) or
// workgroup per sequence; the uniform variate comes from the caller, so the token never visits the host.
#include "bdh_internal.h"

namespace {

constexpr int SAMPLE_THREADS = 256;
constexpr int SAMPLE_MAX_V = 8192;
constexpr int SAMPLE_WAVE_V = 1024;  // up to here one wavefront keeps the whole row in its registers

// Monotone map float -> uint32 (larger float = larger key), so the k-th largest value can be found
// by a bitwise search over keys.  The two zeros are one value, as the comparison of :41-45 has them.
__device__ __forceinline__ uint32_t order_key(float f) {
  const uint32_t u = __float_as_uint(f + 0.0f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// The running sums of :57-67 and of WeightedIndex go in index order.  An entry that is exactly zero (everything below the
// k-th largest value is) changes none of them, so they run over the list of the others: sum, the probabilities v / sum,
// their sum, and the first entry whose cumulative weight exceeds the variate.  w [n] (overwritten) and at [n] are the
// list's values and their indices, ascending.  Called by one wavefront; every lane returns the chosen index.
template <typename I>
__device__ __forceinline__ int weighted_index(float *w, const I *at, int n, int V, float u) {
  const int lane = threadIdx.x & 63;
  // a chain over the list: 64 entries sit in the lanes' registers (zeros past the end, which change no sum) and are handed
  // on by readlane, eight per turn from lanes that the instruction names, so the chain waits for one addition per entry,
  // not for a lane's number, a branch or memory
  auto chain = [&](float start, float v, int lo) {
    float s = start;
#pragma unroll
    for (int j = 0; j < 64; j += 8) {
      if (lo + j >= n) break;  // uniform
#pragma unroll
      for (int e = 0; e < 8; ++e) s += __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(v), j + e));
    }
    return s;
  };
  float sum = 0.f;
  for (int lo = 0; lo < n; lo += 64) sum = chain(sum, lo + lane < n ? w[lo + lane] : 0.f, lo);
  const bool flat = (sum == 0.f) || (sum != sum);
  u = fminf(fmaxf(u, 0.f), 0.99999994f);
  if (flat) {  // the uniform distribution over all V entries
    const float p = 1.0f / (float)V;
    float total = 0.f;
    for (int i = 0; i < V; ++i) total += p;
    const float chosen = u * total;
    float cum = 0.f;
    int idx = 0;
    for (int i = 0; i < V - 1; ++i) {
      cum += p;
      if (cum <= chosen) idx = i + 1;
      else break;
    }
    return idx;
  }
  float total = 0.f;
  for (int lo = 0; lo < n; lo += 64) {
    const float p = lo + lane < n ? w[lo + lane] / sum : 0.f;
    if (lo + lane < n) w[lo + lane] = p;
    total = chain(total, p, lo);
  }
  // WeightedIndex: the variate is uniform in [0, total); the index is the number of cumulative weights (of the first
  // V - 1 entries) <= the variate, i.e. the first listed entry whose cumulative weight exceeds it
  const float chosen = u * total;
  float cum = 0.f;
  for (int lo = 0; lo < n; lo += 64) {
    const float p = lo + lane < n ? w[lo + lane] : 0.f;
#pragma unroll
    for (int j = 0; j < 64; j += 8) {
      if (lo + j >= n) break;  // uniform
      int below = 0;  // the cumulative weights never fall, so those up to the variate come first
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        cum += __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(p), j + e));
        below += cum > chosen ? 0 : 1;
      }
      if (below < 8) return lo + j + below < n ? min((int)at[lo + j + below], V - 1) : V - 1;
    }
  }
  return V - 1;
}

// V <= R * 64: one wavefront per sequence, R values per lane, no barrier.  The k-th largest key is found a bit at a time
// from ballots of register compares, the survivors are listed with ballot prefix counts, and the index-order sums run
// over that list only.  Bound by the length of these chains, not by memory (V = 256, k = 40: 43 us for a workgroup
// with the row in LDS, which paid two barriers per bit and three V-long chains of LDS reads in one lane; 6.9 us with all 32
// bits looked at and a turn of the chains per entry, 4.5 here).
template <int R>
__global__ __launch_bounds__(64) void k_sample_wave(const float *__restrict__ logits, long ld, int V, float temperature,
                                                    int top_k, const float *__restrict__ uniforms,
                                                    int64_t *__restrict__ next_tokens) {
  __shared__ float s_w[R * 64];
  __shared__ int s_at[R * 64];
  const int b = blockIdx.x, lane = threadIdx.x;
  const float *row = logits + (long)b * ld;
  float v[R];
  float m = -INFINITY;
#pragma unroll
  for (int r = 0; r < R; ++r) v[r] = r * 64 + lane < V ? row[r * 64 + lane] : 0.f;
#pragma unroll
  for (int r = 0; r < R; ++r) v[r] = r * 64 + lane < V ? v[r] / temperature : -INFINITY;  // :117 div_scalar
  const float u = uniforms[b];
  uint32_t thr = 0;
  if (top_k > 0 && top_k < V) {  // :35-47 — everything below the k-th largest value becomes -inf
    uint32_t key[R];
#pragma unroll
    for (int r = 0; r < R; ++r) key[r] = r * 64 + lane < V ? order_key(v[r]) : 0u;
    for (int bit = 31; bit >= 0; --bit) {
      const uint32_t cand = thr | (1u << bit);
      int c = 0;
#pragma unroll
      for (int r = 0; r < R; ++r) c += __popcll(__ballot(key[r] >= cand));
      if (c >= top_k) thr = cand;
      if (c == top_k) break;  // no key between cand and the k-th largest: the same entries survive
    }
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (key[r] < thr) v[r] = -INFINITY;
  }
#pragma unroll
  for (int r = 0; r < R; ++r) m = fmaxf(m, v[r]);  // :49-52 (f32::max ignores NaN operands, as fmaxf does)
  for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off, 64));
  int n = 0;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const float e = r * 64 + lane < V ? expf(v[r] - m) : 0.f;  // :53-56
    const unsigned long long mask = __ballot(e != 0.f);        // a NaN counts: it makes the sum NaN
    if (e != 0.f) {
      const int at = n + __popcll(mask & ((1ull << lane) - 1));
      s_w[at] = e;
      s_at[at] = r * 64 + lane;
    }
    n += __popcll(mask);
  }
  __syncthreads();
  const int idx = weighted_index(s_w, s_at, n, V, u);
  if (lane == 0) next_tokens[b] = idx;
}

// V up to 8192: a workgroup per sequence, the row in LDS
__global__ __launch_bounds__(SAMPLE_THREADS) void k_sample_top_k(const float *__restrict__ logits, long ld, int V,
                                                                 float temperature, int top_k,
                                                                 const float *__restrict__ uniforms,
                                                                 int64_t *__restrict__ next_tokens) {
  constexpr int NW = SAMPLE_THREADS / 64;
  __shared__ float s_val[SAMPLE_MAX_V];
  __shared__ unsigned short s_at[SAMPLE_MAX_V];
  __shared__ int s_red[2][NW];
  __shared__ float s_redf[NW];
  const int b = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const float *row = logits + (long)b * ld;
  for (int i = tid; i < V; i += SAMPLE_THREADS) s_val[i] = row[i] / temperature;  // :117 div_scalar
  __syncthreads();

  if (top_k > 0 && top_k < V) {  // :35-47 — everything below the k-th largest value becomes -inf
    uint32_t thr = 0;
    for (int bit = 31; bit >= 0; --bit) {
      const uint32_t cand = thr | (1u << bit);
      int c = 0;
      for (int i = tid; i < V; i += SAMPLE_THREADS) c += order_key(s_val[i]) >= cand;
      for (int off = 32; off > 0; off >>= 1) c += __shfl_xor(c, off, 64);
      if (lane == 0) s_red[bit & 1][wave] = c;  // two buffers in turn: one barrier per bit
      __syncthreads();
      int total = 0;
#pragma unroll
      for (int w = 0; w < NW; ++w) total += s_red[bit & 1][w];
      if (total >= top_k) thr = cand;  // uniform across the workgroup
    }
    for (int i = tid; i < V; i += SAMPLE_THREADS)
      if (order_key(s_val[i]) < thr) s_val[i] = -INFINITY;
    __syncthreads();
  }

  float m = -INFINITY;  // :49-52 (f32::max ignores NaN operands, as fmaxf does)
  for (int i = tid; i < V; i += SAMPLE_THREADS) m = fmaxf(m, s_val[i]);
  for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off, 64));
  if (lane == 0) s_redf[wave] = m;
  __syncthreads();
  m = s_redf[0];
#pragma unroll
  for (int w = 1; w < NW; ++w) m = fmaxf(m, s_redf[w]);
  for (int i = tid; i < V; i += SAMPLE_THREADS) s_val[i] = expf(s_val[i] - m);  // :53-56
  __syncthreads();

  if (wave != 0) return;
  int n = 0;
  for (int i0 = 0; i0 < V; i0 += 64) {  // the non-zero entries to the front, in order (never past the place read last)
    const float e = i0 + lane < V ? s_val[i0 + lane] : 0.f;
    const unsigned long long mask = __ballot(e != 0.f);
    if (e != 0.f) {
      const int at = n + __popcll(mask & ((1ull << lane) - 1));
      s_val[at] = e;
      s_at[at] = (unsigned short)(i0 + lane);
    }
    n += __popcll(mask);
  }
  const int idx = weighted_index(s_val, s_at, n, V, uniforms[b]);
  if (lane == 0) next_tokens[b] = idx;
}

}  // namespace

extern "C" int bdh_sample_top_k(bdh_ctx *ctx, int B, int V, const float *logits, int64_t row_stride,
                                float temperature, int top_k, const float *uniforms, int64_t *next_tokens) {
  if (!ctx) return BDH_E_INVAL;
  if (B < 0 || V < 1) return bdh_fail(ctx, BDH_E_INVAL, "bad batch %d or vocabulary %d", B, V);
  if (V > SAMPLE_MAX_V) return bdh_fail(ctx, BDH_E_SHAPE, "vocabulary %d > %d", V, SAMPLE_MAX_V);
  if (row_stride < V) return bdh_fail(ctx, BDH_E_INVAL, "row stride %lld < vocabulary %d", (long long)row_stride, V);
  if (B == 0) return BDH_OK;
  if (!logits || !uniforms || !next_tokens) return bdh_fail(ctx, BDH_E_INVAL, "null data pointer");
  const long ld = (long)row_stride;
  // one wavefront per sequence while its registers hold the row
  if (V <= 256)
    hipLaunchKernelGGL((k_sample_wave<4>), dim3(B), dim3(64), 0, ctx->stream, logits, ld, V, temperature, top_k, uniforms, next_tokens);
  else if (V <= SAMPLE_WAVE_V)
    hipLaunchKernelGGL((k_sample_wave<SAMPLE_WAVE_V / 64>), dim3(B), dim3(64), 0, ctx->stream, logits, ld, V, temperature,
                       top_k, uniforms, next_tokens);
  else
    hipLaunchKernelGGL(k_sample_top_k, dim3(B), dim3(SAMPLE_THREADS), 0, ctx->stream, logits, ld, V, temperature, top_k,
                       uniforms, next_tokens);
  BDH_LAUNCH_CHECK(ctx, "k_sample_top_k");
  return BDH_OK;
}
