// Dense stages around the state step: ReLU low-rank projections (D_x, D_y), LayerNorm,
// embedding gather, the decoder E with the residual LayerNorms, and lm_head.
// Reference semantics: src/kernel/relu_lowrank.rs:7-37, src/model/bdh.rs:86-89, :319-322,
// :346-350, :370-384, :436-449.
#include "bdh_internal.h"
#include "lds_copy.h"

#include <algorithm>
#include <atomic>
#include <type_traits>

namespace {

constexpr float kLnEps = 1e-5f;  // src/model/bdh.rs:17

// Sum of `v` over a 256-thread workgroup; every thread gets the result.
__device__ __forceinline__ float block_sum_256(float v, float *s_part) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  __syncthreads();  // protects s_part against the previous use
  if ((threadIdx.x & 63) == 0) s_part[threadIdx.x >> 6] = v;
  __syncthreads();
  return s_part[0] + s_part[1] + s_part[2] + s_part[3];
}

// ------------------------------------------------------------------------------------
// relu_lowrank: out[b,hh,t,n] = relu(sum_k in[b,hh|0,t,k] w[hh,k,n] + bias - thr) * mask
// One thread per latent column n (coalesced weight rows), RT input rows per workgroup
// staged in LDS, one k-sequential fmaf chain per output.
// ------------------------------------------------------------------------------------
template <int RT, int UK, int NTHR>
__global__ __launch_bounds__(NTHR) void k_relu_lowrank(const float *__restrict__ in, int h_in, int T, int d,
                                                      const float *__restrict__ w, int h, int N,
                                                      const float *__restrict__ bias, float thr,
                                                      const unsigned char *__restrict__ block_active,
                                                      int block_size, int n_blocks,
                                                      const float *__restrict__ gate, float *__restrict__ out,
                                                      int M) {
  extern __shared__ float s_in[];  // [RT][d]
  const int tid = threadIdx.x;
  const int hh = blockIdx.y;
  const int n = blockIdx.x * NTHR + tid;
  const int m0 = blockIdx.z * RT;
  for (int i = tid; i < RT * d; i += NTHR) {
    const int r = i / d, k = i - r * d;
    const int m = m0 + r;
    float val = 0.0f;
    if (m < M) {
      const int b = m / T, t = m - b * T;
      val = in[(((long)b * h_in + (h_in == 1 ? 0 : hh)) * T + t) * d + k];
    }
    s_in[i] = val;
  }
  __syncthreads();
  if (n >= N) return;

  float acc[RT];
#pragma unroll
  for (int r = 0; r < RT; ++r) acc[r] = 0.0f;
  const float *wp = w + (long)hh * d * N + n;
  int k0 = 0;
  for (; k0 + UK <= d; k0 += UK) {
    float wv[UK];
#pragma unroll
    for (int u = 0; u < UK; ++u) wv[u] = wp[(long)(k0 + u) * N];
#pragma unroll
    for (int u = 0; u < UK; ++u)
#pragma unroll
      for (int r = 0; r < RT; ++r) acc[r] = __builtin_fmaf(s_in[r * d + k0 + u], wv[u], acc[r]);
  }
  if (UK > 16) {  // what a large batch leaves over, 16 rows at a time
    for (; k0 + 16 <= d; k0 += 16) {
      float wv[16];
#pragma unroll
      for (int u = 0; u < 16; ++u) wv[u] = wp[(long)(k0 + u) * N];
#pragma unroll
      for (int u = 0; u < 16; ++u)
#pragma unroll
        for (int r = 0; r < RT; ++r) acc[r] = __builtin_fmaf(s_in[r * d + k0 + u], wv[u], acc[r]);
    }
  }
  for (; k0 < d; ++k0) {
    const float wv = wp[(long)k0 * N];
#pragma unroll
    for (int r = 0; r < RT; ++r) acc[r] = __builtin_fmaf(s_in[r * d + k0], wv, acc[r]);
  }

  const float bv = bias ? bias[(long)hh * N + n] : 0.0f;
  float maskv = 1.0f;
  if (block_active) {
    const int blk = n / block_size;
    maskv = (blk < n_blocks && block_active[blk]) ? 1.0f : 0.0f;
  }
#pragma unroll
  for (int r = 0; r < RT; ++r) {
    const int m = m0 + r;
    if (m < M) {
      const int b = m / T, t = m - b * T;
      float p = acc[r];
      if (bias) p = p + bv;
      if (thr != 0.0f) p = p - thr;
      float y = p > 0.0f ? p : 0.0f;
      if (block_active) y = y * maskv;
      const long o = (((long)b * h + hh) * T + t) * N + n;
      if (gate) y = gate[o] * y;
      out[o] = y;
    }
  }
}

// One input row per head that the kernel makes itself (a decode step of one sequence).  The reductions of a layer whose
// inputs come from other CUs -- the sum of the state step's readout partials with its LayerNorm (src/model/bdh.rs:359),
// the sum of the encoder's partials with the two LayerNorms and the residual (:436-441) -- run in front of the
// projection that consumes their result, in every workgroup, in front of the workgroup's weight loads: as launches
// of their own each is a launch gap plus a chain of dependent trips to memory.
//   MODE 1: row(hh) = LN(sum_g partial[hh][g][:])                      rows = S partial rows per head
//   MODE 2: row     = LN(cur_old + LN(sum_kb partial[kb][:]))          rows = KBN, the same row for every head;
//           workgroup (0, 0) writes it to cur_new (another buffer than cur_old: other workgroups still read that)
//   MODE 3: row     = LN(embed[tokens[0]][:])   (src/model/bdh.rs:319-322; a token outside [0, V) gives a NaN row, as
//           k_embed_ln does)                      partial = the embedding table, rows = V; written to cur_new too
// What bounds it: the stream of the weights, in one trip to memory.  A workgroup of 16 wavefronts owns CW columns and every
// wavefront a sixteenth of k: 16 bytes a lane, all of a workgroup's weights on their way at once, behind the partial rows,
// which are needed first.  The waves split the partial rows, D threads add up the waves' sums, every wave makes the
// LayerNorms itself (the same arithmetic in all of them, so they hold the same bits); a column's sum is sixteen chains of
// D / 16 fused multiply-adds, added in order.  4 heads of 8192 neurons, D = 256 (32 MiB of weights), us, a thread per column
// and a chain of D terms in four trips | now: MODE 1 9.0 | 8.5, MODE 2 10.6 | 9.5 (3.5 to 3.9 TB/s of weights
// that the state's stream has driven out of the caches), a token of 6 layers 242 | 230.
// PIECES: rows of W are whole, aligned 16-byte pieces; else the same lanes read their columns one by one.
struct RowArgs {
  const float *partial;
  int rows;
  const float *cur_old;
  float *cur_new;
  const int64_t *tokens;  // MODE 3
};

template <int MODE, int D, int CW, bool PIECES>
__global__ __launch_bounds__(1024) void k_relu_lowrank_row1(RowArgs a, const float *__restrict__ w, int N, float thr,
                                                           const float *__restrict__ gate, float *__restrict__ out) {
  constexpr int NW = 16, SPAN = D / NW;        // waves, k of a wave
  constexpr int LANES = CW / 4, RPI = 64 / LANES;  // lanes to a row of W, rows to an access
  constexpr int NL = SPAN / RPI;               // accesses of a lane
  constexpr int J = D / 256, U = 8 / J;        // column groups of a lane, partial rows on their way at a time
  __shared__ __attribute__((aligned(16))) float s_grp[NW * D];  // the waves' sums of the partial rows, then of the products
  __shared__ __attribute__((aligned(16))) float s_in[D];        // the sum of the partial rows, then the finished row
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hh = blockIdx.y;
  const int n0 = blockIdx.x * CW;
  const float *src = a.partial + (MODE == 1 ? (long)hh * a.rows * D : 0);
  int n_rows = a.rows;
  bool bad_token = false;
  if (MODE == 3) {
    const long tok = a.tokens[0];
    bad_token = tok < 0 || tok >= a.rows;
    src = a.partial + (bad_token ? 0 : tok) * D;
    n_rows = 1;
  }
  const int per = (n_rows + NW - 1) / NW;
  const int r0 = min(n_rows, wave * per), r1 = min(n_rows, r0 + per);
  // Loads come back in the order of their issue: the first U partial rows of every column group, then the weights, so that
  // the row is made while the weights are on their way.  (No loads under a branch: rows past the end repeat the last one.)
  float4 t[U][J];
#pragma unroll
  for (int u = 0; u < U; ++u)
#pragma unroll
    for (int j = 0; j < J; ++j)
      t[u][j] = *reinterpret_cast<const float4 *>(src + (long)min(r0 + u, n_rows - 1) * D + (j * 64 + lane) * 4);
  float4 res[J];
  if (MODE == 2) {
#pragma unroll
    for (int j = 0; j < J; ++j) res[j] = *reinterpret_cast<const float4 *>(a.cur_old + (j * 64 + lane) * 4);
  }
  const int c = n0 + (lane % LANES) * 4, k_lane = wave * SPAN + lane / LANES;
  float4 wv[NL];
  {
    const float *wp = w + ((long)hh * D + k_lane) * N;
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const float *p = wp + (long)i * RPI * N;
      if (PIECES)
        wv[i] = *reinterpret_cast<const float4 *>(p + min(c, N - 4));  // four columns are all in or all out
      else
        wv[i] = make_float4(p[min(c, N - 1)], p[min(c + 1, N - 1)], p[min(c + 2, N - 1)], p[min(c + 3, N - 1)]);
    }
  }
  const bool mine = tid < CW && n0 + tid < N;  // this thread finishes a column
  float gv = 1.0f;
  if (gate) gv = gate[(long)hh * N + min(n0 + min(tid, CW - 1), N - 1)];
#pragma unroll
  for (int j = 0; j < J; ++j) {
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (r0 + u < r1) {
        v.x += t[u][j].x; v.y += t[u][j].y; v.z += t[u][j].z; v.w += t[u][j].w;
      }
    for (int r = r0 + U; r < r1; ++r) {  // (more partial rows than 16 * U)
      const float4 x = *reinterpret_cast<const float4 *>(src + (long)r * D + (j * 64 + lane) * 4);
      v.x += x.x; v.y += x.y; v.z += x.z; v.w += x.w;
    }
    if (MODE == 3 && bad_token) v = make_float4(NAN, NAN, NAN, NAN);
    *reinterpret_cast<float4 *>(s_grp + wave * D + (j * 64 + lane) * 4) = v;
  }
  __syncthreads();
  if (tid < D) {
    float v = s_grp[tid];
#pragma unroll
    for (int g = 1; g < NW; ++g) v += s_grp[g * D + tid];
    s_in[tid] = v;
  }
  __syncthreads();
  float4 vals[J];
  float s = 0.0f;
#pragma unroll
  for (int j = 0; j < J; ++j) {
    vals[j] = *reinterpret_cast<const float4 *>(s_in + (j * 64 + lane) * 4);
    s += (vals[j].x + vals[j].y) + (vals[j].z + vals[j].w);
  }
  auto layer_norm4 = [&](float total) {  // vals <- (vals - mean) / sqrt(var + eps) over the D columns
    const float mean = bdh_wave_sum(total) / (float)D;
    float q = 0.0f;
#pragma unroll
    for (int j = 0; j < J; ++j) {
      vals[j].x -= mean; vals[j].y -= mean; vals[j].z -= mean; vals[j].w -= mean;
      q += (vals[j].x * vals[j].x + vals[j].y * vals[j].y) + (vals[j].z * vals[j].z + vals[j].w * vals[j].w);
    }
    const float den = sqrtf(bdh_wave_sum(q) / (float)D + kLnEps);
#pragma unroll
    for (int j = 0; j < J; ++j) {
      vals[j].x /= den; vals[j].y /= den; vals[j].z /= den; vals[j].w /= den;
    }
  };
  layer_norm4(s);
  if (MODE == 2) {
    s = 0.0f;
#pragma unroll
    for (int j = 0; j < J; ++j) {
      vals[j].x += res[j].x; vals[j].y += res[j].y; vals[j].z += res[j].z; vals[j].w += res[j].w;
      s += (vals[j].x + vals[j].y) + (vals[j].z + vals[j].w);
    }
    layer_norm4(s);
  }
  __syncthreads();  // every wave has read the sums
  if (wave == 0) {
#pragma unroll
    for (int j = 0; j < J; ++j) {
      *reinterpret_cast<float4 *>(s_in + (j * 64 + lane) * 4) = vals[j];
      if (MODE != 1 && blockIdx.x == 0 && hh == 0) *reinterpret_cast<float4 *>(a.cur_new + (j * 64 + lane) * 4) = vals[j];
    }
  }
  __syncthreads();

  float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
  for (int i = 0; i < NL; ++i) {
    const float x = s_in[k_lane + i * RPI];
    acc.x = __builtin_fmaf(x, wv[i].x, acc.x);
    acc.y = __builtin_fmaf(x, wv[i].y, acc.y);
    acc.z = __builtin_fmaf(x, wv[i].z, acc.z);
    acc.w = __builtin_fmaf(x, wv[i].w, acc.w);
  }
#pragma unroll
  for (int o = LANES; o < 64; o <<= 1) {  // the rows of an access
    acc.x += __shfl_xor(acc.x, o);
    acc.y += __shfl_xor(acc.y, o);
    acc.z += __shfl_xor(acc.z, o);
    acc.w += __shfl_xor(acc.w, o);
  }
  if (lane < LANES) *reinterpret_cast<float4 *>(s_grp + wave * CW + lane * 4) = acc;
  __syncthreads();
  if (!mine) return;
  float pv = s_grp[tid];
#pragma unroll
  for (int g = 1; g < NW; ++g) pv += s_grp[g * CW + tid];
  if (thr != 0.0f) pv = pv - thr;
  float y = pv > 0.0f ? pv : 0.0f;
  if (gate) y = gv * y;
  out[(long)hh * N + n0 + tid] = y;
}

// A few input rows against a SMALL weight matrix (a few MiB: it sits in the L2): with one thread per column there
// are only a handful of workgroups and each thread walks k in rounds of loads.  Here NW waves share 64
// columns: each wave asks for its own 64-row span of k at once, so every weight of the matrix is in flight
// together, and the waves then extend the column's fmaf chain one after the other in k order (the accumulator
// is handed on through LDS) -- the same k-sequential chain per output as k_relu_lowrank.  Measured per decode
// step of a whole model: 4 x 1 MiB (d=256) 141 -> 132 us, 8 x 4 MiB (d=512) 389 -> 317 us; 32 MiB a tie; at
// 256 MiB the column-per-thread kernel is 1 % ahead, hence the size limit at the call site.
template <int NW, int RT>
__global__ __launch_bounds__(NW * 64) void k_relu_lowrank_row(const float *__restrict__ in, int h_in, int T, int d,
                                                             const float *__restrict__ w, int h, int N,
                                                             const float *__restrict__ bias, float thr,
                                                             const unsigned char *__restrict__ block_active,
                                                             int block_size, int n_blocks,
                                                             const float *__restrict__ gate, float *__restrict__ out,
                                                             int M) {
  __shared__ float s_in[RT][NW * 64];
  __shared__ float s_acc[RT][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int hh = blockIdx.y;
  const int n = blockIdx.x * 64 + lane;
  const int m0 = blockIdx.z * RT;
  const bool valid = n < N;
  const int k_lo = wave * 64;
  // loads return in issue order: the input rows first, they are needed first
  float xin[RT];
#pragma unroll
  for (int r = 0; r < RT; ++r) {
    const int m = m0 + r;
    xin[r] = 0.0f;
    if ((int)threadIdx.x < d && m < M) {
      const int b = m / T, t = m - b * T;
      xin[r] = in[(((long)b * h_in + (h_in == 1 ? 0 : hh)) * T + t) * d + threadIdx.x];
    }
  }
  // unconditional loads (rows past d are clamped to the last one and not used): a load under a branch would
  // be waited for before the next one is issued
  const float *wp = w + (long)hh * d * N + (valid ? n : 0);
  float wv[64];
#pragma unroll
  for (int u = 0; u < 64; ++u) {
    const float t = wp[(long)min(k_lo + u, d - 1) * N];
    wv[u] = k_lo + u < d ? t : 0.0f;  // a select, not a branch; s_in is zero there too, so the term is +0
  }
  float gv[RT], bv = 0.0f;
#pragma unroll
  for (int r = 0; r < RT; ++r) {
    const int m = m0 + r;
    gv[r] = 1.0f;
    if (wave == NW - 1 && valid && gate && m < M) {
      const int b = m / T, t = m - b * T;
      gv[r] = gate[(((long)b * h + hh) * T + t) * N + n];
    }
  }
  if (wave == NW - 1 && valid && bias) bv = bias[(long)hh * N + n];
#pragma unroll
  for (int r = 0; r < RT; ++r) s_in[r][threadIdx.x] = xin[r];
  __syncthreads();
  float acc[RT];
#pragma unroll
  for (int r = 0; r < RT; ++r) acc[r] = 0.0f;
#pragma unroll
  for (int stage = 0; stage < NW; ++stage) {
    if (wave == stage) {
      if (stage > 0) {
#pragma unroll
        for (int r = 0; r < RT; ++r) acc[r] = s_acc[r][lane];
      }
      // unconditional, so that the LDS reads of the inputs are issued together
#pragma unroll
      for (int u = 0; u < 64; ++u)
#pragma unroll
        for (int r = 0; r < RT; ++r) acc[r] = __builtin_fmaf(s_in[r][k_lo + u], wv[u], acc[r]);
      if (stage < NW - 1) {
#pragma unroll
        for (int r = 0; r < RT; ++r) s_acc[r][lane] = acc[r];
      }
    }
    if (stage < NW - 1) __syncthreads();
  }
  if (wave != NW - 1 || !valid) return;
  float maskv = 1.0f;
  if (block_active) {
    const int blk = n / block_size;
    maskv = (blk < n_blocks && block_active[blk]) ? 1.0f : 0.0f;
  }
#pragma unroll
  for (int r = 0; r < RT; ++r) {
    const int m = m0 + r;
    if (m < M) {
      const int b = m / T, t = m - b * T;
      float p = acc[r];
      if (bias) p = p + bv;
      if (thr != 0.0f) p = p - thr;
      float y = p > 0.0f ? p : 0.0f;
      if (block_active) y = y * maskv;
      if (gate) y = gv[r] * y;
      out[(((long)b * h + hh) * T + t) * N + n] = y;
    }
  }
}

// ------------------------------------------------------------------------------------
// LayerNorm rows (one workgroup per row); in == out allowed.  The row is staged in LDS and
// every thread walks it in index order, so mean and variance are the same left-to-right f32
// sums a scalar loop produces, independent of the launch shape.
// ------------------------------------------------------------------------------------
// (s_row is 16-byte aligned; four values per LDS read, added one after the other in index order)
__device__ __forceinline__ void ln_stats_in_order(const float *s_row, int d, float &mean, float &den) {
  float sum = 0.0f;
  int i = 0;
#pragma unroll 4
  for (; i + 4 <= d; i += 4) {
    const float4 v = *reinterpret_cast<const float4 *>(s_row + i);
    sum += v.x;
    sum += v.y;
    sum += v.z;
    sum += v.w;
  }
  for (; i < d; ++i) sum += s_row[i];
  mean = sum / (float)d;
  float sq = 0.0f;
  i = 0;
#pragma unroll 4
  for (; i + 4 <= d; i += 4) {
    const float4 v = *reinterpret_cast<const float4 *>(s_row + i);
    float c;
    c = v.x - mean; sq += c * c;
    c = v.y - mean; sq += c * c;
    c = v.z - mean; sq += c * c;
    c = v.w - mean; sq += c * c;
  }
  for (; i < d; ++i) {
    const float c = s_row[i] - mean;
    sq += c * c;
  }
  den = sqrtf(sq / (float)d + kLnEps);
}

// `per` rows per workgroup of 256 threads, 256 / per threads each (see ln_rows_per_wg).
__global__ __launch_bounds__(256) void k_layer_norm(const float *__restrict__ in, float *__restrict__ out, int d, long rows,
                                                    int per) {
  extern __shared__ float s_rows[];
  const int nt = 256 / per, lane = threadIdx.x % nt;
  const long row = (long)blockIdx.x * per + threadIdx.x / nt;
  float *s_row = s_rows + (long)(threadIdx.x / nt) * ((d + 3) & ~3);
  if (row < rows)
    for (int c = lane; c < d; c += nt) s_row[c] = in[row * d + c];
  __syncthreads();
  if (row >= rows) return;
  float mean, den;
  ln_stats_in_order(s_row, d, mean, den);
  for (int c = lane; c < d; c += nt) out[row * d + c] = (s_row[c] - mean) / den;
}

// LayerNorm of many rows for internal use (the readout of a many-token state step): one wave per row, the
// statistics by wave reduction instead of the index-order sums above (d <= 64 * J).  What bounds it: a row's trip to memory
// and two sums over a wave, so all loads of a row are on their way at once and the sums are made with register moves (16352 rows of 256:
// 9.5 -> 7.7 us = 4.4 TB/s).
template <int J>
__global__ __launch_bounds__(256) void k_layer_norm_wave(const float *__restrict__ in, float *__restrict__ out, int d,
                                                         long rows) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const long row = (long)blockIdx.x * 4 + wave;
  if (row >= rows) return;
  const float *x = in + row * d;
  float *y = out + row * d;
  float v[J], s = 0.0f;
#pragma unroll
  for (int j = 0; j < J; ++j) v[j] = x[min(j * 64 + lane, d - 1)];
#pragma unroll
  for (int j = 0; j < J; ++j) s += j * 64 + lane < d ? v[j] : 0.0f;
  const float mean = bdh_wave_sum(s) / (float)d;
  float q = 0.0f;
#pragma unroll
  for (int j = 0; j < J; ++j) {
    v[j] -= mean;
    q += j * 64 + lane < d ? v[j] * v[j] : 0.0f;
  }
  const float den = sqrtf(bdh_wave_sum(q) / (float)d + kLnEps);
#pragma unroll
  for (int j = 0; j < J; ++j)
    if (j * 64 + lane < d) y[j * 64 + lane] = v[j] / den;
}

// embed gather + LayerNorm (src/model/bdh.rs:319-322), rows laid out like k_layer_norm's
__global__ __launch_bounds__(256) void k_embed_ln(const int64_t *__restrict__ tokens, int d, int V,
                                                  const float *__restrict__ embed, float *__restrict__ out, long rows, int per) {
  extern __shared__ float s_rows[];
  const int nt = 256 / per, lane = threadIdx.x % nt;
  const long row = (long)blockIdx.x * per + threadIdx.x / nt;
  float *s_row = s_rows + (long)(threadIdx.x / nt) * ((d + 3) & ~3);
  const int64_t tok = row < rows ? tokens[row] : -1;
  const bool known = tok >= 0 && tok < V;
  if (known)
    for (int c = lane; c < d; c += nt) s_row[c] = embed[tok * d + c];
  __syncthreads();
  if (row >= rows) return;
  if (!known) {  // the reference's gather would panic; poison the row instead
    for (int c = lane; c < d; c += nt) out[row * d + c] = __int_as_float(0x7fc00000);
    return;
  }
  float mean, den;
  ln_stats_in_order(s_row, d, mean, den);
  for (int c = lane; c < d; c += nt) out[row * d + c] = (s_row[c] - mean) / den;
}

__device__ const float4 g_zero_f4 = {0.0f, 0.0f, 0.0f, 0.0f};  // what a copy reads where its piece lies outside the operand

// ------------------------------------------------------------------------------------
// decoder: partial[kb][m][:] = sum_{k in block kb} mixed[m,k] * E[k,:]
// mixed[m = b*T+t, k = hh*N+n] = xy[b,hh,t,n].  Rows of E whose xy is zero for every row
// of the tile are never loaded.
// ------------------------------------------------------------------------------------
template <int RT, int MAXV, int UF = 4>
__global__ __launch_bounds__(256) void k_decoder_partial(const float *__restrict__ xy,
                                                         const float *__restrict__ E,
                                                         float *__restrict__ partial, int T, int h, int N,
                                                         int d, int KB, int M) {
  extern __shared__ float s_mem[];  // [RT][KB] xy tile, then reused for the wave reduction
  // MAXV float4 column groups per lane: columns c = (j*64+lane)*4, d <= 256*MAXV
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int kb = blockIdx.x;
  const int m0 = blockIdx.y * RT;
  const int K = h * N;
  const int nv = (d + 255) >> 8;  // float4 groups per lane
  float *s_xy = s_mem;
  for (int i = tid; i < RT * KB; i += 256) {
    const int r = i / KB, kk = i - r * KB;
    const int m = m0 + r, k = kb * KB + kk;
    float val = 0.0f;
    if (m < M && k < K) {
      const int b = m / T, t = m - b * T;
      const int hh = k / N, n = k - hh * N;
      val = xy[(((long)b * h + hh) * T + t) * N + n];
    }
    s_xy[i] = val;
  }
  __syncthreads();

  float4 acc[RT][MAXV];
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int j = 0; j < MAXV; ++j) acc[r][j] = make_float4(0.f, 0.f, 0.f, 0.f);

  // each wave takes k = wave, wave+4, ...; UF of its E rows are in flight at a time
  for (int kk0 = wave; kk0 < KB; kk0 += 4 * UF) {
    float xs[UF][RT];
    bool any[UF];
    float4 e[UF][MAXV];
#pragma unroll
    for (int u = 0; u < UF; ++u) {
      const int kk = kk0 + 4 * u;
      const int k = kb * KB + kk;
      any[u] = false;
      if (kk < KB && k < K) {
#pragma unroll
        for (int r = 0; r < RT; ++r) {
          xs[u][r] = s_xy[r * KB + kk];
          any[u] = any[u] || (xs[u][r] != 0.0f);
        }
      }
      if (any[u]) {
        const float *erow = E + (long)k * d;
#pragma unroll
        for (int j = 0; j < MAXV; ++j) {
          const int c = (j * 64 + lane) * 4;
          if (j < nv && c < d) e[u][j] = *reinterpret_cast<const float4 *>(erow + c);
        }
      }
    }
#pragma unroll
    for (int u = 0; u < UF; ++u) {
      if (any[u]) {
#pragma unroll
        for (int j = 0; j < MAXV; ++j) {
          const int c = (j * 64 + lane) * 4;
          if (j < nv && c < d) {
#pragma unroll
            for (int r = 0; r < RT; ++r) {
              acc[r][j].x = __builtin_fmaf(xs[u][r], e[u][j].x, acc[r][j].x);
              acc[r][j].y = __builtin_fmaf(xs[u][r], e[u][j].y, acc[r][j].y);
              acc[r][j].z = __builtin_fmaf(xs[u][r], e[u][j].z, acc[r][j].z);
              acc[r][j].w = __builtin_fmaf(xs[u][r], e[u][j].w, acc[r][j].w);
            }
          }
        }
      }
    }
  }
  __syncthreads();
  // cross-wave reduction, one row of the tile at a time, through LDS [4][d]
  float *s_red = s_mem;
  for (int r = 0; r < RT; ++r) {
#pragma unroll
    for (int j = 0; j < MAXV; ++j) {
      const int c = (j * 64 + lane) * 4;
      if (j < nv && c < d) *reinterpret_cast<float4 *>(s_red + wave * d + c) = acc[r][j];
    }
    __syncthreads();
    const int m = m0 + r;
    if (m < M)
      for (int c = tid; c < d; c += 256)
        partial[((long)kb * M + m) * d + c] = s_red[c] + s_red[d + c] + s_red[2 * d + c] + s_red[3 * d + c];
    __syncthreads();
  }
}

// The encoder's first stage for a batch of decoding sequences (T = 1, so a row of xy is K contiguous values): the sums of
// k_decoder_partial -- per k-block of KB rows of E four chains of fused multiply-adds over k = w, w + 4, ..., added as
// ((c0 + c1) + c2) + c3 -- on the f32 matrix cores, whose v_mfma_f32_16x16x4_f32 adds its four k one after the other.
// Four accumulators per tile, instruction w of a 16 deep step taking k = w, w + 4, w + 8, w + 12: the same bits, with
// every row of E read once per 16 * RT sequences instead of once per eight.  (SPLIT: the k-blocks of 1024 of the form for
// many sequences and a large E, one chain per block that runs 0, 8, 1, 9, ..., 7, 15 through each 16.)
// A workgroup takes the k-blocks [blk * bpw, +bpw) and adds their sums in order: bpw is a sixteenth of the blocks, as
// k_decoder_finalize would group them, or one; with SPLIT as many as leave four workgroups for every CU, and at most 64 parts
// (launch_decoder_rows).
// Tile 16 * RT x 64, copied straight to LDS 32 k at a time into a ring of NS stages, the operands of a stage read into registers
// while those of the stage before are multiplied.  What bounds it: the trips to memory of a few workgroups per CU, which is
// why the copies run NS - 1 stages ahead (two stages | now, us: 48 sequences, K = 2048, d = 512 6.3 | 5.6; 60, 16384, 256
// 30 | 19; 60, 32768, 512 65 | 36; 24, 131072, 512 189 | 71).
template <int RT, bool SPLIT, int NS>
__global__ __launch_bounds__(256) void k_decoder_rows(const float *__restrict__ xy, const float *__restrict__ E,
                                                      float *__restrict__ partial, long K, int d, int KB, int bpw, int M) {
  typedef float f32x4 __attribute__((ext_vector_type(4)));
  constexpr int BM = 16 * RT, BN = 64, SK = 32, STAGE = (BM + BN) * SK, NA = SPLIT ? 1 : 4;
  extern __shared__ __attribute__((aligned(1024))) float s_tiles[];  // NS stages of xy [BM][32], E [32][64]
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n0 = blockIdx.x * BN, m0 = blockIdx.y * BM;
  const long k_lo = (long)blockIdx.z * bpw * KB, k_hi = min(K, k_lo + (long)bpw * KB);
  // piece c of 16 bytes of row r of xy sits at place c ^ r / 2; of a row of E at place c ^ 4 x, x = which of the four k of
  // an instruction the row is: the reads below then cover the 64 banks once
  auto k_turn = [](int k) { return SPLIT ? ((k >> 3) & 1) | ((k & 1) << 1) : (k >> 2) & 3; };
  constexpr int CA = (BM * 8 + 255) / 256;
  const float *pa[CA], *pb[2];
  int ka[CA], kb[2];  // this thread's k inside a stage
#pragma unroll
  for (int c = 0; c < CA; ++c) {
    const int piece = c * 256 + tid, row = piece >> 3;
    ka[c] = ((piece & 7) ^ ((row >> 1) & 7)) * 4;
    pa[c] = xy + (long)min(m0 + row, M - 1) * K + k_lo + ka[c];
  }
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const int piece = c * 256 + tid;
    kb[c] = piece >> 4;
    pb[c] = E + (k_lo + kb[c]) * d + min(n0 + ((piece & 15) ^ (k_turn(kb[c]) << 2)) * 4, d - 4);
  }
  const float *zero = reinterpret_cast<const float *>(&g_zero_f4);
  const bool carries_xy = BM * 8 >= 256 || wave * 64 < BM * 8;  // does this wave copy pieces of xy
  auto issue = [&](long k0, int buf) {  // rows of E and values of xy beyond K are zero (K % 4 == 0)
    float *s = s_tiles + buf * STAGE;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      bdh_copy_to_lds(k0 + kb[c] < K ? pb[c] : zero, s + BM * SK + (c * 256 + wave * 64) * 4);
      pb[c] += (long)SK * d;
    }
#pragma unroll
    for (int c = 0; c < CA; ++c) {
      if (carries_xy) bdh_copy_to_lds(k0 + ka[c] < K ? pa[c] : zero, s + (c * 256 + wave * 64) * 4);
      pa[c] += SK;
    }
  };
  f32x4 total[RT], acc[NA][RT];
#pragma unroll
  for (int i = 0; i < RT; ++i) {
    total[i] = (f32x4)(0.0f);
#pragma unroll
    for (int a = 0; a < NA; ++a) acc[a][i] = (f32x4)(0.0f);
  }
  const int r = lane & 15, q = lane >> 4;
  // The operands of a stage are read into registers while those of the stage before are multiplied.
  const int stages = (int)((k_hi - k_lo + SK - 1) / SK), per_block = KB / SK;  // KB % 32 == 0
  float fa[2][2][4][RT], fb[2][2][4];
  auto read = [&](int st, int into) {
    const float *sa = s_tiles + st % NS * STAGE, *sb = sa + BM * SK;
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const int k = 16 * s + (SPLIT ? 2 * w + (q >> 1) + 8 * (q & 1) : 4 * q + w);
        fb[into][s][w] = sb[k * BN + ((wave * 16 + r) ^ (q << 4))];
#pragma unroll
        for (int i = 0; i < RT; ++i) {
          const int row = i * 16 + r;
          fa[into][s][w][i] = sa[row * SK + ((k >> 2) ^ ((row >> 1) & 7)) * 4 + (k & 3)];
        }
      }
  };
  int in_block = 0;
  auto multiply = [&](int from, bool last) {
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int w = 0; w < 4; ++w)
#pragma unroll
        for (int i = 0; i < RT; ++i)
          acc[SPLIT ? 0 : w][i] =
              __builtin_amdgcn_mfma_f32_16x16x4f32(fa[from][s][w][i], fb[from][s][w], acc[SPLIT ? 0 : w][i], 0, 0, 0);
    if (++in_block == per_block || last) {  // a k-block ends
      in_block = 0;
#pragma unroll
      for (int i = 0; i < RT; ++i) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          float v = acc[0][i][e];
          if constexpr (!SPLIT) v = ((v + acc[1][i][e]) + acc[2][i][e]) + acc[3][i][e];
          total[i][e] += v;
        }
#pragma unroll
        for (int a = 0; a < NA; ++a) acc[a][i] = (f32x4)(0.0f);
      }
    }
  };
  auto step = [&](int st, int into) {
    const int later = min(NS - 2, stages - 1 - st);
    if (carries_xy) bdh_wait_for_stage<2 + CA, NS - 2>(later);
    else bdh_wait_for_stage<2, NS - 2>(later);
    __syncthreads();  // stage st is there for every wave, and the one before has been read: its place takes stage st + NS - 1
    if (st + NS - 1 < stages) issue(k_lo + (long)(st + NS - 1) * SK, (st + NS - 1) % NS);
    read(st, into);
    if (st > 0) multiply(into ^ 1, false);
  };
  for (int st = 0; st < NS - 1 && st < stages; ++st) issue(k_lo + (long)st * SK, st);
  for (int st = 0; st < stages; st += 2) {  // two at a time: the registers have fixed names
    step(st, 0);
    if (st + 1 < stages) step(st + 1, 1);
  }
  if (stages & 1) multiply(0, true);
  else multiply(1, true);
  // element e of lane l: row = (l/16)*4 + e, column = l%16
  const int col = n0 + wave * 16 + r;
  if (col >= d) return;
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int m = m0 + i * 16 + q * 4 + e;
      if (m < M) partial[((long)blockIdx.z * M + m) * d + col] = total[i][e];
    }
}

// The encoder's first stage for ONE row (a decode step of one sequence): partial[kb][:] = sum over the KB rows of
// k-block kb of xy[k] * E[k,:], rows whose xy is zero never loaded.  Grid (k-blocks, column parts): a workgroup of NWV
// waves owns 64 * VW adjacent columns, a lane VW of them; wave w takes k = w, w + NWV, ... with UF rows in flight.
// More column parts mean fewer, larger k-blocks for the same number of waves in flight -- fewer partial rows for the
// consumer to add.
template <int VW, int UF, int NWV>
__global__ __launch_bounds__(NWV * 64) void k_decoder_partial_row(const float *__restrict__ xy,
                                                                  const float *__restrict__ E,
                                                                  float *__restrict__ partial, long K, int d, int KB) {
  extern __shared__ float s_mem[];  // [KB] xy of the block, then [NWV][64 * VW] for the wave reduction
  typedef float vec_t __attribute__((ext_vector_type(VW)));
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int kb = blockIdx.x;
  const int c = (blockIdx.y * 64 + lane) * VW;
  for (int i = tid; i < KB; i += NWV * 64) {
    const long k = (long)kb * KB + i;
    s_mem[i] = k < K ? xy[k] : 0.0f;
  }
  __syncthreads();
  float acc[VW];
#pragma unroll
  for (int e = 0; e < VW; ++e) acc[e] = 0.0f;
  for (int kk0 = wave; kk0 < KB; kk0 += NWV * UF) {
    float xs[UF];
    vec_t ev[UF];
#pragma unroll
    for (int u = 0; u < UF; ++u) {
      const int kk = kk0 + NWV * u;
      xs[u] = kk < KB ? s_mem[kk] : 0.0f;
      if (xs[u] != 0.0f && c < d) ev[u] = *reinterpret_cast<const vec_t *>(E + ((long)kb * KB + kk) * d + c);
    }
#pragma unroll
    for (int u = 0; u < UF; ++u)
      if (xs[u] != 0.0f && c < d) {
#pragma unroll
        for (int e = 0; e < VW; ++e) acc[e] = __builtin_fmaf(xs[u], ev[u][e], acc[e]);
      }
  }
  __syncthreads();
  float *s_red = s_mem;
#pragma unroll
  for (int e = 0; e < VW; ++e) s_red[wave * 64 * VW + lane * VW + e] = acc[e];
  __syncthreads();
  for (int j = tid; j < 64 * VW; j += NWV * 64) {
    const int cc = blockIdx.y * 64 * VW + j;
    if (cc < d) {
      float v = s_red[j];
#pragma unroll
      for (int g = 1; g < NWV; ++g) v += s_red[g * 64 * VW + j];
      partial[(long)kb * d + cc] = v;
    }
  }
}

// logits[m,:] = cur[m,:] . lm_head ; optional argmax of the last token of each sequence.
// 1024 threads: 256 vocabulary columns x 4 groups over k; the four partial dot products of a
// logit are added in group order.  s_cur holds the input row (every thread sees it), s_acc has 1024 floats.
__device__ __forceinline__ void lm_head_row(const float *s_cur, float *s_acc, float *s_best, int *s_arg, int m,
                                            const float *__restrict__ W, int T, int d, int V,
                                            float *__restrict__ logits, int64_t *__restrict__ next_tokens) {
  const int tid = threadIdx.x & 255, grp = threadIdx.x >> 8;
  const int lane = tid & 63, wave = tid >> 6;
  const int per = (d + 3) >> 2;
  const int k0 = grp * per, k1 = min(d, k0 + per);
  float best = -INFINITY;
  int arg = 0x7fffffff;
  for (int c0 = 0; c0 < V; c0 += 256) {
    const int c = c0 + tid;
    float acc = 0.0f;
    if (c < V) {
      int k = k0;
      for (; k + 16 <= k1; k += 16) {  // 16 independent loads in flight, then the chain
        float w[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) w[u] = W[(long)(k + u) * V + c];
#pragma unroll
        for (int u = 0; u < 16; ++u) acc = __builtin_fmaf(s_cur[k + u], w[u], acc);
      }
      for (; k < k1; ++k) acc = __builtin_fmaf(s_cur[k], W[(long)k * V + c], acc);
    }
    s_acc[grp * 256 + tid] = acc;
    __syncthreads();
    if (grp == 0 && c < V) {
      const float v = ((s_acc[tid] + s_acc[256 + tid]) + s_acc[512 + tid]) + s_acc[768 + tid];
      logits[(long)m * V + c] = v;
      if (v > best) {  // increasing c: keeps the lowest index on ties
        best = v;
        arg = c;
      }
    }
    __syncthreads();
  }
  const int b = m / T, t = m - b * T;
  const bool want = next_tokens && t == T - 1;  // uniform over the workgroup
  if (!want) return;
  for (int o = 32; o > 0; o >>= 1) {
    const float ob = __shfl_xor(best, o);
    const int oa = __shfl_xor(arg, o);
    if (ob > best || (ob == best && oa < arg)) {
      best = ob;
      arg = oa;
    }
  }
  if (grp == 0 && lane == 0) {
    s_best[wave] = best;
    s_arg[wave] = arg;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < 4; ++w)
      if (s_best[w] > best || (s_best[w] == best && s_arg[w] < arg)) {
        best = s_best[w];
        arg = s_arg[w];
      }
    next_tokens[b] = arg == 0x7fffffff ? 0 : arg;
  }
}

// cur[m,:] = LN(cur[m,:] + LN(sum_kb partial[kb][m][:]))   (src/model/bdh.rs:438-441)
// 1024 threads = 16 groups of 64 lanes; a lane owns four adjacent columns (one 16-byte load per partial
// row), a group adds a sixteenth of the k-block partials in index order with up to 16 loads in flight,
// the groups are combined in order; after the one barrier the first wavefront applies the two LayerNorms
// with wave shuffles only.
// HEAD: the output head of the same row follows in the same launch (the last layer of a model): the finished row
// goes to LDS as well, and all 1024 threads run lm_head_row on it -- the arithmetic of k_lm_head, one launch less.
template <bool HEAD>
__global__ __launch_bounds__(1024) void k_decoder_finalize(const float *__restrict__ partial, int KBN, int M,
                                                           int d, float *__restrict__ cur, DecoderHead head) {
  __shared__ float s_grp[16][1024];
  __shared__ float s_best[4];
  __shared__ int s_arg[4];
  const int m = blockIdx.x, lane = threadIdx.x & 63, grp = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int per = (KBN + 15) >> 4;
  const int kb0 = min(KBN, grp * per), kb1 = min(KBN, kb0 + per);
  // the residual row is fetched while the partials are summed: it was written by another
  // workgroup of an earlier launch, so the load is a trip to memory
  float res[16];
  if (grp == 0) {
#pragma unroll
    for (int j = 0; j < 16; ++j) res[j] = (j * 64 + lane < d) ? cur[(long)m * d + j * 64 + lane] : 0.0f;
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int c = (j * 64 + lane) * 4;  // d % 4 == 0
    if (c < d) {
      typedef float Quad __attribute__((ext_vector_type(4)));
      const Quad q = bdh_sum_in_order(reinterpret_cast<const Quad *>(partial + ((long)kb0 * M + m) * d + c), (long)M * d / 4, kb1 - kb0);
      *reinterpret_cast<Quad *>(&s_grp[grp][c]) = q;
    }
  }
  __syncthreads();
  if (threadIdx.x >= 64) {  // the first wave finishes the row alone
    if (!HEAD) return;      // (no barrier follows)
  } else {
  float vals[16];  // column c = j*64 + lane, d <= 1024
  float s = 0.0f;
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    const int c = j * 64 + lane;
    float v = 0.0f;
    if (c < d) {
      v = s_grp[0][c];
#pragma unroll
      for (int g = 1; g < 16; ++g) v += s_grp[g][c];
      s += v;
    }
    vals[j] = v;
  }
  float mean = bdh_wave_sum(s) / (float)d;
  float q = 0.0f;
#pragma unroll
  for (int j = 0; j < 16; ++j)
    if (j * 64 + lane < d) {
      const float t = vals[j] - mean;
      q += t * t;
    }
  float den = sqrtf(bdh_wave_sum(q) / (float)d + kLnEps);
  s = 0.0f;
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    const int c = j * 64 + lane;
    if (c < d) {
      const float mlp = (vals[j] - mean) / den;
      vals[j] = res[j] + mlp;
      s += vals[j];
    }
  }
  mean = bdh_wave_sum(s) / (float)d;
  q = 0.0f;
#pragma unroll
  for (int j = 0; j < 16; ++j)
    if (j * 64 + lane < d) {
      const float t = vals[j] - mean;
      q += t * t;
    }
  den = sqrtf(bdh_wave_sum(q) / (float)d + kLnEps);
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    const int c = j * 64 + lane;
    if (c < d) {
      const float y = (vals[j] - mean) / den;
      cur[(long)m * d + c] = y;
      if (HEAD) s_grp[2][c] = y;  // only this wave reads s_grp after the barrier above, and it has read all of it
    }
  }
  }
  if (!HEAD) return;
  __syncthreads();  // the row is in s_grp[2]; rows 3.. are free for the partial dot products
  lm_head_row(s_grp[2], s_grp[3], s_best, s_arg, m, head.lm_head, head.T, d, head.V, head.logits, head.next_tokens);
}

// k_decoder_finalize<false> for many rows: a wavefront per row (d <= 64 * J), the partials of a column added in the same order
// (sixteen groups, each in index order), then the same wave-wide LayerNorms, so the same bits.  What bounds it: the reads of
// the partials, U of them for all columns on their way at once; a workgroup of sixteen wavefronts per row spends most of its
// time in its one barrier once the rows alone fill the chip (4088 rows of 256, 4 partials: 56 us against 7).
// One column after the other, a trip to memory each, it took 9.7; 1500 rows of 256, 16 partials 22 -> 9.
template <int J, int U>
__global__ __launch_bounds__(256) void k_decoder_finalize_rows(const float *__restrict__ partial, int KBN, int M, int d,
                                                               float *__restrict__ cur) {
  const int lane = threadIdx.x & 63;
  const long m = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (m >= M) return;
  const int per = (KBN + 15) >> 4;
  const long step = (long)M * d;
  const float *p = partial + m * d;
  float vals[J], t[J], res[J];
  float s = 0.0f;
  int col[J];
#pragma unroll
  for (int j = 0; j < J; ++j) {
    col[j] = min(j * 64 + lane, d - 1);
    res[j] = cur[m * d + col[j]];
    vals[j] = t[j] = 0.0f;
  }
  int in_group = 0;
  for (int kb = 0; kb < KBN; kb += U) {
    float x[U][J];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int j = 0; j < J; ++j) x[u][j] = p[min(kb + u, KBN - 1) * step + col[j]];
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (kb + u < KBN) {
        const bool first = in_group == 0, last = in_group + 1 == per || kb + u == KBN - 1;
#pragma unroll
        for (int j = 0; j < J; ++j) {
          t[j] = first ? x[u][j] : t[j] + x[u][j];
          if (last) vals[j] = kb + u < per ? t[j] : vals[j] + t[j];
        }
        in_group = last ? 0 : in_group + 1;
      }
  }
#pragma unroll
  for (int j = 0; j < J; ++j) s += j * 64 + lane < d ? vals[j] : 0.0f;
  auto spread = [&](float mean) {  // sqrt(var + eps)
    float q = 0.0f;
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const float c = vals[j] - mean;
      q += j * 64 + lane < d ? c * c : 0.0f;
    }
    return sqrtf(bdh_wave_sum(q) / (float)d + kLnEps);
  };
  float mean = bdh_wave_sum(s) / (float)d;
  float den = spread(mean);
  s = 0.0f;
#pragma unroll
  for (int j = 0; j < J; ++j) {
    vals[j] = res[j] + (vals[j] - mean) / den;
    s += j * 64 + lane < d ? vals[j] : 0.0f;
  }
  mean = bdh_wave_sum(s) / (float)d;
  den = spread(mean);
#pragma unroll
  for (int j = 0; j < J; ++j)
    if (j * 64 + lane < d) cur[m * d + j * 64 + lane] = (vals[j] - mean) / den;
}

// The output head of many rows: RT rows share every weight that is read, a thread per vocabulary column; each logit is the
// same four k-sequential chains as in lm_head_row, added in order.  (One row per workgroup reads all of W again for every
// row: 66 against 24 us for 4088 rows, d = 256, V = 256.)  With next_tokens the greedy token of a sequence's last row.
template <int RT>
__global__ __launch_bounds__(256) void k_lm_head_rows(const float *__restrict__ cur, const float *__restrict__ W, int M,
                                                      int T, int d, int V, float *__restrict__ logits,
                                                      int64_t *__restrict__ next_tokens) {
  extern __shared__ float s_x[];  // [d][RT]
  __shared__ float s_best[4];
  __shared__ int s_arg[4];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int m0 = blockIdx.x * RT;
  for (int i = tid; i < RT * d; i += 256) {
    const int r = i / d, k = i - r * d;
    s_x[k * RT + r] = cur[(long)min(m0 + r, M - 1) * d + k];
  }
  __syncthreads();
  const int per = (d + 3) >> 2;
  float best[RT];
  int arg[RT];
#pragma unroll
  for (int r = 0; r < RT; ++r) {
    best[r] = -INFINITY;
    arg[r] = 0x7fffffff;
  }
  for (int c0 = 0; c0 < V; c0 += 256) {
    const int c = c0 + tid, cc = min(c, V - 1);
    float sum[RT];
    for (int grp = 0; grp < 4; ++grp) {
      const int k0 = grp * per, k1 = min(d, k0 + per);
      float acc[RT];
#pragma unroll
      for (int r = 0; r < RT; ++r) acc[r] = 0.0f;
      int k = k0;
      for (; k + 32 <= k1; k += 32) {  // 32 independent loads in flight, then the chains
        float w[32];
#pragma unroll
        for (int u = 0; u < 32; ++u) w[u] = W[(long)(k + u) * V + cc];
#pragma unroll
        for (int u = 0; u < 32; ++u)
#pragma unroll
          for (int r = 0; r < RT; ++r) acc[r] = __builtin_fmaf(s_x[(k + u) * RT + r], w[u], acc[r]);
      }
      for (; k < k1; ++k) {
        const float w = W[(long)k * V + cc];
#pragma unroll
        for (int r = 0; r < RT; ++r) acc[r] = __builtin_fmaf(s_x[k * RT + r], w, acc[r]);
      }
#pragma unroll
      for (int r = 0; r < RT; ++r) sum[r] = grp == 0 ? acc[r] : sum[r] + acc[r];
    }
    if (c < V) {
#pragma unroll
      for (int r = 0; r < RT; ++r) {
        if (m0 + r < M) logits[(long)(m0 + r) * V + c] = sum[r];
        if (sum[r] > best[r]) {  // increasing c: keeps the lowest index on ties
          best[r] = sum[r];
          arg[r] = c;
        }
      }
    }
  }
  if (!next_tokens) return;
#pragma unroll
  for (int r = 0; r < RT; ++r) {
    const int m = m0 + r;
    if (m >= M || m % T != T - 1) continue;  // uniform over the workgroup
    float bv = best[r];
    int ba = arg[r];
    for (int o = 32; o > 0; o >>= 1) {
      const float ob = __shfl_xor(bv, o);
      const int oa = __shfl_xor(ba, o);
      if (ob > bv || (ob == bv && oa < ba)) {
        bv = ob;
        ba = oa;
      }
    }
    __syncthreads();  // the previous row's result has been read
    if (lane == 0) {
      s_best[wave] = bv;
      s_arg[wave] = ba;
    }
    __syncthreads();
    if (tid == 0) {
      for (int w = 1; w < 4; ++w)
        if (s_best[w] > bv || (s_best[w] == bv && s_arg[w] < ba)) {
          bv = s_best[w];
          ba = s_arg[w];
        }
      next_tokens[m / T] = ba == 0x7fffffff ? 0 : ba;
    }
  }
}

__global__ __launch_bounds__(1024) void k_lm_head(const float *__restrict__ cur, const float *__restrict__ W,
                                                  int T, int d, int V, float *__restrict__ logits,
                                                  int64_t *__restrict__ next_tokens) {
  extern __shared__ float s_dyn[];  // [d] input row, then [4][256] partials
  __shared__ float s_best[4];
  __shared__ int s_arg[4];
  const int m = blockIdx.x;
  for (int k = threadIdx.x; k < d; k += 1024) s_dyn[k] = cur[(long)m * d + k];
  __syncthreads();
  lm_head_row(s_dyn, s_dyn + d, s_best, s_arg, m, W, T, d, V, logits, next_tokens);
}

__global__ void k_advance_positions(int32_t *pos, int B, int delta) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b < B) {
    const long v = (long)pos[b] + delta;
    pos[b] = v > 0x7fffffffL ? 0x7fffffff : (int32_t)v;  // saturating, as state.position (src/model/bdh.rs:445)
  }
}

template <int RT>
void launch_relu(hipStream_t st, dim3 grid, size_t lds, const ReluLowrankParams &p, const unsigned char *mask,
                 int M) {
  constexpr int UK = RT == 1 ? 64 : 16;      // weight rows in flight per thread (the counter of outstanding loads ends at 63)
  constexpr int NTHR = RT == 1 ? 128 : 256;  // a single input row: smaller workgroups, one per CU at N*h = 32768
  grid.x = (p.N + NTHR - 1) / NTHR;
  hipLaunchKernelGGL((k_relu_lowrank<RT, UK, NTHR>), grid, dim3(NTHR), lds, st, p.in, p.h_in, p.T, p.d, p.weight,
                     p.h, p.N, p.bias, p.threshold, mask, p.block_size, p.n_blocks, p.gate, p.out, M);
}

}  // namespace

int bdh_launch_relu_lowrank(bdh_ctx *ctx, const ReluLowrankParams &p) {
  const long M = (long)p.B * p.T;
  if (M > 0x7fffffffL) return bdh_fail(ctx, BDH_E_SHAPE, "B*T too large");
  const unsigned char *mask_dev = nullptr;
  if (p.active_blocks_host) {
    // The device copy of the mask is kept with the bytes it was made from: the two projections of every layer of
    // a call (and the calls after it) pass the same pattern, and only a new pattern costs a copy and a wait (the
    // caller's host buffer may go away on return, and kernels still queued may read the old copy).
    const size_t nb = (size_t)std::max(p.n_blocks, 0);
    const bool same = ctx->lat_mask && ctx->lat_mask_key.size() == nb &&
                      (nb == 0 || memcmp(ctx->lat_mask_key.data(), p.active_blocks_host, nb) == 0);
    if (!same) {
      BDH_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));
      if (ctx->lat_mask_bytes < nb + 256) {
        if (ctx->lat_mask) BDH_HIP_CHECK(ctx, hipFree(ctx->lat_mask));
        ctx->lat_mask = nullptr;
        ctx->lat_mask_bytes = 0;
        ctx->lat_mask_key.clear();
        if (hipMalloc(&ctx->lat_mask, nb + 256) != hipSuccess) {
          (void)hipGetLastError();
          return bdh_fail(ctx, BDH_E_NOMEM, "latent block mask of %zu bytes", nb);
        }
        ctx->lat_mask_bytes = nb + 256;
      }
      if (nb > 0) BDH_HIP_CHECK(ctx, hipMemcpy(ctx->lat_mask, p.active_blocks_host, nb, hipMemcpyHostToDevice));
      ctx->lat_mask_key.assign(p.active_blocks_host, p.active_blocks_host + nb);
    }
    mask_dev = static_cast<const unsigned char *>(ctx->lat_mask);
  }
  // D_y of a prompt has no order to keep (it decides no active set): split-bf16 products where those are faster
  if (p.any_order && p.gate && !p.bias && !mask_dev && p.d > 0 && p.N > 0 && ctx->opt_lowrank_split != 0 &&
      (ctx->opt_lowrank_split == 1 || bdh_relu_lowrank_split_pays(ctx, p)))
    return bdh_launch_relu_lowrank_split(ctx, p);
  const bool pieces = p.d % 32 == 0 && p.N % 4 == 0 && bdh_aligned(p.in, 16) && bdh_aligned(p.weight, 16);
  // A matrix of up to 16 MiB (it sits in the L2) and few outputs: 64 columns per workgroup, every weight in flight at once,
  // as many rows per workgroup (1, 2, 4, 8) as still give a workgroup per CU.  The line is at 32768 outputs, 128 for every
  // CU (us, this | 16-row matrix-core tiles: h*N = 2048, d = 512, 16 rows 7.6 | 8.8, 24 rows 12.8 | 8.9; 1024, 256, 32 rows
  // 5.4 | 6.0, 48 rows 6.3 | 6.0; 4096, 256, 8 rows 5.4 | 6.0, 16 rows 7.6 | 6.0; 8192, 512, 4 rows 7.5 | 8.9, 8 rows 11.1 | 8.9).
  // Fewer than 64 rows that do not come in 16-byte pieces have the thread-per-column kernel for an alternative, a chain of d
  // LDS reads: four times as many outputs then, eight times up to d = 256 (us, this | that: h*N = 4088, d = 250, 63 rows
  // 13.0 | 17.6; 16376, 200, 16 rows 12.8 | 15.0, 24 rows 20 | 15; 4104, 500, 24 rows 19 | 29, 32 rows 33 | 29; 8192, 260, 8 rows
  // 10.5 | 17.2, 24 rows 33 | 17.5).
  const long n_cu_rl = ctx->n_cu > 0 ? ctx->n_cu : 256;
  const long row_line = (pieces || M >= 64 ? 128 : p.d <= 256 ? 1024 : 512) * n_cu_rl;
  if (p.d >= 128 && p.d <= 512 && ctx->opt_lowrank_row != 0 &&
      sizeof(float) * (size_t)p.h * p.d * p.N <= (size_t(16) << 20) && (M == 1 || M * p.h * p.N <= row_line)) {
    const long col_blocks = (p.N + 63) / 64;
    int rt = 1;
    if (M > 1) {
      rt = 8;
      while (rt > 1 && col_blocks * p.h * ((M + rt - 1) / rt) < n_cu_rl) rt >>= 1;
      while (rt > M) rt >>= 1;
    }
    const long row_tiles = (M + rt - 1) / rt;
    if (row_tiles > 65535 || p.h > 65535) return bdh_fail(ctx, BDH_E_SHAPE, "grid too large (row tiles %ld)", row_tiles);
    const dim3 grid((unsigned)col_blocks, p.h, (unsigned)row_tiles);
#define BDH_ROW(NW_, RT_)                                                                                             \
  hipLaunchKernelGGL((k_relu_lowrank_row<NW_, RT_>), grid, dim3(NW_ * 64), 0, ctx->stream, p.in, p.h_in, p.T, p.d,   \
                     p.weight, p.h, p.N, p.bias, p.threshold, mask_dev, p.block_size, p.n_blocks, p.gate, p.out, (int)M)
#define BDH_ROW_RT(NW_)                                                                           \
  do {                                                                                            \
    if (rt == 8) BDH_ROW(NW_, 8); else if (rt == 4) BDH_ROW(NW_, 4); else if (rt == 2) BDH_ROW(NW_, 2); \
    else BDH_ROW(NW_, 1);                                                                         \
  } while (0)
    if (p.d <= 128) BDH_ROW_RT(2); else if (p.d <= 256) BDH_ROW_RT(4); else BDH_ROW_RT(8);
#undef BDH_ROW_RT
#undef BDH_ROW
    BDH_LAUNCH_CHECK(ctx, "k_relu_lowrank_row");
    return BDH_OK;
  }
  // Two rows and more: the f32 matrix cores, same values, the weights streamed once per row tile (options: fewer than 64
  // rows from mfma_rows on, more from gemm_rows on; 0 = never).  Fewer than 32 rows want the 16-byte pieces of the copying
  // kernels; what is left, and a single row of a larger matrix, runs a thread per column with its input rows in LDS, which
  // reads the weights again for every eight rows (without pieces, us, this | the checked 64 x 64 tiles: h*N = 65520, d = 250,
  // 16 rows 26 | 35, 24 rows 35 | 35, 32 rows 44 | 36, 63 rows 79 | 41; d = 100, 24 rows 16 | 18, 48 rows 26 | 20).  Eight rows
  // and more that do not fit there (d above 2048) take the matrix cores whatever the options say.
  const int mc_rows = std::abs(M < 64 ? ctx->opt_lowrank_mfma_rows : ctx->opt_lowrank_gemm_rows);
  const int RT = M >= 8 ? 8 : (M >= 4 ? 4 : (M >= 2 ? 2 : 1));
  const size_t lds = sizeof(float) * (size_t)RT * (p.d > 0 ? p.d : 1);
  if (p.d > 0 && p.N > 0 && M > 1 &&
      ((mc_rows > 0 && M >= mc_rows && (M >= 32 || pieces)) || (RT == 8 && lds > 64 * 1024)))
    return bdh_launch_relu_lowrank_gemm(ctx, p, mask_dev);
  if (lds > 64 * 1024) return bdh_fail(ctx, BDH_E_SHAPE, "d=%d too large for the projection tile", p.d);
  const long row_tiles = (M + RT - 1) / RT;
  if (row_tiles > 65535 || p.h > 65535) return bdh_fail(ctx, BDH_E_SHAPE, "grid too large (row tiles %ld)", row_tiles);
  dim3 grid((p.N + 255) / 256, p.h, (unsigned)row_tiles);
  switch (RT) {
    case 8: launch_relu<8>(ctx->stream, grid, lds, p, mask_dev, (int)M); break;
    case 4: launch_relu<4>(ctx->stream, grid, lds, p, mask_dev, (int)M); break;
    case 2: launch_relu<2>(ctx->stream, grid, lds, p, mask_dev, (int)M); break;
    default: launch_relu<1>(ctx->stream, grid, lds, p, mask_dev, (int)M); break;
  }
  BDH_LAUNCH_CHECK(ctx, "k_relu_lowrank");
  return BDH_OK;
}

// Rows of an index-order LayerNorm kernel per workgroup of 256 threads.  The sums are the same work in every wavefront, so four
// rows to a workgroup once there are more than two workgroups of one for every CU (us, one | four rows: 1536 x 256 10.3 | 6.7,
// 1024 x 1000 26 | 18, 512 x 1000 16.1 | 17.6, 64 x 4096 55 | 63: with few rows the loads and stores of a row want all four
// wavefronts); wider rows than 4096 fit into LDS one at a time.
static int ln_rows_per_wg(const bdh_ctx *ctx, int64_t rows, int d) { return d <= 4096 && rows > 2L * (ctx->n_cu > 0 ? ctx->n_cu : 256) ? 4 : 1; }
static size_t ln_lds(int d, int per) { return sizeof(float) * (size_t)((d + 3) & ~3) * per; }

int bdh_launch_layer_norm(bdh_ctx *ctx, int64_t rows, int d, const float *in, float *out) {
  if (rows > 0x7fffffffL) return bdh_fail(ctx, BDH_E_SHAPE, "too many rows");
  if (d > 16384) return bdh_fail(ctx, BDH_E_SHAPE, "LayerNorm row of %d floats does not fit in LDS", d);
  if (rows == 0) return BDH_OK;
  const int per = ln_rows_per_wg(ctx, rows, d);
  hipLaunchKernelGGL(k_layer_norm, dim3((unsigned)((rows + per - 1) / per)), dim3(256), ln_lds(d, per), ctx->stream, in, out, d,
                     (long)rows, per);
  BDH_LAUNCH_CHECK(ctx, "k_layer_norm");
  return BDH_OK;
}

int bdh_launch_layer_norm_rows(bdh_ctx *ctx, int64_t rows, int d, const float *in, float *out) {
  if (d > 1024) return bdh_launch_layer_norm(ctx, rows, d, in, out);
  const int64_t blocks = (rows + 3) / 4;
  if (blocks > 0x7fffffffL) return bdh_fail(ctx, BDH_E_SHAPE, "too many rows");
  if (rows == 0) return BDH_OK;
  auto *kernel = d <= 256 ? k_layer_norm_wave<4> : d <= 512 ? k_layer_norm_wave<8> : k_layer_norm_wave<16>;
  hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(256), 0, ctx->stream, in, out, d, (long)rows);
  BDH_LAUNCH_CHECK(ctx, "k_layer_norm_wave");
  return BDH_OK;
}

int bdh_launch_embed_ln(bdh_ctx *ctx, const int64_t *tokens, int64_t rows, int d, int V, const float *embed,
                        float *out) {
  if (rows == 0) return BDH_OK;
  const int per = ln_rows_per_wg(ctx, rows, d);
  hipLaunchKernelGGL(k_embed_ln, dim3((unsigned)((rows + per - 1) / per)), dim3(256), ln_lds(d, per), ctx->stream, tokens, d, V,
                     embed, out, (long)rows, per);
  BDH_LAUNCH_CHECK(ctx, "k_embed_ln");
  return BDH_OK;
}

// From this many rows on they fill the chip a wavefront (second stage) or four to a workgroup (head) each; fewer rows want
// many wavefronts on one row: with 4 to 32 partials to add, one wavefront is a chain of trips to memory.
constexpr int kManyRows = 256;

static void launch_lm_head(bdh_ctx *ctx, int M, int T, int d, int V, const float *cur, const float *lm_head, float *logits,
                           int64_t *next_tokens) {
  constexpr int RT = 4;
  if (M >= kManyRows && sizeof(float) * RT * (size_t)d <= 64 * 1024)
    hipLaunchKernelGGL((k_lm_head_rows<RT>), dim3((M + RT - 1) / RT), dim3(256), sizeof(float) * RT * (size_t)d, ctx->stream,
                       cur, lm_head, M, T, d, V, logits, next_tokens);
  else
    hipLaunchKernelGGL(k_lm_head, dim3(M), dim3(1024), sizeof(float) * ((size_t)d + 1024), ctx->stream, cur, lm_head, T, d, V,
                       logits, next_tokens);
}

static void launch_decoder_finalize(bdh_ctx *ctx, const float *partial, int KBN, int M, int d, float *cur,
                                    const DecoderHead *head) {
  if (M >= kManyRows) {
    auto *kernel = d <= 256   ? k_decoder_finalize_rows<4, 4>
                   : d <= 512 ? k_decoder_finalize_rows<8, 4>
                              : k_decoder_finalize_rows<16, 2>;
    hipLaunchKernelGGL(kernel, dim3((M + 3) / 4), dim3(256), 0, ctx->stream, partial, KBN, M, d, cur);
    if (head) launch_lm_head(ctx, M, head->T, d, head->V, cur, head->lm_head, head->logits, head->next_tokens);
  } else if (head) {
    hipLaunchKernelGGL(k_decoder_finalize<true>, dim3(M), dim3(1024), 0, ctx->stream, partial, KBN, M, d, cur, *head);
  } else {
    hipLaunchKernelGGL(k_decoder_finalize<false>, dim3(M), dim3(1024), 0, ctx->stream, partial, KBN, M, d, cur,
                       DecoderHead{});
  }
}

// The whole encoder of a batch of decoding sequences by k_decoder_rows.  In the form with the VALU kernel's bits the second
// stage adds the k-blocks in sixteen groups, and a workgroup adds up a whole group where the groups alone give every CU a
// workgroup; the tile is 16 rows while that leaves at most four workgroups for every CU, the chain of one tile being what
// counts, else 32, or 64 for more rows than that, so that E passes fewer times.  In the other form (one chain per k-block of
// 1024) a workgroup takes as many k-blocks as leave four workgroups for every CU, and at most 64 parts for the second stage;
// 32 rows a tile where those tiles give every CU two (us of both kernels: 24 sequences, K = 131072, d = 512, 32 rows, two
// k-blocks 71 + 8, one 75 + 11, eight with 16 rows 131 + 6; 60, 32768, 512, one 36 + 7, two with 16 rows 47 + 6; 48, 131072,
// 512, 32 rows, two 110, 64 rows, two 114).
static int launch_decoder_rows(bdh_ctx *ctx, int M, long K, int d, int KB, bool split, const float *xy, const float *decoder,
                               float *cur, const DecoderHead *head) {
  const long n_cu = ctx->n_cu > 0 ? ctx->n_cu : 256;
  const int KBN = (int)((K + KB - 1) / KB), per = (KBN + 15) / 16;
  auto tiles = [&](int rows) { return (long)((d + 63) / 64) * ((M + rows - 1) / rows); };
  int bpw, rt;
  if (split) {
    rt = M > 16 && tiles(32) * KBN >= 2 * n_cu ? 2 : 1;
    bpw = (int)std::max<long>((KBN + 63) / 64, std::min<long>(per, tiles(16 * rt) * KBN / (4 * n_cu)));
  } else {
    bpw = tiles(16) * ((KBN + per - 1) / per) >= n_cu ? per : 1;
    rt = tiles(16) * ((KBN + bpw - 1) / bpw) <= 4 * n_cu ? 1 : M <= 32 ? 2 : 4;
  }
  int parts = (KBN + bpw - 1) / bpw;
  int rc = bdh_ws_reserve(ctx, sizeof(float) * (size_t)parts * M * d);
  if (rc == BDH_E_NOMEM && split && bpw < per) {  // less room: sixteen parts
    bpw = per;
    parts = (KBN + bpw - 1) / bpw;
    rc = bdh_ws_reserve(ctx, sizeof(float) * (size_t)parts * M * d);
  }
  if (rc != BDH_OK) return rc;
  float *partial = static_cast<float *>(ctx->ws);
  const dim3 grid((d + 63) / 64, (M + 16 * rt - 1) / (16 * rt), parts);
  if (grid.y > 65535 || grid.z > 65535) return bdh_fail(ctx, BDH_E_SHAPE, "grid too large (%d rows, %d parts)", M, parts);
#define BDH_DR(RT_, SPLIT_, NS_)                                                                                       \
  hipLaunchKernelGGL((k_decoder_rows<RT_, SPLIT_, NS_>), grid, dim3(256), NS_ * (16 * RT_ + 64) * 32 * sizeof(float), \
                     ctx->stream, xy, decoder, partial, K, d, KB, bpw, M)
  if (split) {
    if (rt == 1) BDH_DR(1, true, 4); else BDH_DR(2, true, 3);
  } else {
    if (rt == 1) BDH_DR(1, false, 4); else if (rt == 2) BDH_DR(2, false, 3); else BDH_DR(4, false, 3);
  }
#undef BDH_DR
  BDH_LAUNCH_CHECK(ctx, "k_decoder_rows");
  launch_decoder_finalize(ctx, partial, parts, M, d, cur, head);
  BDH_LAUNCH_CHECK(ctx, "k_decoder_finalize");
  return BDH_OK;
}

int bdh_launch_decoder_residual(bdh_ctx *ctx, int B, int T, int h, int N, int d, const float *xy,
                                const float *decoder, float *cur, const DecoderHead *head) {
  const int M = B * T;
  const long K = (long)h * N;
  if (d > 1024 || (d & 3)) return bdh_fail(ctx, BDH_E_SHAPE, "decoder needs d %% 4 == 0 and d <= 1024, got %d", d);
  // a prompt: products on the matrix cores, all of E streamed once per row tile (fewer rows skip the inactive rows of E)
  if (T >= 16 && M >= 24 && ctx->opt_decoder_mfma != 0) {
    int rows = 0;
    int rc = bdh_launch_decoder_partials_f32(ctx, B, T, h, N, d, xy, decoder, &rows);
    if (rc != BDH_OK) return rc;
    launch_decoder_finalize(ctx, static_cast<float *>(ctx->ws), rows, M, d, cur, head);
    BDH_LAUNCH_CHECK(ctx, "k_decoder_finalize");
    return BDH_OK;
  }
  const long n_cu = ctx->n_cu > 0 ? ctx->n_cu : 256;
  const int RT = M >= 8 && d <= 512 ? 8 : (M >= 4 ? 4 : (M >= 2 ? 2 : 1));  // (wider rows: four in registers)
  const int row_tiles = (M + RT - 1) / RT;
  // k-block size: enough workgroups to fill the chip, few enough partials
  // about two workgroups per CU: more k-blocks only add partials for the second stage to read
  int KB = 1024;
  while (KB > 128 && ((K + KB - 1) / KB) * row_tiles < 2 * n_cu) KB >>= 1;
  // a small model: down to 32 rows of E per workgroup, until there is a workgroup per CU
  while (KB > 32 && ((K + KB - 1) / KB) * row_tiles < n_cu) KB >>= 1;
  // A batch of decoding sequences: the f32 matrix cores, the same bits; k-blocks of 1024 with a chain each once those fill
  // half the chip in 32 x 64 tiles (a negative option value -r: from r sequences on, whatever the size).  The VALU kernel
  // skips the rows of E that no sequence needs and reads the others once per eight sequences: the longer the rows, the larger E
  // and the fewer neurons fire, the longer it is the better one.  Its time a step over this kernel's, half of the neurons firing |
  // a twentieth: E of 4 to 8 MiB, 2 sequences 1.02 to 1.06 | 1.00 to 1.02; d = 256, 10 to 16 MiB, 2 sequences 0.95 to 1.03 | 0.90 to
  // 0.96, 3 sequences 1.04 to 1.09 | 0.98 to 1.02, 32 MiB, 8 sequences 1.09 | 1.05, 48 MiB 1.04 | 0.95; d = 128, 64 MiB, 8 sequences 1.07 |
  // 1.04; d = 384 to 768, 10 to 16 MiB, 2 sequences 0.92 to 0.97 | 0.88 to 0.95, 8 sequences 0.99 to 1.02 | 0.96 to 1.01, 12 sequences 1.00
  // to 1.06 | 0.97 to 1.07.
  const int sk_rows = ctx->opt_decoder_splitk_rows;
  const long many = std::abs(sk_rows);
  const long mib = (K * d * 4 + (1L << 20) - 1) >> 20;
  const long few = many > 24 ? many
                   : std::min<long>(many, mib <= 8 ? 2 : d > 256 ? (mib <= 16 ? 12 : 24) : mib <= 16 ? 3 : d <= 128 || mib <= 32 ? 8 : 24);
  if (T == 1 && M >= few && (K & 3) == 0 && bdh_aligned(xy, 16) && bdh_aligned(decoder, 16)) {
    const bool split = M >= many && K % 1024 == 0 &&
                       (sk_rows < 0 || K / 1024 * ((d + 63) / 64) * ((M + 31) / 32) >= n_cu / 2);
    if (split) KB = 1024;
    return launch_decoder_rows(ctx, M, K, d, KB, split, xy, decoder, cur, head);
  }
  const int KBN = (int)((K + KB - 1) / KB);
  size_t lds = sizeof(float) * (size_t)RT * KB;
  if (lds < sizeof(float) * 4u * d) lds = sizeof(float) * 4u * d;
  const size_t pbytes = sizeof(float) * (size_t)KBN * M * d;
  int rc = bdh_ws_reserve(ctx, pbytes);
  if (rc != BDH_OK) return rc;
  float *partial = static_cast<float *>(ctx->ws);
  dim3 grid(KBN, row_tiles);
#define BDH_DEC(RT_, MV_)                                                                                   \
  hipLaunchKernelGGL((k_decoder_partial<RT_, MV_>), grid, dim3(256), lds, ctx->stream, xy, decoder, partial, T, h, \
                     N, d, KB, M)
  const int mv = d <= 256 ? 1 : (d <= 512 ? 2 : 4);
  if (mv == 1) {
    if (RT == 8) BDH_DEC(8, 1); else if (RT == 4) BDH_DEC(4, 1); else if (RT == 2) BDH_DEC(2, 1);
    else  // one row: the kernel is a chain of round trips, so more E rows per trip
      hipLaunchKernelGGL((k_decoder_partial<1, 1, 16>), grid, dim3(256), lds, ctx->stream, xy, decoder, partial, T, h, N, d,
                         KB, M);
  } else if (mv == 2) {
    if (RT == 8) BDH_DEC(8, 2); else if (RT == 4) BDH_DEC(4, 2); else if (RT == 2) BDH_DEC(2, 2);
    else
      hipLaunchKernelGGL((k_decoder_partial<1, 2, 8>), grid, dim3(256), lds, ctx->stream, xy, decoder, partial, T, h, N, d,
                         KB, M);
  } else {
    if (RT == 4) BDH_DEC(4, 4); else if (RT == 2) BDH_DEC(2, 4); else BDH_DEC(1, 4);
  }
#undef BDH_DEC
  BDH_LAUNCH_CHECK(ctx, "k_decoder_partial");
  launch_decoder_finalize(ctx, partial, KBN, M, d, cur, head);
  BDH_LAUNCH_CHECK(ctx, "k_decoder_finalize");
  return BDH_OK;
}

int bdh_launch_relu_lowrank_row(bdh_ctx *ctx, const ReluLowrankRowParams &p) {
  if ((p.d != 256 && p.d != 512) || p.N < 1 || p.rows < 1)
    return bdh_fail(ctx, BDH_E_SHAPE, "fused row projection: d=%d N=%d rows=%d", p.d, p.N, p.rows);
  const RowArgs a{p.partial, p.rows, p.cur_old, p.cur_new, p.tokens};
  const bool pieces = p.N % 4 == 0 && bdh_aligned(p.weight, 16);
  // Columns of a workgroup: a workgroup for every CU if narrower ones give that; wider ones add up the partial rows less often.
  const long n_cu = ctx->n_cu > 0 ? ctx->n_cu : 256;
  auto groups = [&](int cw) { return (long)((p.N + cw - 1) / cw) * p.h; };
  const int cw = groups(128) >= n_cu ? 128 : groups(64) >= n_cu ? 64 : 32;
  const dim3 grid((p.N + cw - 1) / cw, p.h);
#define BDH_ROW1(MODE_, D_, CW_, PIECES_)                                                                                   \
  hipLaunchKernelGGL((k_relu_lowrank_row1<MODE_, D_, CW_, PIECES_>), grid, dim3(1024), 0, ctx->stream, a, p.weight, p.N, \
                     p.threshold, p.gate, p.out)
#define BDH_ROW1_P(MODE_, D_, CW_) \
  do { if (pieces) BDH_ROW1(MODE_, D_, CW_, true); else BDH_ROW1(MODE_, D_, CW_, false); } while (0)
#define BDH_ROW1_C(MODE_, D_) \
  do { if (cw == 128) BDH_ROW1_P(MODE_, D_, 128); else if (cw == 64) BDH_ROW1_P(MODE_, D_, 64); else BDH_ROW1_P(MODE_, D_, 32); } while (0)
#define BDH_ROW1_D(MODE_) \
  do { if (p.d == 256) BDH_ROW1_C(MODE_, 256); else BDH_ROW1_C(MODE_, 512); } while (0)
  if (p.mode == 1) BDH_ROW1_D(1);
  else if (p.mode == 2) BDH_ROW1_D(2);
  else BDH_ROW1_D(3);
#undef BDH_ROW1_D
#undef BDH_ROW1_C
#undef BDH_ROW1_P
#undef BDH_ROW1
  BDH_LAUNCH_CHECK(ctx, "k_relu_lowrank_row1");
  return BDH_OK;
}

int bdh_launch_decoder_partial_row(bdh_ctx *ctx, int h, int N, int d, const float *xy, const float *decoder, int KB,
                                   float *partial, int *KBN_out) {
  const long K = (long)h * N;
  if (d > 1024 || (d & 3)) return bdh_fail(ctx, BDH_E_SHAPE, "decoder needs d %% 4 == 0 and d <= 1024, got %d", d);
  const int KBN = (int)((K + KB - 1) / KB);
  // 16 waves per workgroup; two columns per lane (128-column parts) up to d = 256, four beyond
  constexpr int NWV = 16;
  const int VW = d <= 256 ? 2 : 4;
  const size_t lds = sizeof(float) * std::max<size_t>((size_t)KB, (size_t)NWV * 64 * VW);
  const dim3 grid(KBN, (d + 64 * VW - 1) / (64 * VW));
  if (VW == 2)
    hipLaunchKernelGGL((k_decoder_partial_row<2, 16, NWV>), grid, dim3(NWV * 64), lds, ctx->stream, xy, decoder, partial, K, d, KB);
  else
    hipLaunchKernelGGL((k_decoder_partial_row<4, 16, NWV>), grid, dim3(NWV * 64), lds, ctx->stream, xy, decoder, partial, K, d, KB);
  BDH_LAUNCH_CHECK(ctx, "k_decoder_partial_row");
  *KBN_out = KBN;
  return BDH_OK;
}

int bdh_launch_decoder_finalize_head(bdh_ctx *ctx, const float *partial, int KBN, int M, int d, float *cur,
                                     const DecoderHead *head) {
  if (d > 1024 || (d & 3) != 0) return bdh_fail(ctx, BDH_E_SHAPE, "encoder second stage needs d %% 4 == 0 and d <= 1024");
  launch_decoder_finalize(ctx, partial, KBN, M, d, cur, head);
  BDH_LAUNCH_CHECK(ctx, "k_decoder_finalize");
  return BDH_OK;
}

int bdh_launch_decoder_finalize(bdh_ctx *ctx, const float *partial, int KBN, int M, int d, float *cur) {
  if (d > 1024 || (d & 3) != 0) return bdh_fail(ctx, BDH_E_SHAPE, "encoder second stage needs d %% 4 == 0 and d <= 1024");
  launch_decoder_finalize(ctx, partial, KBN, M, d, cur, nullptr);
  BDH_LAUNCH_CHECK(ctx, "k_decoder_finalize");
  return BDH_OK;
}

int bdh_launch_lm_head(bdh_ctx *ctx, int B, int T, int d, int V, const float *cur, const float *lm_head,
                       float *logits, int64_t *next_tokens) {
  launch_lm_head(ctx, B * T, T, d, V, cur, lm_head, logits, next_tokens);
  BDH_LAUNCH_CHECK(ctx, "k_lm_head");
  return BDH_OK;
}

int bdh_launch_advance_positions(bdh_ctx *ctx, int32_t *positions_dev, int B, int delta) {
  hipLaunchKernelGGL(k_advance_positions, dim3((B + 255) / 256), dim3(256), 0, ctx->stream, positions_dev, B, delta);
  BDH_LAUNCH_CHECK(ctx, "k_advance_positions");
  return BDH_OK;
}
