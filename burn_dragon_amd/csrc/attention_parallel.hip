// Parallel (all tokens at once) normalised causal linear attention in f32:
// kernel::linear_attention::fused_state_aligned (src/kernel/linear_attention.rs:11-115) and, with
// the dense block pattern, Attention::forward (src/model/attention.rs:142-175).
//
// This is the reference's training-path form; it is kept in f32 and follows the reference's
// block semantics exactly (including the ALiBi term being added to every entry of an active
// block).  Small problems take a row-per-workgroup kernel; from T = 128 on the two products run
// on the matrix cores (gemm_f32.hip): S = mask(Q Q^T) + bias is materialised per slice, and
// out = (S V) / (norm + eps) sums |S| on the way.  The bf16 form for inference is in prefill.hip.
// The many-token form of the state step, the encoder E over many rows and relu_lowrank over many
// rows are here as well.
#include <algorithm>
#include <cstring>
#include <vector>

#include "gemm_f32.h"
#include "lds_copy.h"

namespace {

struct FsaSlopes {
  float v[64];
};


constexpr float kTwoPi = 6.28318530717958647692f;
constexpr float kRowNormEps = 1e-6f;  // src/kernel/linear_attention.rs:9
constexpr float kLnEps = 1e-5f;       // src/model/bdh.rs:17

// q_rot [S,T,Nq] from query [S,T,N], positions 0..T (src/kernel/linear_attention.rs:23-40)
__global__ __launch_bounds__(256) void k_rotate_f32(const float *__restrict__ x, const float *__restrict__ freqs,
                                                    float *__restrict__ q, int T, int N, int rotary) {
  const long row = blockIdx.x;  // slice * T + t
  const int t = (int)(row % T);
  const float pos = (float)t;
  const float *xr = x + row * N;
  const int Nq = rotary == BDH_POPE ? 2 * N : N;
  float *qr = q + row * Nq;
  for (int n = threadIdx.x; n < N; n += 256) {
    const float raw = pos * freqs[n];
    const float ph = (raw - floorf(raw)) * kTwoPi;
    float s, c;
    sincosf(ph, &s, &c);
    if (rotary == BDH_ROPE) {
      const float rot = (n & 1) ? xr[n - 1] : -xr[n + 1];
      const float a = xr[n] * c, r = rot * s;
      qr[n] = a + r;
    } else {
      const float m = logf(expf(xr[n] * 1.0f) + 1.0f) / 1.0f;  // softplus(x, 1)
      qr[n] = m * c;
      qr[N + n] = m * s;
    }
  }
}

// q [S,Tc,Nq] from rows t0..t0+Tc of x [S][T][N] (x points at row t0 of slice 0), token t of the chunk at
// position pos0 + t, or pos_dev[b] + pos_add + t with per-sequence positions.  The arithmetic is that of
// the decode step kernels (src/model/attention.rs:305-330), so the rotated values are the same bits.
__global__ __launch_bounds__(256) void k_rotate_chunk_f32(const float *__restrict__ x, long x_slice_stride,
                                                          const float *__restrict__ freqs, float *__restrict__ q,
                                                          int Tc, int N, int rotary, long pos0,
                                                          const int32_t *__restrict__ pos_dev, int pos_add, int h) {
  const long row = blockIdx.x;  // slice * Tc + t
  const long slice = row / Tc;
  const int t = (int)(row - slice * Tc);
  const float pos = (float)((pos_dev ? (long)pos_dev[slice / h] + pos_add : pos0) + t);
  const float *xr = x + slice * x_slice_stride + (long)t * N;
  const int Nq = rotary == BDH_POPE ? 2 * N : N;
  float *qr = q + row * Nq;
  if (rotary == BDH_ROPE) {  // N is even: one lane per pair
    for (int pr = threadIdx.x; pr < (N >> 1); pr += 256) {
      const float2 xv = reinterpret_cast<const float2 *>(xr)[pr];
      float2 o = make_float2(0.0f, 0.0f);
      if (xv.x != 0.0f || xv.y != 0.0f) {
        const float2 fv = reinterpret_cast<const float2 *>(freqs)[pr];
        const float raw0 = pos * fv.x, raw1 = pos * fv.y;
        float s0, c0, s1, c1;
        sincosf((raw0 - floorf(raw0)) * kTwoPi, &s0, &c0);
        sincosf((raw1 - floorf(raw1)) * kTwoPi, &s1, &c1);
        const float a0 = xv.x * c0, r0 = (-xv.y) * s0;
        const float a1 = xv.y * c1, r1 = xv.x * s1;
        o.x = a0 + r0;
        o.y = a1 + r1;
      }
      reinterpret_cast<float2 *>(qr)[pr] = o;
    }
    return;
  }
  for (int n = threadIdx.x; n < N; n += 256) {
    const float raw = pos * freqs[n];
    const float ph = (raw - floorf(raw)) * kTwoPi;
    float sn, cs;
    sincosf(ph, &sn, &cs);
    const float m = logf(expf(xr[n] * 1.0f) + 1.0f) / 1.0f;  // softplus(x, 1)
    qr[n] = m * cs;
    qr[N + n] = m * sn;
  }
}

// stamps[b,h,n] = clock (or clocks_dev[b] + add), saturated to the stamp range
__global__ __launch_bounds__(256) void k_set_stamps(int32_t *__restrict__ stamps, long rows, long rows_per_seq,
                                                    long clock, const int32_t *__restrict__ clocks_dev, int add) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= rows) return;
  const long c = clocks_dev ? (long)clocks_dev[i / rows_per_seq] + add : clock;
  stamps[i] = (int32_t)min(c, 0x7fffffffL);
}

// bf16 <-> f32 copies of a whole state (grid-stride); f32 -> bf16 rounds to nearest even
__global__ __launch_bounds__(256) void k_widen_bf16(const unsigned short *__restrict__ in, float *__restrict__ out,
                                                    size_t n) {
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256)
    out[i] = __uint_as_float(static_cast<unsigned int>(in[i]) << 16);
}
__global__ __launch_bounds__(256) void k_narrow_bf16(const float *__restrict__ in, unsigned short *__restrict__ out,
                                                     size_t n) {
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) {
    unsigned int u = __float_as_uint(in[i]);
    if ((u & 0x7fffffffu) > 0x7f800000u) {
      out[i] = static_cast<unsigned short>((u >> 16) | 0x40);
    } else {
      u += 0x7fffu + ((u >> 16) & 1u);
      out[i] = static_cast<unsigned short>(u >> 16);
    }
  }
}

// one workgroup per (slice, query row i)
__global__ __launch_bounds__(256) void k_fsa_row(const float *__restrict__ q, const float *__restrict__ v,
                                                 FsaSlopes slopes_dev, int use_alibi, int h,
                                                 int T, int Nq, int dv, int block_size,
                                                 const unsigned char *__restrict__ active,  // [tb*tb] or null
                                                 int tb, int row_normalize, float *__restrict__ out) {
  extern __shared__ float s_mem[];
  float *s_q = s_mem;          // [Nq]
  float *s_sc = s_mem + Nq;    // [T]
  __shared__ float s_part[4];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const long slice = blockIdx.x / T;
  const int i = (int)(blockIdx.x - slice * T);
  const int hh = (int)(slice % h);
  const long b = slice / h;
  const float *Q = q + slice * (long)T * Nq;
  const float *V = v + b * (long)T * dv;
  const int rb = i / block_size;
  const float slope = use_alibi ? slopes_dev.v[hh] : 0.0f;
  for (int n = tid; n < Nq; n += 256) s_q[n] = Q[(long)i * Nq + n];
  __syncthreads();
  bool any = false;
  float nsum = 0.0f;
  for (int j = wave; j < T; j += 4) {
    const int cb = j / block_size;
    const bool act = active ? (active[(long)rb * tb + cb] != 0) : (cb <= rb);
    float s = 0.0f;
    if (act) {
      any = true;
      if (!(rb == cb && j >= i)) {  // tril(-1) on diagonal blocks
        const float *qj = Q + (long)j * Nq;
        float part = 0.0f;
        for (int n = lane; n < Nq; n += 64) part = __builtin_fmaf(s_q[n], qj[n], part);
        for (int o = 32; o > 0; o >>= 1) part += __shfl_xor(part, o);
        s = part;
      }
      if (use_alibi) {
        const float al = slope * ((float)j - (float)i);
        s = s + al;
      }
      nsum += fabsf(s);
    }
    if (lane == 0) s_sc[j] = s;
  }
  // any / norm across waves (each wave saw a different subset of j; lanes of a wave agree)
  if (lane == 0) s_part[wave] = nsum;
  const int any_all = __syncthreads_or(any ? 1 : 0);
  const float norm = s_part[0] + s_part[1] + s_part[2] + s_part[3];
  const float den = norm + kRowNormEps;
  float *o = out + (slice * (long)T + i) * dv;
  for (int c = tid; c < dv; c += 256) {
    float acc = 0.0f;
    for (int j = 0; j < T; ++j) {
      const float s = s_sc[j];
      if (s != 0.0f) acc = __builtin_fmaf(s, V[(long)j * dv + c], acc);
    }
    o[c] = (any_all && row_normalize) ? acc / den : acc;
  }
}

// The sums of a scores product whose K was cut into parts: S[row][col] = sum of the parts in order, then the mask, the
// decay and the ALiBi term of the GEMM_SCORES epilogue.  One workgroup per row; columns up to the end of the last time
// block of the row's 128-row group (nothing reads beyond it), all of them with a sparse pattern.
__global__ __launch_bounds__(256) void k_scores_reduce(const float *__restrict__ parts, long c_split, GemmF32 g) {
  const long r = blockIdx.x;
  const int slice = (int)(r / g.M), row = (int)(r - (long)slice * g.M);
  const int bs = g.block_size;
  const int end = g.active ? g.N : min(g.N, ((min((row | 127) + 1, g.M) - 1) / bs + 1) * bs);
  const float *p = parts + ((long)slice * g.M + row) * g.N;
  float *C = g.C + (long)(slice / g.mod) * g.c_s1 + (long)(slice % g.mod) * g.c_s2 + (long)row * g.ldc;
  const int rb = bdh_time_block(g, row);
  const float ld = g.log_decay[slice % g.heads], slope = g.slopes[slice % g.heads];
  for (int col = threadIdx.x; col < end; col += 256) {
    const int cb = bdh_time_block(g, col);
    const bool act = g.active ? g.active[(long)rb * g.tb + cb] != 0 : cb <= rb;
    float v = 0.0f;
    if (act) {
      if (!(rb == cb && col >= row)) {
        int k = 0;
        for (; k + 4 <= g.ks; k += 4) {  // four parts on their way at a time
          float t[4];
#pragma unroll
          for (int u = 0; u < 4; ++u) t[u] = p[(k + u) * c_split + col];
#pragma unroll
          for (int u = 0; u < 4; ++u) v += t[u];
        }
        for (; k < g.ks; ++k) v += p[k * c_split + col];
      }
      if (g.decay_scores && col < row) v = v * expf((float)(row - col) * ld);
      if (g.use_alibi) {
        const float al = slope * ((float)col - (float)row);
        v = v + al;
      }
    }
    C[col] = v;
  }
}

// out[slice][t0 + t][:] = the sum of the parts [part][slice][tc][d], in order, and, when out_ln is given, its LayerNorm
// (src/model/bdh.rs:359).  One wavefront per row, d <= 64 * J.  What bounds it: the trips to memory, one for U parts of the whole
// row (one part and 64 columns at a time, us: 32 parts, 140 rows of 384 25.8 | 6.2; 8 parts, 786 rows of 512 19.2 | 5.2; 2 parts, 5496 rows of
// 128 5.0 | 4.9).
template <int J, int U>
__global__ __launch_bounds__(256) void k_rows_reduce(const float *__restrict__ parts, int ks, long c_split, int tc, int d,
                                                     long rows, float *__restrict__ out, float *__restrict__ out_ln,
                                                     long slice_stride) {
  const int lane = threadIdx.x & 63;
  const long r = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (r >= rows) return;
  const long o = r / tc * slice_stride + r % tc * d;
  const float *p = parts + r * d;
  float v[J], s = 0.0f;
  int col[J];
#pragma unroll
  for (int j = 0; j < J; ++j) {
    col[j] = min(j * 64 + lane, d - 1);
    v[j] = 0.0f;
  }
  for (int k = 0; k < ks; k += U) {
    float x[U][J];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int j = 0; j < J; ++j) x[u][j] = p[min(k + u, ks - 1) * c_split + col[j]];
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (k + u < ks) {
#pragma unroll
        for (int j = 0; j < J; ++j) v[j] += x[u][j];
      }
  }
#pragma unroll
  for (int j = 0; j < J; ++j)
    if (j * 64 + lane < d) {
      out[o + j * 64 + lane] = v[j];
      s += v[j];
    }
  if (!out_ln) return;
  const float mean = bdh_wave_sum(s) / (float)d;
  float q = 0.0f;
#pragma unroll
  for (int j = 0; j < J; ++j)
    if (j * 64 + lane < d) q += (v[j] - mean) * (v[j] - mean);
  const float den = sqrtf(bdh_wave_sum(q) / (float)d + kLnEps);
#pragma unroll
  for (int j = 0; j < J; ++j)
    if (j * 64 + lane < d) out_ln[o + j * 64 + lane] = (v[j] - mean) / den;
}

// ------------------------------------------------------------------------------------
// relu_lowrank over many rows on the f32 matrix cores: [M, d] x [d, N] per head.
// The eight matrix instructions of a 16-wide k stage take k = 0,1 | 2,3 | ...; v_mfma_f32_32x32x2_f32 adds its two k-steps
// one after the other as fused multiply-adds, so every output is ONE k-sequential fmaf chain -- the bits of k_relu_lowrank.
// The rows of all sequences of the call form one list (row m = token m % T of sequence m / T): a ragged T costs at most
// one partly filled tile per head and not one per sequence.
// ------------------------------------------------------------------------------------
typedef float f32x16 __attribute__((ext_vector_type(16)));
constexpr int FK = 16;    // k per LDS stage
constexpr int FLD = 20;   // LDS row stride of A in floats (80 bytes: 16-byte aligned, spreads the banks)

struct RlArgs {
  const float *A, *W;
  float *C;
  long a_outer, a_head;     // row m of head hh: A + (m / T) * a_outer + hh * a_head + (m % T) * d
  int T, M, N, d, h;
  int mt, nt;               // tile grid of one head
  const float *bias;        // [h][N] or null
  float thr;
  const unsigned char *mask;  // one byte per latent block (device) or null
  int block, n_blocks;
  const float *gate;        // laid out like C, or null
};

// What the two kernels below share: which tile, and what becomes of the sums.
template <int BM, int BN, int NWM, int NWN>
struct RlTile {
  static constexpr int MI = BM / NWM / 32, NJ = BN / NWN / 32;
  int hh, m0, n0, lane, wm, wn;
  // false: a workgroup of the rounding-up.  Each XCD takes one contiguous eighth of the (head, tile) list (workgroup ids are
  // dealt round-robin to the XCDs), tiles column by column: neighbours share a block of weight columns in one L2.
  __device__ __forceinline__ bool init(const RlArgs &g) {
    const int tiles = g.mt * g.nt;
    const long total = (long)g.h * tiles;
    const int xcd = blockIdx.x & 7;
    const long at = total * xcd / 8 + (blockIdx.x >> 3);
    if (at >= total * (xcd + 1) / 8) return false;
    hh = (int)(at / tiles);
    const int tile = (int)(at % tiles);
    m0 = (tile % g.mt) * BM;
    n0 = (tile / g.mt) * BN;
    lane = threadIdx.x & 63;
    wm = (threadIdx.x >> 6) / NWN;
    wn = (threadIdx.x >> 6) % NWN;
    return true;
  }
  // row m of A, clamped to the last one (the sums of the repeats are not stored)
  __device__ __forceinline__ const float *a_row(const RlArgs &g, int m) const {
    m = min(m, g.M - 1);
    return g.A + (long)(m / g.T) * g.a_outer + (long)hh * g.a_head + (long)(m % g.T) * g.d;
  }
  // C = gate * mask * relu(acc + bias - thr) (src/kernel/relu_lowrank.rs:7-37); accumulator element e of lane l in a
  // 32x32 tile: row = (e/4)*8 + (l/32)*4 + (e%4), col = l%32.  The place of a row is worked out once per four adjacent
  // rows, and the gate values of a 32x32 tile are all asked for, under no branch, before the first of them is used.
  __device__ __forceinline__ void finish(const RlArgs &g, const f32x16 (&acc)[MI][NJ]) const {
    const bool whole = m0 + BM <= g.M && n0 + BN <= g.N;
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      long at_row[16];
      int rows[16];
#pragma unroll
      for (int e4 = 0; e4 < 4; ++e4) {
        const int row = m0 + wm * (BM / NWM) + i * 32 + e4 * 8 + (lane >> 5) * 4;
        int b = row / g.T, t = row - b * g.T;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          rows[e4 * 4 + e] = row + e;
          at_row[e4 * 4 + e] = (((long)b * g.h + hh) * g.T + t) * g.N;
          if (++t == g.T) { t = 0; ++b; }
        }
      }
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        const int col = n0 + wn * (BN / NWN) + j * 32 + (lane & 31);
        const int cc = min(col, g.N - 1);
        const float bv = g.bias ? g.bias[(long)hh * g.N + cc] : 0.0f;
        float mk = 1.0f;
        if (g.mask) {
          const int blk = cc / g.block;
          mk = (blk < g.n_blocks && g.mask[blk]) ? 1.0f : 0.0f;
        }
        // the gate and the output are touched once per call: streaming accesses leave the L2 to the operand tiles
        float gv[16];
        if (g.gate) {
          const long last = (((long)(g.M / g.T - 1) * g.h + hh) * g.T + g.T - 1) * g.N;
#pragma unroll
          for (int e = 0; e < 16; ++e) gv[e] = __builtin_nontemporal_load(g.gate + min(at_row[e], last) + cc);
        }
        float y[16];
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          float pv = acc[i][j][e];
          if (g.bias) pv = pv + bv;
          if (g.thr != 0.0f) pv = pv - g.thr;
          y[e] = pv > 0.0f ? pv : 0.0f;
          if (g.mask) y[e] = y[e] * mk;
          if (g.gate) y[e] = gv[e] * y[e];
        }
        if (whole) {
#pragma unroll
          for (int e = 0; e < 16; ++e) __builtin_nontemporal_store(y[e], g.C + at_row[e] + col);
        } else if (col < g.N) {
#pragma unroll
          for (int e = 0; e < 16; ++e)
            if (rows[e] < g.M) __builtin_nontemporal_store(y[e], g.C + at_row[e] + col);
        }
      }
    }
  }
};

// d a multiple of 32, N of 4, 16-byte aligned operands: both tiles go from memory straight into LDS (no registers, no
// address arithmetic to wait for), 32 k at a time into two buffers in turn, one barrier per stage.  The 16-byte pieces of
// a row of A (128 bytes), and those of an odd k row of W, are rotated against each other so that the 16-byte reads of 16
// consecutive rows of A, and the 4-byte reads of two k rows of W, cover the 64 banks once.  What bounds it: the f32 matrix
// instruction (64 cycles for 32 x 32 x 2: 157 TFLOP/s); [1500 x 256] x [256 x 32768] 412 -> 273 us (92 TFLOP/s, of which
// about 60 us the 200 MB of output), [8192 x 512] x [512 x 131072] 9.8 -> 9.1 ms (120), [128 x 256] x [256 x 1024] 17 -> 10 us
// against the same products staged through registers, whose loads were waited for where they were issued.
template <int BM, int BN>
__global__ __launch_bounds__(256) void k_relu_lowrank_direct(RlArgs g) {
  using Tl = RlTile<BM, BN, 2, 2>;
  constexpr int MI = Tl::MI, NJ = Tl::NJ, SK = 32;
  constexpr int AP = SK / 4;  // pieces of a row of A
  auto a_turn = [](int row) { return (row >> 1) & 7; };
  constexpr int CA = BM * SK / 4 / 256, CB = BN * SK / 4 / 256;  // 16-byte pieces per thread and stage
  extern __shared__ __attribute__((aligned(1024))) float s_tiles[];  // two stages of A [BM][32], W [32][BN]
  constexpr int STAGE = (BM + BN) * SK;
  Tl t;
  if (!t.init(g)) return;
  const int tid = threadIdx.x, lane = t.lane, wave = tid >> 6;
  const float *W = g.W + (long)t.hh * g.d * g.N;
  const float *pa[CA], *pb[CB];
#pragma unroll
  for (int c = 0; c < CA; ++c) {
    const int piece = c * 256 + tid, row = piece / AP;
    pa[c] = t.a_row(g, t.m0 + row) + ((piece % AP) ^ a_turn(row)) * 4;
  }
#pragma unroll
  for (int c = 0; c < CB; ++c) {
    const int piece = c * 256 + tid, k = piece / (BN / 4);
    const int nc = ((piece % (BN / 4)) ^ ((k & 1) << 3)) * 4;
    pb[c] = W + (long)k * g.N + min(t.n0 + nc, g.N - 4);  // four columns are all in or all out
  }
  const long b_step = (long)SK * g.N;
  auto issue = [&](int buf) {
#pragma unroll
    for (int c = 0; c < CA; ++c) {
      bdh_copy_to_lds(pa[c], s_tiles + buf * STAGE + (c * 256 + wave * 64) * 4);
      pa[c] += SK;
    }
#pragma unroll
    for (int c = 0; c < CB; ++c) {
      bdh_copy_to_lds(pb[c], s_tiles + buf * STAGE + BM * SK + (c * 256 + wave * 64) * 4);
      pb[c] += b_step;
    }
  };
  f32x16 acc[MI][NJ];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;
  const int r = lane & 31, half = lane >> 5;
  issue(0);
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  int cur = 0;
  for (int k0 = 0; k0 < g.d; k0 += SK) {
    if (k0 + SK < g.d) issue(cur ^ 1);  // lands while the matrix cores work on this stage
    const float *sa = s_tiles + cur * STAGE, *sb = sa + BM * SK;
    // four k at a time: instruction 0 takes k = 4c, 4c + 1, instruction 1 takes 4c + 2, 4c + 3.  The operands of the next
    // four are on their way while these are multiplied.
    float4 va[2][MI];
    float vb[2][2][NJ];
    auto fragments = [&](int c) {
#pragma unroll
      for (int i = 0; i < MI; ++i) {
        const int row = t.wm * (BM / 2) + i * 32 + r;
        va[c & 1][i] = *reinterpret_cast<const float4 *>(sa + row * SK + (c ^ a_turn(row)) * 4);
      }
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        const int col = (t.wn * (BN / 2) + j * 32 + r) ^ (half << 5);
        vb[c & 1][0][j] = sb[(4 * c + half) * BN + col];
        vb[c & 1][1][j] = sb[(4 * c + 2 + half) * BN + col];
      }
    };
    fragments(0);
#pragma unroll
    for (int c = 0; c < AP; ++c) {
      if (c + 1 < AP) fragments(c + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int i = 0; i < MI; ++i) {
          const float4 v = va[c & 1][i];
          const float a = q == 0 ? (half ? v.y : v.x) : (half ? v.w : v.z);
#pragma unroll
          for (int j = 0; j < NJ; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, vb[c & 1][q][j], acc[i][j], 0, 0, 0);
        }
    }
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    cur ^= 1;
  }
  t.finish(g, acc);
}

// Few rows, or few tiles: 16 * RT rows x 64 columns per workgroup on v_mfma_f32_16x16x4_f32, whose four k-steps are also
// added one after the other (the bits of the scalar chain again).  A wavefront owns 16 columns, so a chain of d steps takes
// 8 cycles a step and row tile where the 32 x 32 instruction takes 32, and a few rows give four times the wavefronts: what
// bounds it is the stream of the weights, every one of them copied to LDS once per 16 * RT rows.
// Where the workgroups are few, it is the chain of waits: a stage's copies are NS - 1 stages ahead, its operands are read
// into registers while those of the stage before are multiplied, and the gate is asked for with the first copies (us, before | now, D_x
// and D_y of a decode step: 8 heads of 256, d = 512, 48 sequences 10.5 | 8.2; 4 heads of 4096, d = 256, 3 sequences 8.0 | 6.1).
// WHOLE: LDS holds all NS stages of d = 32 NS, the whole tile is on its way before the first wait, four stages to a barrier
// (us, ring of four | whole: d = 512, 32 to 256 workgroups 8.2 | 6.5, d = 256, up to 512 of them 5.6 | 4.5; what is left is the chain
// of d / 4 instructions, 32 cycles each).
// us per call, the VALU and matrix-core kernels it took over from | this: 8192, 512, 48 rows 52.5 | 11.5; 32768, 256, 16 rows
// 29.7 | 8.4; 131072, 512 (268 MB of weights), 16 rows 57.9 | 47.8, 32 rows 65.5 | 58.6.
template <int RT, int NS, bool WHOLE>
__global__ __launch_bounds__(256) void k_relu_lowrank_rows(RlArgs g) {
  typedef float f32x4 __attribute__((ext_vector_type(4)));
  constexpr int BM = 16 * RT, BN = 64, SK = 32;
  constexpr int STAGE = (BM + BN) * SK;
  __shared__ __attribute__((aligned(1024))) float s_tiles[NS * STAGE];  // NS stages of A [BM][32], W [32][64]
  const int tiles = g.mt * g.nt, total = g.h * tiles;  // the launcher keeps the total within an int
  const int xcd = blockIdx.x & 7;
  const int lo = (int)((long)total * xcd / 8), hi = (int)((long)total * (xcd + 1) / 8);
  const int at = lo + (int)(blockIdx.x >> 3);
  if (at >= hi) return;
  const int hh = at / tiles, tile = at - hh * tiles;
  const int col_tile = tile / g.mt;
  const int m0 = (tile - col_tile * g.mt) * BM, n0 = col_tile * BN;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const float *W = g.W + (long)hh * g.d * g.N;
  // row m of A and of C: sequence, token
  auto place = [&](int m, int &b, int &t) {
    b = g.T == 1 ? m : m / g.T;
    t = g.T == 1 ? 0 : m - b * g.T;
  };
  // A: BM * 8 pieces of 16 bytes, W: 512; a piece of row r of A sits at place (piece ^ r / 2), one of k row k of W at place
  // (piece ^ 4 (k % 4)): the 4-byte reads below then cover the 64 banks once
  constexpr int CA = (BM * 8 + 255) / 256;
  const float *pa[CA], *pb[2];
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const int piece = c * 256 + tid, k = piece >> 4;
    pb[c] = W + (long)k * g.N + min(n0 + ((piece & 15) ^ ((k & 3) << 2)) * 4, g.N - 4);
  }
#pragma unroll
  for (int c = 0; c < CA; ++c) {
    const int piece = c * 256 + tid, row = piece >> 3;
    int b, t;
    place(min(m0 + row, g.M - 1), b, t);
    pa[c] = g.A + (long)b * g.a_outer + (long)hh * g.a_head + (long)t * g.d + ((piece & 7) ^ ((row >> 1) & 7)) * 4;
  }
  const long b_step = (long)SK * g.N;
  const bool carries_a = BM * 8 >= 256 || wave * 64 < BM * 8;  // does this wave copy pieces of A
  auto issue = [&](int buf) {
    float *s = s_tiles + buf * STAGE;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      bdh_copy_to_lds(pb[c], s + BM * SK + (c * 256 + wave * 64) * 4);
      pb[c] += b_step;
    }
#pragma unroll
    for (int c = 0; c < CA; ++c) {
      if (carries_a) bdh_copy_to_lds(pa[c], s + (c * 256 + wave * 64) * 4);
      pa[c] += SK;
    }
  };
  // where element e of row tile i of this lane goes (element e of lane l: row = (l/16)*4 + e, column = l%16), its gate
  const int r = lane & 15, q = lane >> 4;
  const int col = n0 + wave * 16 + r;
  const int stages = WHOLE ? NS : g.d / SK;
  float gv[RT][4];
  auto ask_gate = [&]() {
    if (!g.gate) return;
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        int b, t;
        place(min(m0 + i * 16 + q * 4 + e, g.M - 1), b, t);
        gv[i][e] = g.gate[(((long)b * g.h + hh) * g.T + t) * g.N + min(col, g.N - 1)];
      }
  };
  if constexpr (WHOLE) {
    ask_gate();
#pragma unroll
    for (int s = 0; s < NS; ++s) issue(s);
  } else {
    for (int s = 0; s < NS - 1 && s < stages; ++s) issue(s);
    // Behind the first copies, so that their trip to memory runs beside those of the first stages.  The waits below count
    // them as well: the first stage is used when these are there too, not only its own copies.
    ask_gate();
  }
  f32x4 acc[RT];
#pragma unroll
  for (int i = 0; i < RT; ++i) acc[i] = (f32x4)(0.0f);
  // The operands of a stage are read into registers while those of the stage before are multiplied.
  float fa[2][SK / 4][RT], fb[2][SK / 4];
  auto read = [&](int s, int into) {
    const float *sa = s_tiles + s % NS * STAGE, *sb = sa + BM * SK;
#pragma unroll
    for (int c = 0; c < SK / 4; ++c) {
      fb[into][c] = sb[(4 * c + q) * BN + ((wave * 16 + r) ^ (q << 4))];
#pragma unroll
      for (int i = 0; i < RT; ++i) {
        const int row = i * 16 + r;
        fa[into][c][i] = sa[row * SK + (c ^ ((row >> 1) & 7)) * 4 + q];
      }
    }
  };
  auto multiply = [&](int from) {
#pragma unroll
    for (int c = 0; c < SK / 4; ++c)
#pragma unroll
      for (int i = 0; i < RT; ++i)
        acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[from][c][i], fb[from][c], acc[i], 0, 0, 0);
  };
  auto step = [&](int s, int into) {
    const int later = min(NS - 2, stages - 1 - s);
    if (carries_a) bdh_wait_for_stage<2 + CA, NS - 2>(later);
    else bdh_wait_for_stage<2, NS - 2>(later);
    __syncthreads();  // stage s is there for every wave, and stage s - 1 has been read: its place takes stage s + NS - 1
    if (s + NS - 1 < stages) issue((s + NS - 1) % NS);
    read(s, into);
    if (s > 0) multiply(into ^ 1);
  };
  if constexpr (WHOLE) {
    constexpr int GRP = 4;  // stages to a wait and a barrier
    static_assert(NS % GRP == 0, "whole groups, the last stage's operands in the second set");
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      if (s % GRP == 0) {  // the next GRP stages are there for every wave
        if (carries_a) bdh_wait_for_stage<2 + CA, NS - GRP>(NS - GRP - s);
        else bdh_wait_for_stage<2, NS - GRP>(NS - GRP - s);
        __syncthreads();
      }
      read(s, s & 1);
      __builtin_amdgcn_sched_barrier(0);  // left alone, the scheduler sinks these reads to their use
      if (s > 0) multiply((s & 1) ^ 1);
    }
    multiply(1);
  } else {
    for (int s = 0; s < stages; s += 2) {  // two at a time: the registers have fixed names
      step(s, 0);
      if (s + 1 < stages) step(s + 1, 1);
    }
    if (stages & 1) multiply(0);
    else multiply(1);
  }
  if (col >= g.N) return;
  const float bv = g.bias ? g.bias[(long)hh * g.N + col] : 0.0f;
  float mk = 1.0f;
  if (g.mask) {
    const int blk = col / g.block;
    mk = (blk < g.n_blocks && g.mask[blk]) ? 1.0f : 0.0f;
  }
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int m = m0 + i * 16 + q * 4 + e;
      float pv = acc[i][e];
      if (g.bias) pv = pv + bv;
      if (g.thr != 0.0f) pv = pv - g.thr;
      float y = pv > 0.0f ? pv : 0.0f;
      if (g.mask) y = y * mk;
      if (g.gate) y = gv[i][e] * y;
      int b, t;
      place(m, b, t);
      if (m < g.M) g.C[(((long)b * g.h + hh) * g.T + t) * g.N + col] = y;
    }
}

// any d and N: 64 x 64 tiles staged through registers, with checks
__global__ __launch_bounds__(256) void k_relu_lowrank_gemm(RlArgs g) {
  constexpr int BM = 64, BN = 64;
  using Tl = RlTile<BM, BN, 2, 2>;
  __shared__ __attribute__((aligned(16))) float s_a[BM * FLD];
  __shared__ __attribute__((aligned(16))) float s_b[FK * (BN + 32)];
  Tl t;
  if (!t.init(g)) return;
  const int tid = threadIdx.x, lane = t.lane;
  const float *W = g.W + (long)t.hh * g.d * g.N;
  const int K = g.d;
  const float *pa = t.a_row(g, t.m0 + (tid >> 2));
  const int kb = tid >> 4, nc = (tid & 15) * 4;
  f32x16 acc[1][1];
#pragma unroll
  for (int e = 0; e < 16; ++e) acc[0][0][e] = 0.0f;
  float ra[4], rb[4];
  auto load = [&](int k0) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int k = k0 + (tid & 3) * 4 + u;
      ra[u] = k < K ? pa[k] : 0.0f;
      rb[u] = k0 + kb < K ? W[(long)(k0 + kb) * g.N + min(t.n0 + nc + u, g.N - 1)] : 0.0f;
    }
  };
  load(0);
  for (int k0 = 0; k0 < K; k0 += FK) {
    __syncthreads();  // the previous step's fragment reads are done
    // k = kc, kc + 2 to places kc / 2, kc / 2 + 1 of a row; k = kc + 1, kc + 3 to places 8 + kc / 2, ...: the two
    // 16-byte reads below then give a half-wave k = 2 q + half
    float *sa = s_a + (tid >> 2) * FLD + (tid & 3) * 2;
    sa[0] = ra[0]; sa[1] = ra[2]; sa[8] = ra[1]; sa[9] = ra[3];
    *reinterpret_cast<float4 *>(s_b + kb * (BN + 32) + nc) = make_float4(rb[0], rb[1], rb[2], rb[3]);
    __syncthreads();
    if (k0 + FK < K) load(k0 + FK);
    const int r = lane & 31, half = lane >> 5;
    const float *p = s_a + (t.wm * 32 + r) * FLD + half * 8;
    const float *q = s_b + half * (BN + 32) + t.wn * 32 + r;
#pragma unroll
    for (int u = 0; u < 8; ++u)
      acc[0][0] = __builtin_amdgcn_mfma_f32_32x32x2f32(p[u], q[2 * u * (BN + 32)], acc[0][0], 0, 0, 0);
  }
  t.finish(g, acc);
}

// the scores product and, when its K is cut into parts, their reduction
int launch_scores(bdh_ctx *ctx, const GemmF32 &g, const GemmPlan &plan, float *parts) {
  const int rc = bdh_launch_gemm_f32(ctx, g, false, false, plan, parts);
  if (rc != BDH_OK || plan.ks == 1) return rc;
  GemmF32 r = g;
  r.ks = plan.ks;
  r.block_shift = g.block_size > 0 && (g.block_size & (g.block_size - 1)) == 0 ? __builtin_ctz(g.block_size) : -1;
  hipLaunchKernelGGL(k_scores_reduce, dim3((unsigned)((long)g.n_slices * g.M)), dim3(256), 0, ctx->stream, parts,
                     (long)g.n_slices * g.M * g.N, r);
  BDH_LAUNCH_CHECK(ctx, "k_scores_reduce");
  return BDH_OK;
}

}  // namespace

extern "C" int bdh_fused_state_aligned(bdh_ctx *ctx, int B, int h, int T, int N, int dv, const float *query,
                                       const float *value, const float *freqs, const float *alibi_slopes_host,
                                       int block_size, const int32_t *block_pairs_host, int n_pairs, int rotary,
                                       int row_normalize, float *out) {
  if (!ctx) return BDH_E_INVAL;
  if (B < 0 || h < 0 || T < 0 || N < 0 || dv < 0) return bdh_fail(ctx, BDH_E_INVAL, "negative dimension");
  if (rotary != BDH_ROPE && rotary != BDH_ALIBI && rotary != BDH_POPE)
    return bdh_fail(ctx, BDH_E_INVAL, "rotary %d is not a bdh_rotary value", rotary);
  if (rotary == BDH_ROPE && (N & 1)) return bdh_fail(ctx, BDH_E_SHAPE, "RoPE needs an even latent size, got N=%d", N);
  if (h > 64) return bdh_fail(ctx, BDH_E_SHAPE, "n_head %d > 64", h);
  if (n_pairs < 0 || (n_pairs > 0 && !block_pairs_host)) return bdh_fail(ctx, BDH_E_INVAL, "bad block pair list");
  if (B == 0 || h == 0 || T == 0 || dv == 0) return BDH_OK;
  if (!query || !value || !out || (rotary != BDH_ALIBI && !freqs)) return bdh_fail(ctx, BDH_E_INVAL, "null data pointer");
  if (block_size < 1) block_size = 1;  // usize::max(layout.block_size(), 1), linear_attention.rs:46
  const int Nq = rotary == BDH_POPE ? 2 * N : N;
  const long S = (long)B * h;
  const int tb = (T + block_size - 1) / block_size;
  const bool sparse = block_pairs_host != nullptr;
  if (sparse && tb > 4096) return bdh_fail(ctx, BDH_E_SHAPE, "sparse time pattern with %d blocks", tb);
  // opt-in: the dense layout, row-normalised, on the bf16 matrix cores (inputs and scores rounded to bf16: 2e-2)
  if (ctx->opt_fsa_path == 2 && !sparse && row_normalize && (N & 7) == 0 && bdh_aligned(query, 16) && bdh_aligned(out, 16))
    return bdh_launch_fsa_bf16(ctx, B, h, T, N, dv, query, value, freqs, alibi_slopes_host, block_size, rotary, out);
  const size_t lds = sizeof(float) * ((size_t)Nq + T);
  int path = ctx->opt_fsa_path == 2 ? -1 : ctx->opt_fsa_path;  // -1 choose, 0 row kernel, 1 matrix cores
  if (path < 0) path = T >= 128 ? 1 : 0;
  if (path == 0 && lds > 150 * 1024) path = 1;
  if (S * T > 0x7fffffffL || (S + 7) / 8 * 8 * (long)(((T + 127) / 128) * ((T + 127) / 128)) > 0x7fffffffL) return bdh_fail(ctx, BDH_E_SHAPE, "B*h*T too large");

  const int Tp = (T + 3) & ~3;  // row stride of the score matrix
  FsaSlopes slopes_dev{};
  if (alibi_slopes_host) memcpy(slopes_dev.v, alibi_slopes_host, sizeof(float) * h);
  // the two products of the matrix-core path: S = mask(Q Q^T) + bias, then (S V) / (sum |S| + eps)
  GemmF32 g, o;
  GemmPlan plan_g, plan_o;
  size_t part_bytes = 0;
  if (path == 1) {
    g.epilogue = GEMM_SCORES;
    g.a_s1 = g.b_s1 = (long)T * Nq; g.c_s1 = (long)T * Tp;
    g.lda = g.ldb = Nq; g.ldc = Tp; g.M = g.N = T; g.K = Nq; g.n_slices = (int)S; g.heads = h;
    g.block_size = block_size; g.tb = tb; g.use_alibi = alibi_slopes_host != nullptr;
    memcpy(g.slopes, slopes_dev.v, sizeof(g.slopes));
    g.sparse_pattern = sparse;
    o.epilogue = row_normalize ? GEMM_NORM : GEMM_STORE;
    o.mod = h;
    o.a_s1 = (long)h * T * Tp; o.a_s2 = (long)T * Tp; o.b_s1 = (long)T * dv; o.c_s1 = (long)h * T * dv; o.c_s2 = (long)T * dv;
    o.lda = Tp; o.ldb = dv; o.ldc = dv; o.M = T; o.N = dv; o.K = T; o.n_slices = (int)S; o.heads = h;
    o.block_size = block_size; o.causal_k = !sparse;
    plan_o = bdh_gemm_f32_plan(ctx, o, 1);
    g.reader_rows = bdh_gemm_f32_rows(plan_o);
    const size_t one = sizeof(float) * (size_t)S * T * T;
    plan_g = bdh_gemm_f32_plan(ctx, g, (int)std::min<size_t>(16, (size_t(256) << 20) / one));
    if (plan_g.ks > 1) part_bytes = bdh_align_up(one * plan_g.ks, 256);
  }
  const size_t q_bytes = rotary == BDH_ALIBI ? 0 : bdh_align_up(sizeof(float) * (size_t)S * T * Nq, 256);
  const size_t sc_bytes = path == 1 ? bdh_align_up(sizeof(float) * (size_t)S * T * Tp, 256) : 0;
  int rc = bdh_ws_reserve(ctx, q_bytes + sc_bytes + part_bytes);
  if (rc != BDH_OK) return rc;
  char *ws = static_cast<char *>(ctx->ws);
  float *rotated = reinterpret_cast<float *>(ws);
  float *scores = reinterpret_cast<float *>(ws + q_bytes);
  float *parts = reinterpret_cast<float *>(ws + q_bytes + sc_bytes);
  // The time-block mask of a sparse pattern lives in memory the context owns and is uploaded only when the
  // pattern differs from the one already there (a model calls with the same pattern every time): no copy and
  // no host synchronisation on the usual call.  The ALiBi slopes travel as a kernel argument.
  unsigned char *active = nullptr;
  if (sparse) {
    std::vector<int> key;
    key.reserve(2 * (size_t)n_pairs + 1);
    key.push_back(tb);
    key.insert(key.end(), block_pairs_host, block_pairs_host + 2 * (size_t)n_pairs);
    if (!ctx->fsa_mask || ctx->fsa_mask_key != key) {
      std::vector<unsigned char> m((size_t)tb * tb, 0);
      for (int p = 0; p < n_pairs; ++p) {
        const int r = block_pairs_host[2 * p], c = block_pairs_host[2 * p + 1];
        if (r >= 0 && r < tb && c >= 0 && c < tb) m[(size_t)r * tb + c] = 1;  // iter_cols drops c >= total_blocks
      }
      BDH_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));  // earlier calls may still read the old mask
      if (ctx->fsa_mask_bytes < m.size()) {
        if (ctx->fsa_mask) BDH_HIP_CHECK(ctx, hipFree(ctx->fsa_mask));
        ctx->fsa_mask = nullptr;
        ctx->fsa_mask_bytes = 0;
        ctx->fsa_mask_key.clear();
        if (hipMalloc(&ctx->fsa_mask, m.size()) != hipSuccess) {
          (void)hipGetLastError();
          return bdh_fail(ctx, BDH_E_NOMEM, "time-block mask of %zu bytes", m.size());
        }
        ctx->fsa_mask_bytes = m.size();
      }
      BDH_HIP_CHECK(ctx, hipMemcpy(ctx->fsa_mask, m.data(), m.size(), hipMemcpyHostToDevice));
      ctx->fsa_mask_key = std::move(key);
    }
    active = static_cast<unsigned char *>(ctx->fsa_mask);
  }
  const float *q = query;  // ALiBi does not rotate
  if (rotary != BDH_ALIBI) {
    hipLaunchKernelGGL(k_rotate_f32, dim3((unsigned)(S * T)), dim3(256), 0, ctx->stream, query, freqs, rotated, T, N, rotary);
    BDH_LAUNCH_CHECK(ctx, "k_rotate_f32");
    q = rotated;
  }
  if (path == 1) {
    g.A = g.B = q; g.C = scores; g.active = active;
    rc = launch_scores(ctx, g, plan_g, parts);
    if (rc != BDH_OK) return rc;
    o.A = scores; o.B = value; o.C = out;
    return bdh_launch_gemm_f32(ctx, o, false, true, plan_o, nullptr);
  }
  hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(k_fsa_row),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e != hipSuccess) {
    (void)hipGetLastError();
    return bdh_fail(ctx, BDH_E_HIP, "dynamic LDS of %zu bytes refused: %s", lds, hipGetErrorString(e));
  }
  hipLaunchKernelGGL(k_fsa_row, dim3((unsigned)(S * T)), dim3(256), lds, ctx->stream, q, value, slopes_dev,
                     alibi_slopes_host ? 1 : 0, h, T, Nq, dv, block_size, active, tb, row_normalize, out);
  BDH_LAUNCH_CHECK(ctx, "k_fsa_row");
  return BDH_OK;
}

// ------------------------------------------------------------------------------------
// BDH::recurrent_attention (src/model/bdh.rs:258-307) over many tokens at once, f32, RoPE or PoPE:
// for a chunk of Tc tokens  out = tril(-1)(Q Q^T) V + Q rho,  rho += Q^T V  — the same sums as the
// token-by-token loop, reassociated, as four products on the f32 matrix cores.  The cost does not
// depend on how many neurons are active, which is what a prompt through a densely firing model needs
// (the sparse step kernels move every touched state row once per token).
// ------------------------------------------------------------------------------------
int bdh_launch_state_chunks_f32(bdh_ctx *ctx, const StateStepParams &p, float *out_ln) {
  const int B = p.B, h = p.h, T = p.T, N = p.N, d = p.d;
  const int Nq = p.rotary == BDH_POPE ? 2 * N : N;
  const long S = (long)B * h;
  const bool bf16_state = p.rho_dtype == BDH_BF16;
  const bool alibi = p.rotary == BDH_ALIBI;
  if (p.stamps && !alibi) return bdh_fail(ctx, BDH_E_INVAL, "decay stamps only apply to ALiBi");
  float log_decay[64] = {0};
  if (alibi)
    for (int i = 0; i < h; ++i) log_decay[i] = bdh_log_decay(p.slopes_host[i]);
  if (S > 0x7fffffffL / 4096) return bdh_fail(ctx, BDH_E_SHAPE, "B*h too large");
  // chunk length: a multiple of 128 between 128 and 512 whose rotated activations stay under 4 GiB
  const size_t per_token = sizeof(float) * (size_t)S * Nq;
  long Tc = (long)((size_t(4) << 30) / per_token) / 128 * 128;
  Tc = std::min<long>(512, std::max<long>(128, Tc));
  Tc = std::min<long>(Tc, T);
  const int Tcp = ((int)Tc + 3) & ~3;
  if (S * Tc > 0x7fffffffL) return bdh_fail(ctx, BDH_E_SHAPE, "B*h*T too large");
  // the products of a chunk of tc tokens; what differs from chunk to chunk is filled in below
  auto with_decay = [&](GemmF32 &g) {
    g.heads = h;
    if (alibi) memcpy(g.log_decay, log_decay, sizeof(g.log_decay));
  };
  struct Chunk {
    GemmF32 scores, out, state;
    GemmPlan p_scores, p_out, p_state;
    size_t parts_bytes = 0;
  };
  auto chunk_of = [&](int tc, long q_batch) {
    Chunk c;
    GemmF32 &g = c.scores;  // S = tril(-1)(Q Q^T)   (ALiBi: S[t,s] *= decay^(t-s))
    g.epilogue = GEMM_SCORES;
    g.a_s1 = g.b_s1 = q_batch; g.c_s1 = (long)Tc * Tcp;
    g.lda = g.ldb = Nq; g.ldc = Tcp; g.M = g.N = tc; g.K = Nq; g.n_slices = (int)S;
    with_decay(g);
    g.decay_scores = alibi;
    // out = Q rho + S V   (the state before this chunk; S limited to the causal prefix of each row tile; ALiBi: the
    // first term's row t *= decay^t)
    GemmF32 &o = c.out;
    o.mod = h;
    o.a_s1 = h * q_batch; o.a_s2 = q_batch; o.b_s1 = (long)h * Nq * d; o.b_s2 = (long)Nq * d;
    o.c_s1 = (long)h * T * d; o.c_s2 = (long)T * d;
    o.lda = Nq; o.ldb = d; o.ldc = d; o.M = tc; o.N = d; o.K = Nq; o.n_slices = (int)S;
    o.a2_s1 = (long)h * Tc * Tcp; o.a2_s2 = (long)Tc * Tcp; o.b2_s1 = (long)T * d; o.lda2 = Tcp; o.ldb2 = d; o.K2 = tc;
    o.causal_k = true;
    with_decay(o);
    o.decay_rows = alibi;
    // rho += Q^T V   (both operands k-major: the reduction runs over the tokens; ALiBi: rho = decay^tc rho +
    // sum_s decay^(tc-s) q_s (x) v_s)
    GemmF32 &r = c.state;
    r.mod = h;
    r.a_s1 = h * q_batch; r.a_s2 = q_batch; r.b_s1 = (long)T * d; r.c_s1 = (long)h * Nq * d; r.c_s2 = (long)Nq * d;
    r.lda = Nq; r.ldb = d; r.ldc = d; r.M = Nq; r.N = d; r.K = tc; r.n_slices = (int)S;
    r.accumulate = true;
    with_decay(r);
    r.decay_state = alibi;
    const size_t most = size_t(256) << 20;
    const size_t one_s = sizeof(float) * (size_t)S * tc * tc, one_o = sizeof(float) * (size_t)S * tc * d;
    c.p_out = bdh_gemm_f32_plan(ctx, o, (int)std::min<size_t>(32, std::max<size_t>(1, most / one_o)));
    g.reader_rows = bdh_gemm_f32_rows(c.p_out);
    c.p_scores = bdh_gemm_f32_plan(ctx, g, (int)std::min<size_t>(32, std::max<size_t>(1, most / one_s)));
    c.p_state = bdh_gemm_f32_plan(ctx, r, 1);
    // the parts of the scores are used up before those of the readout are written
    c.parts_bytes = std::max(c.p_scores.ks > 1 ? one_s * c.p_scores.ks : 0, c.p_out.ks > 1 ? one_o * c.p_out.ks : 0);
    return c;
  };
  const int tc_last = T % Tc ? T % (int)Tc : (int)Tc;
  const size_t parts_bytes = bdh_align_up(std::max(chunk_of((int)Tc, 0).parts_bytes, chunk_of(tc_last, 0).parts_bytes), 256);
  const size_t q_bytes = alibi ? 0 : bdh_align_up(per_token * (size_t)Tc, 256);  // ALiBi does not rotate: q = x
  const size_t sc_bytes = bdh_align_up(sizeof(float) * (size_t)S * Tc * Tcp, 256);
  // a bf16 state is widened to f32 for the call and rounded back once at its end (the token loop rounds
  // after every token)
  const size_t n_state = (size_t)S * Nq * d;
  const size_t wide_bytes = bf16_state ? bdh_align_up(sizeof(float) * n_state, 256) : 0;
  int rc = bdh_ws_reserve(ctx, q_bytes + sc_bytes + parts_bytes + wide_bytes);
  if (rc != BDH_OK) return rc;
  if (p.stamps) {  // a lazily decayed state: apply what is pending, the products below decay every row themselves
    int rc0 = bdh_launch_alibi_materialize(ctx, B, h, N, d, p.slopes_host, p.position, p.positions_dev, p.rho,
                                           p.rho_dtype, p.stamps);
    if (rc0 != BDH_OK) return rc0;
  }
  char *ws = static_cast<char *>(ctx->ws);
  float *q = reinterpret_cast<float *>(ws);
  float *scores = reinterpret_cast<float *>(ws + q_bytes);
  float *parts = reinterpret_cast<float *>(ws + q_bytes + sc_bytes);
  float *rho = static_cast<float *>(p.rho);
  if (bf16_state) {
    rho = reinterpret_cast<float *>(ws + q_bytes + sc_bytes + parts_bytes);
    hipLaunchKernelGGL(k_widen_bf16, dim3((unsigned)std::min<size_t>((n_state + 255) / 256, 1u << 20)), dim3(256), 0,
                       ctx->stream, static_cast<const unsigned short *>(p.rho), rho, n_state);
    BDH_LAUNCH_CHECK(ctx, "k_widen_bf16");
  }
  bool normed = false;
  for (int t0 = 0; t0 < T; t0 += (int)Tc) {
    const int tc = (int)std::min<long>(Tc, T - t0);
    const float *qc = q;           // this chunk's rotated activations [S][tc][Nq]
    long q_batch = (long)tc * Nq;
    if (alibi) {
      qc = p.x + (long)t0 * N;
      q_batch = (long)T * N;
    } else {
      hipLaunchKernelGGL(k_rotate_chunk_f32, dim3((unsigned)(S * tc)), dim3(256), 0, ctx->stream, p.x + (long)t0 * N,
                         (long)T * N, p.freqs, q, tc, N, p.rotary, (long)(p.position + t0), p.positions_dev, t0, h);
      BDH_LAUNCH_CHECK(ctx, "k_rotate_chunk_f32");
    }
    Chunk c = chunk_of(tc, q_batch);
    c.scores.A = c.scores.B = qc; c.scores.C = scores;
    rc = launch_scores(ctx, c.scores, c.p_scores, parts);
    if (rc != BDH_OK) return rc;
    c.out.A = qc; c.out.B = rho; c.out.A2 = scores; c.out.B2 = p.v + (long)t0 * d; c.out.C = p.out + (long)t0 * d;
    rc = bdh_launch_gemm_f32(ctx, c.out, false, true, c.p_out, parts);
    if (rc != BDH_OK) return rc;
    if (c.p_out.ks > 1) {
      const long rows = S * tc;
      auto *kernel = d <= 256 ? k_rows_reduce<4, 8> : d <= 512 ? k_rows_reduce<8, 4> : k_rows_reduce<16, 2>;
      hipLaunchKernelGGL(kernel, dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, ctx->stream, parts, c.p_out.ks,
                         rows * d, tc, d, rows, p.out + (long)t0 * d, out_ln ? out_ln + (long)t0 * d : nullptr, (long)T * d);
      BDH_LAUNCH_CHECK(ctx, "k_rows_reduce");
      normed = tc == T;
    }
    c.state.A = qc; c.state.B = p.v + (long)t0 * d; c.state.C = rho;
    rc = bdh_launch_gemm_f32(ctx, c.state, true, true, c.p_state, nullptr);
    if (rc != BDH_OK) return rc;
  }
  if (bf16_state) {
    hipLaunchKernelGGL(k_narrow_bf16, dim3((unsigned)std::min<size_t>((n_state + 255) / 256, 1u << 20)), dim3(256), 0,
                       ctx->stream, rho, static_cast<unsigned short *>(p.rho), n_state);
    BDH_LAUNCH_CHECK(ctx, "k_narrow_bf16");
  }
  if (p.stamps) {  // every row is now up to date as of the end of the call
    const long rows = S * N;
    hipLaunchKernelGGL(k_set_stamps, dim3((unsigned)((rows + 255) / 256)), dim3(256), 0, ctx->stream, p.stamps, rows,
                       (long)h * N, (long)(p.position + T), p.positions_dev, T);
    BDH_LAUNCH_CHECK(ctx, "k_set_stamps");
  }
  if (out_ln && !normed) return bdh_launch_layer_norm_rows(ctx, (int64_t)S * T, d, p.out, out_ln);
  return BDH_OK;
}

// The encoder E over the rows of prompts (src/model/bdh.rs:383,436-438): mixed [B*T, h*N] . decoder [h*N, d] as one product
// per head, K cut into as many parts as the chip wants.
// partial [*rows_out][B*T][d] receives the terms of every output row; the caller sums them in order.
int bdh_launch_decoder_partials_f32(bdh_ctx *ctx, int B, int T, int h, int N, int d, const float *xy, const float *decoder,
                                    int *rows_out) {
  GemmF32 g;
  g.A = xy; g.B = decoder;
  g.lda = N; g.ldb = d; g.ldc = d; g.M = B * T; g.N = d;
  g.K = N; g.n_slices = h; g.mod = h;
  g.a_s2 = (long)T * N; g.b_s2 = (long)N * d; g.c_s2 = (long)B * T * d;
  g.rows_per = T; g.a_outer = (long)h * T * N;
  g.c_outer = (long)T * d;
  const size_t one = sizeof(float) * (size_t)g.n_slices * g.M * d;
  const GemmPlan plan = bdh_gemm_f32_plan(ctx, g, (int)std::min<size_t>(64, std::max<size_t>(1, (size_t(256) << 20) / one)));
  int rc = bdh_ws_reserve(ctx, one * plan.ks);
  if (rc != BDH_OK) return rc;
  g.C = static_cast<float *>(ctx->ws);
  *rows_out = g.n_slices * plan.ks;
  return bdh_launch_gemm_f32(ctx, g, false, true, plan, g.C);
}

// D_y of a prompt: gate * relu(in . W - thr) as split-bf16 products, a slice per head.
static GemmF32 gated_product(const ReluLowrankParams &p) {
  GemmF32 g;
  g.epilogue = GEMM_GATE;
  g.A = p.in; g.B = p.weight; g.C = p.out; g.gate = p.gate;
  g.threshold = p.threshold;
  g.M = p.B * p.T; g.N = p.N; g.K = p.d;
  g.lda = p.d; g.ldb = g.ldc = p.N;
  g.n_slices = g.mod = p.h;
  g.a_s2 = p.h_in == 1 ? 0 : (long)p.T * p.d; g.b_s2 = (long)p.d * p.N; g.c_s2 = (long)p.T * p.N;
  g.rows_per = p.T; g.a_outer = (long)p.h_in * p.T * p.d; g.c_outer = (long)p.h * p.T * p.N;
  return g;
}

// Whether they are faster than the f32 chain.  From three 128 x 128 tiles for every two CUs on (us a prompt, 4 layers, chain | split:
// 4 x 8192 neurons, d = 256, 200 rows 1083 | 1042, 1500 rows 4969 | 4739; 8 x 256, d = 512, 1500 rows (192 tiles) 1041 | 1030,
// 4088 rows 2281 | 2184; 4 x 256, d = 256, 4088 rows (256 tiles) 843 | 850; 4 x 2048, d = 128, 4088 rows 2620 | 2540), but
//  - few rows are bound by the weights, which the 16 and 32 row tiles of the chain stream (us, chain | split: 4 x 12288, d = 128, 1
//    row 5.8 | 11.3, 16 rows 7.8 | 11.8, 32 rows 11.7 | 12.3, 33 rows 17.3 | 13.4; d = 384, 16 rows 14.2 | 21.9, 32 rows 20.2 | 22.2,
//    33 rows 31.9 | 25.9; 4 x 16384, d = 256, 16 rows 14.2 | 17.8, 17 rows 19.1 | 17.7, 32 rows 20.5 | 18.3; 4 x 12288, d = 64,
//    32 rows 9.1 | 14.8; without 16-byte pieces, d = 260, 4 x 12289, 8 rows 24.3 | 25.5, 16 rows 29.5 | 25.7);
//  - rows that end in the first half of a 128 row tile have less padding in the chain's 64 x 64 tiles.  Those take 1.3 us and 0.73
//    for every 32 of K, a CU one after the other; two 128 x 128 tiles on a CU 12.4 and 2.95, one by itself 8.8 and 2.2 (us, 129 | 193
//    rows: 4 x 12288, d = 128 chain 38 | 51, split 42 | 43; 4 x 8192, d = 128 27 | 34, 25 | 26; 257 rows: 4 x 6144, d = 192 44.2, 46.6).
bool bdh_relu_lowrank_split_pays(const bdh_ctx *ctx, const ReluLowrankParams &p) {
  const long n_cu = ctx->n_cu > 0 ? ctx->n_cu : 256, M = (long)p.B * p.T;
  auto tiles = [&](int side) { return p.h * ((M + side - 1) / side) * ((p.N + side - 1) / side); };
  const long big = tiles(128);
  if (2 * big < 3 * n_cu) return false;
  const bool pieces = p.d % 32 == 0 && p.N % 4 == 0 && bdh_aligned(p.in, 16) && bdh_aligned(p.weight, 16);
  if (M <= (pieces ? 16 : 8)) return false;
  if (!pieces) return true;
  if (M <= 32) return p.d >= 128 && big >= 2 * n_cu;
  if (big >= 4 * n_cu || bdh_gemm_f32_rows(bdh_gemm_f32_plan(ctx, gated_product(p), 1)) != 128) return true;
  const double stages = p.d / 32, per_cu = (double)tiles(64) / n_cu;
  const long rest = big % (2 * n_cu);
  const double two = 12.4 + 2.95 * stages, one = 8.8 + 2.2 * stages;
  return big / (2 * n_cu) * two + (rest > n_cu ? two : rest > 0 ? one : 0.0) <= per_cu * (1.3 + 0.73 * stages);
}

int bdh_launch_relu_lowrank_split(bdh_ctx *ctx, const ReluLowrankParams &p) {
  const GemmF32 g = gated_product(p);
  return bdh_launch_gemm_f32(ctx, g, false, true, bdh_gemm_f32_plan(ctx, g, 1), nullptr);
}

extern "C" int bdh_rotate(bdh_ctx *ctx, int B, int h, int T, int N, int rotary, const float *x, const float *freqs,
                          int64_t position, const int32_t *positions_dev, float *q) {
  if (!ctx) return BDH_E_INVAL;
  if (B < 0 || h < 0 || T < 0 || N < 0) return bdh_fail(ctx, BDH_E_INVAL, "negative dimension");
  if (rotary != BDH_ROPE && rotary != BDH_ALIBI && rotary != BDH_POPE)
    return bdh_fail(ctx, BDH_E_INVAL, "rotary %d is not a bdh_rotary value", rotary);
  if (position < 0) return bdh_fail(ctx, BDH_E_INVAL, "negative position");
  if (rotary == BDH_ROPE && (N & 1)) return bdh_fail(ctx, BDH_E_SHAPE, "RoPE needs an even latent size, got N=%d", N);
  const long rows = (long)B * h * T;
  if (rows == 0 || N == 0) return BDH_OK;
  if (!x || !q || (rotary != BDH_ALIBI && !freqs)) return bdh_fail(ctx, BDH_E_INVAL, "null data pointer");
  if (!bdh_aligned(x, 8) || !bdh_aligned(q, 8) || !bdh_aligned(freqs, 8))
    return bdh_fail(ctx, BDH_E_ALIGN, "x, q and freqs need 8-byte alignment");
  if (rows > 0x7fffffffL) return bdh_fail(ctx, BDH_E_SHAPE, "B*h*T too large");
  if (rotary == BDH_ALIBI) {  // Attention::rotate returns its input (src/model/attention.rs:333-335)
    if (q != x)
      BDH_HIP_CHECK(ctx, hipMemcpyAsync(q, x, sizeof(float) * (size_t)rows * N, hipMemcpyDeviceToDevice, ctx->stream));
    return BDH_OK;
  }
  hipLaunchKernelGGL(k_rotate_chunk_f32, dim3((unsigned)rows), dim3(256), 0, ctx->stream, x, (long)T * N, freqs, q, T, N,
                     rotary, (long)position, positions_dev, 0, h);
  BDH_LAUNCH_CHECK(ctx, "k_rotate_chunk_f32");
  return BDH_OK;
}

// relu_lowrank for many rows on the f32 matrix cores with the k order of a scalar loop, so the outputs are the bits of
// k_relu_lowrank.  mask_dev: one byte per latent block in device memory, or null.
int bdh_launch_relu_lowrank_gemm(bdh_ctx *ctx, const ReluLowrankParams &p, const unsigned char *mask_dev) {
  RlArgs g{};
  g.A = p.in;
  g.W = p.weight;
  g.C = p.out;
  g.T = p.T;
  g.a_outer = (long)p.h_in * p.T * p.d;
  g.a_head = p.h_in == 1 ? 0 : (long)p.T * p.d;
  g.M = p.B * p.T;
  g.N = p.N;
  g.d = p.d;
  g.h = p.h;
  g.bias = p.bias;
  g.thr = p.threshold;
  g.mask = mask_dev;
  g.block = p.block_size > 0 ? p.block_size : 1;
  g.n_blocks = p.n_blocks;
  g.gate = p.gate;
  const long n_cu = ctx->n_cu > 0 ? ctx->n_cu : 256;
  auto tiles = [&](int bm, int bn) {
    g.mt = (g.M + bm - 1) / bm;
    g.nt = (g.N + bn - 1) / bn;
    return (long)g.h * g.mt * g.nt;
  };
  // Narrow tiles (16 rows) while there are no more than four for every CU: the latency of one tile is what counts.  Beyond
  // that up to 32 and 64 rows in one tile, so that the weights pass once; more rows 64 x 64, and 128 x 128 once there are
  // four of those for every CU (us, 16-row | 32-row | 64-row | 64 x 64 tiles: [128 x 256] x [256 x 4096] 7.7 | 8.4 | 12.2 |
  // 10.2, [256 x ..] 11.3 | 10.9 | 12.8 | 11.0, [512 x ..] 18.1 | 17.0 | 17.3 | 16.2; [32 x 512] x [512 x 131072] 67 | 59 | 85 |
  // 153, [63 x ..] 118 | 100 | 94 | 157; 128 x 128 | 64 x 64: [1536 x 256] x [256 x 32768] 253 | 273, [512 x 512] x
  // [512 x 20480] 111 | 104)
  const bool direct = p.d % 32 == 0 && p.N % 4 == 0 && bdh_aligned(p.in, 16) && bdh_aligned(p.weight, 16);
  const bool big = direct && tiles(128, 128) >= 4 * n_cu;
  const int rt = !direct ? 0 : g.M <= 16 || tiles(16, 64) <= 4 * n_cu ? 1 : g.M <= 32 ? 2 : g.M <= 64 ? 4 : 0;
  const long total = rt ? tiles(16 * rt, 64) : big ? tiles(128, 128) : tiles(64, 64);
  if (total + 8 > 0x7fffffffL) return bdh_fail(ctx, BDH_E_SHAPE, "too many tiles");
  const dim3 grid((unsigned)(8 * ((total + 7) / 8)));
#define BDH_RLD(KERNEL_, ROWS_, COLS_) \
  hipLaunchKernelGGL((KERNEL_), grid, dim3(256), 2 * (ROWS_ + COLS_) * 32 * sizeof(float), ctx->stream, g)
  // Stages of the ring: more copies in flight where the workgroups are too few to cover each other's trips, fewer where LDS
  // decides how many of them a CU holds (us, two | four stages: 96 workgroups 9.3 | 8.3, 256 6.8 | 6.1, 1024 13.8 | 15.0); all of
  // them where the 10 KiB a stage leave a CU its share of the workgroups: one with d = 512, two with d = 256.
#define BDH_RLR(RT_, NS_, WHOLE_) hipLaunchKernelGGL((k_relu_lowrank_rows<RT_, NS_, WHOLE_>), grid, dim3(256), 0, ctx->stream, g)
  if (rt == 1 && total <= n_cu && g.d == 512) BDH_RLR(1, 16, true);
  else if (rt == 1 && total <= 2 * n_cu && g.d == 256) BDH_RLR(1, 8, true);
  else if (rt == 1 && total <= 2 * n_cu) BDH_RLR(1, 4, false);
  else if (rt == 1) BDH_RLR(1, 2, false);
  else if (rt == 2) BDH_RLR(2, 3, false);
  else if (rt == 4) BDH_RLR(4, 2, false);
#undef BDH_RLR
  else if (big) BDH_RLD((k_relu_lowrank_direct<128, 128>), 128, 128);
  else if (direct) BDH_RLD((k_relu_lowrank_direct<64, 64>), 64, 64);
  else hipLaunchKernelGGL(k_relu_lowrank_gemm, grid, dim3(256), 0, ctx->stream, g);
#undef BDH_RLD
  BDH_LAUNCH_CHECK(ctx, "k_relu_lowrank_gemm");
  return BDH_OK;
}
