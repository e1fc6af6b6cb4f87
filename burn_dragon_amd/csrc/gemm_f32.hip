// Dense f32 products on the bf16 matrix cores (see gemm_f32.h).
//
// Every f32 operand is taken as a sum of three bf16 terms h + m + l and a product as six bf16 matrix instructions, so
// the results carry f32-level accuracy at a sixth of the bf16 rate (417 TFLOP/s against 157 of the f32 instruction).
// The split is made once per element and workgroup, on the way into LDS: a stage holds 32 k of both tiles as three bf16
// planes, chunks of eight k of one row (16 bytes) being what a lane feeds to one 32 x 32 x 16 instruction.
// The five smaller products have accumulators of their own: the large sum is then rounded once per 16 k and not six times
// (2-norm distance from float64 of the row-normalised attention of 200 tokens, N = 256: 2.7e-7 -> 1.1e-7; of a prompt of 64
// tokens, N = 256: readout 2.1e-7 -> 0.9e-7, state 1.1e-7 -> 0.6e-7).  They cost 64 registers at 128 x 128, two workgroups
// per CU instead of three there: 0.6 to 1.7 % of the prompts and of scoring.
#include "gemm_f32.h"

#include "tile_index.h"

#include <algorithm>
#include <cfloat>

namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

constexpr float kRowNormEps = 1e-6f;  // src/kernel/linear_attention.rs:9
constexpr int FK = 32;                // k per LDS stage

// Eight floats as three bf16x8 operands h + m + l that add up to the floats exactly: each term is the remainder so far
// rounded to bf16 (v_cvt_pk_bf16_f32, round to nearest even); a remainder is a difference of neighbours and therefore
// exact, and the third one has at most eight significant bits.  A product of two such sums is taken as the six matrix
// instructions l h, h l, m m, m h, h m, h h (smallest terms first); what is left out (m l, l m, l l) is below 2^-23 of
// |a b|, the size of one f32 rounding.  An infinite input, or a finite one that rounds to an infinite bf16 (above
// 3.389e38), gives NaN (inf - inf in the remainder).
__device__ __forceinline__ void split3(const float (&a)[8], u32x4 &ph, u32x4 &pm, u32x4 &pl) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
#pragma unroll
  for (int q = 0; q < 4; ++q) {  // element 2q in the low half of a dword, 2q + 1 in the high half
    const f32x2 a2 = {a[2 * q], a[2 * q + 1]};
    ph[q] = __builtin_bit_cast(unsigned int, __builtin_convertvector(a2, bf16x2));
    const f32x2 r1 = {a2[0] - __uint_as_float(ph[q] << 16), a2[1] - __uint_as_float(ph[q] & 0xffff0000u)};
    pm[q] = __builtin_bit_cast(unsigned int, __builtin_convertvector(r1, bf16x2));
    const f32x2 r2 = {r1[0] - __uint_as_float(pm[q] << 16), r1[1] - __uint_as_float(pm[q] & 0xffff0000u)};
    pl[q] = __builtin_bit_cast(unsigned int, __builtin_convertvector(r2, bf16x2));
  }
}

// Byte offset of chunk c (eight k) of row r inside a plane: rows are 64 bytes, and the four chunks of a row are rotated
// so that eight lanes reading one chunk column of consecutive rows, or writing it to every second row, take eight
// different 16-byte columns of the 64 banks.
__device__ __forceinline__ int chunk_at(int r, int c) { return r * 64 + ((c ^ ((r >> 2) & 3)) << 4); }

// One operand's tile of R rows (or columns) x 32 k, on its way from memory to LDS.  A thread carries CH chunks of eight
// k.  Row-major: four lanes cover the 128 bytes of a row's stage.  k-major: a thread owns CH adjacent rows and eight
// consecutive k, so the transposition happens in its registers and a wavefront reads whole pieces of a k row.
enum { IN, TAIL, CHECKED };
template <int R, int NT, bool KM>
struct Tile {
  static constexpr int CH = R * 4 / NT > 0 ? R * 4 / NT : 1;
  static constexpr int USED = R * 4 / CH;  // threads that carry something
  float v[CH][8];
  const float *p[CH];
  int k_off, row[CH];

  __device__ __forceinline__ void init(const float *base, int ld, int r0, int rows, int rows_per, long outer) {
    const int tid = threadIdx.x;
    if (USED < NT && tid >= USED) return;
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      if (!KM) {
        row[c] = (c * USED + tid) >> 2;
        const int r = min(r0 + row[c], rows - 1);  // a row past the end repeats the last one; its sums are not stored
        p[c] = base + (rows_per > 0 ? (long)(r / rows_per) * outer + (long)(r % rows_per) * ld : (long)r * ld);
      } else {
        row[c] = (tid % (R / CH)) * CH + c;
        p[c] = base + bdh_kmajor_row(r0, row[0], c, CH, rows);
      }
    }
    k_off = KM ? (tid / (R / CH)) * 8 : (tid & 3) * 8;
  }
  // IN: the stage lies inside K and the accesses are aligned.  TAIL: aligned accesses, clamped into the operand, with what
  // lies beyond K set to zero.  CHECKED: one element at a time.
  template <int MODE>
  __device__ __forceinline__ void load(int k0, int K, int ld) {
    if (USED < NT && (int)threadIdx.x >= USED) return;
    const int k = k0 + k_off;
    if constexpr (MODE == CHECKED) {
#pragma unroll
      for (int c = 0; c < CH; ++c)
#pragma unroll
        for (int q = 0; q < 8; ++q) v[c][q] = k + q < K ? (KM ? p[c][(long)(k + q) * ld] : p[c][k + q]) : 0.0f;
      return;
    }
    if constexpr (!KM) {
      const int last = (K - 1) & ~3;  // the last aligned piece that holds something
      const int k_lo = MODE == TAIL ? min(k, last) : k, k_hi = MODE == TAIL ? min(k + 4, last) : k + 4;
#pragma unroll
      for (int c = 0; c < CH; ++c) {
        const float4 lo = *reinterpret_cast<const float4 *>(p[c] + k_lo), hi = *reinterpret_cast<const float4 *>(p[c] + k_hi);
        v[c][0] = lo.x; v[c][1] = lo.y; v[c][2] = lo.z; v[c][3] = lo.w;
        v[c][4] = hi.x; v[c][5] = hi.y; v[c][6] = hi.z; v[c][7] = hi.w;
      }
    } else {
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const long at = (long)(MODE == TAIL ? min(k + q, K - 1) : k + q) * ld;
        if constexpr (CH == 2) {
          const float2 t = *reinterpret_cast<const float2 *>(p[0] + at);
          v[0][q] = t.x;
          v[1][q] = t.y;
        } else {
#pragma unroll
          for (int c = 0; c < CH; ++c) v[c][q] = p[c][at];
        }
      }
    }
    if constexpr (MODE == TAIL) {
#pragma unroll
      for (int c = 0; c < CH; ++c)
#pragma unroll
        for (int q = 0; q < 8; ++q) v[c][q] = k + q < K ? v[c][q] : 0.0f;
    }
  }
  // planes of R * 64 bytes each
  __device__ __forceinline__ void store(unsigned char *s) const {
    if (USED < NT && (int)threadIdx.x >= USED) return;
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      u32x4 h, m, l;
      split3(v[c], h, m, l);
      unsigned char *q = s + chunk_at(row[c], k_off >> 3);
      *reinterpret_cast<u32x4 *>(q) = h;
      *reinterpret_cast<u32x4 *>(q + R * 64) = m;
      *reinterpret_cast<u32x4 *>(q + 2 * R * 64) = l;
    }
  }
};

// What a scores product stores for the sum v of (row, col), col < g.N.
__device__ __forceinline__ float score_value(const GemmF32 &g, float v, int row, int col, float ld, float slope) {
  const int rb = bdh_time_block(g, row), cb = bdh_time_block(g, col);
  if (!(g.active ? g.active[(long)rb * g.tb + cb] != 0 : cb <= rb)) return 0.0f;
  if (rb == cb && col >= row) v = 0.0f;  // tril(-1) on diagonal blocks (:88-90)
  if (g.decay_scores && col < row) v = v * expf((float)(row - col) * ld);
  if (g.use_alibi) {  // added to every entry of an active block (:97-100)
    const float al = slope * ((float)col - (float)row);
    v = v + al;
  }
  return v;
}

// The tile of this workgroup.  XCD-aware mapping: workgroup ids are dealt round-robin to the 8 XCDs, so ids with the same
// (id % 8) share an L2.  Each XCD takes one contiguous eighth of the (slice, part of K, tile) list: neighbouring tiles reuse
// their operand rows in one L2, and every XCD has the same number of tiles whatever the number of slices.
struct TileAt {
  int part, slice, ti, tj;
  __device__ __forceinline__ bool find(const GemmF32 &g) {
    // (the launcher keeps the total within an int; 64-bit divisions are a hundred instructions each)
    const unsigned int tiles = g.tri ? g.mt * (g.mt + 1) / 2 : g.mt * g.nt, total = (unsigned int)g.n_slices * g.ks * tiles;
    const unsigned int xcd = blockIdx.x & 7, lo = (total >> 3) * xcd + ((total & 7) * xcd >> 3);
    const unsigned int hi = (total >> 3) * (xcd + 1) + ((total & 7) * (xcd + 1) >> 3), at = lo + (blockIdx.x >> 3);
    if (at >= hi) return false;
    const unsigned int whole = at / tiles;
    int tile = (int)(at - whole * tiles);
    slice = g.ks == 1 ? (int)whole : (int)(whole / (unsigned int)g.ks);
    part = (int)whole - slice * g.ks;
    // A CU often gets the same tile of several slices: after a long row tile a short one (32 slices of [511 x 511] x [511 x
    // 256], row tiles of 2 to 16 stages: 38 -> 30 us).
    if (g.causal_k && (slice & 1)) tile = (int)tiles - 1 - tile;
    if (g.tri) {  // lower triangle of square tiles, row by row
      ti = (int)((sqrtf(8.0f * (float)tile + 1.0f) - 1.0f) * 0.5f);
      while ((ti + 1) * (ti + 2) / 2 <= tile) ++ti;
      while (ti * (ti + 1) / 2 > tile) --ti;
      tj = tile - ti * (ti + 1) / 2;
    } else {
      ti = tile / g.nt;
      tj = tile - ti * g.nt;
    }
    return true;
  }
};

// Where row m of C begins.  The place of the first of 32 neighbouring rows is worked out once, the others follow from it: a
// division only where they run into the next sequence.
struct RowPlaces {
  int first, b0, t0;
  __device__ __forceinline__ RowPlaces(const GemmF32 &g, int first_row) : first(first_row) {
    b0 = g.rows_per > 0 ? first_row / g.rows_per : 0;
    t0 = g.rows_per > 0 ? first_row - b0 * g.rows_per : 0;
  }
  __device__ __forceinline__ long at(const GemmF32 &g, int off) const {
    if (g.rows_per <= 0) return (long)(first + off) * g.ldc;
    int b = b0, t = t0 + off;
    if (t >= g.rows_per) {
      b += t / g.rows_per;
      t %= g.rows_per;
    }
    return (long)b * g.c_outer + (long)t * g.ldc;
  }
};

// What a gated projection stores for the sum v: a NaN counts as not above the threshold, as in every other projection.
__device__ __forceinline__ float gated(const GemmF32 &g, float v, float gate) {
  v -= g.threshold;
  return gate * (v > 0.0f ? v : 0.0f);
}

// ROWS x COLS sums of A . B as one k-sequential fused multiply-add chain each, as the projections that have no split compute
// them.  Where an operand is infinite, a NaN or rounds to an infinite bf16, or a sum leaves the floats, the terms' sum is no
// number (inf - inf in a remainder, split3) and never a wrong finite one: a projection is then made again in this way.
template <int ROWS, int COLS>
__device__ __forceinline__ void chains(const float *const (&a)[ROWS], const float *const (&b)[COLS], int ldb, int K,
                                       float (&s)[ROWS][COLS]) {
#pragma unroll
  for (int r = 0; r < ROWS; ++r)
#pragma unroll
    for (int c = 0; c < COLS; ++c) s[r][c] = 0.0f;
#pragma unroll 4
  for (int k = 0; k < K; ++k)
#pragma unroll
    for (int r = 0; r < ROWS; ++r)
#pragma unroll
      for (int c = 0; c < COLS; ++c) s[r][c] = __builtin_fmaf(a[r][k], b[c][(long)k * ldb], s[r][c]);
}
__device__ __forceinline__ const float *row_of_a(const GemmF32 &g, const float *A, int row) {
  return A + (g.rows_per > 0 ? (long)(row / g.rows_per) * g.a_outer + (long)(row % g.rows_per) * g.lda : (long)row * g.lda);
}

// The ends of K for a tile of rows [m0, m0 + bm) and columns from n0 on: of A . B and of A2 . B2.
__device__ __forceinline__ void ends_of_k(const GemmF32 &g, bool scores, int m0, int bm, int n0, int &K1, int &K2) {
  const int bs = g.block_size, last = min(m0 + bm, g.M) - 1, k_causal = (last / bs + 1) * bs;
  K1 = g.K;
  K2 = g.A2 ? g.K2 : 0;
  if (g.causal_k) {
    if (g.A2) K2 = min(K2, k_causal);
    else K1 = min(K1, k_causal);
  }
  // a scores tile above the diagonal of the block pattern only writes zeros
  if (scores && !g.active && n0 / bs > last / bs) K1 = 0;
}

// BM x BN tile per workgroup of WM x WN wavefronts.  With four wavefronts LDS holds one stage (192 bytes per tile row and column: 48 KiB at
// 128 x 128; the registers allow two workgroups per CU); the next stage's loads are in flight in registers while this one is multiplied,
// and the other workgroups of the CU fill the two barriers.  What bounds it: at 128 x 128 a wavefront spends 1536 cycles
// of a stage in matrix instructions, 700 in the split and the LDS pipe moves 144 KiB.
// Eight wavefronts (TURNS): two stages in LDS, two on every SIMD (wavefronts w and w + 4).  Between two barriers one of the
// two multiplies the stage that is there and then splits the next one into the other buffer, its partner does the two in the
// other order: the conversions of one run under the matrix instructions of the other.
template <int BM, int BN, int WM, int WN, bool AK, bool BK, int EPI>
__global__ __launch_bounds__(WM * WN * 64, 2) void k_gemm_f32(GemmF32 g) {
  constexpr bool TURNS = WM * WN == 8;
  constexpr int NT = WM * WN * 64;
  constexpr int MI = BM / WM / 32, NJ = BN / WN / 32;
  __shared__ __attribute__((aligned(16))) unsigned char s_a[(TURNS ? 2 : 1) * 3 * BM * 64];
  __shared__ __attribute__((aligned(16))) unsigned char s_b[(TURNS ? 2 : 1) * 3 * BN * 64];
  __shared__ float s_norm[EPI == GEMM_NORM ? BM : 1];
  TileAt here;
  if (!here.find(g)) return;
  const int part = here.part, slice = here.slice;
  const int m0 = here.ti * BM, n0 = here.tj * BN;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN;
  const long s1 = slice / g.mod, s2 = slice % g.mod;
  const float *A = g.A + s1 * g.a_s1 + s2 * g.a_s2;
  const float *B = g.B + s1 * g.b_s1 + s2 * g.b_s2;
  float *C = g.C + s1 * g.c_s1 + s2 * g.c_s2;
  const float ld = (g.decay_rows || g.decay_state || g.decay_scores) ? g.log_decay[slice % g.heads] : 0.0f;

  // the k blocks of this part: first those of A . B, then those of A2 . B2
  int K1, K2;
  ends_of_k(g, EPI == GEMM_SCORES, m0, BM, n0, K1, K2);
  const int nb1 = (K1 + FK - 1) / FK, nb = nb1 + (K2 + FK - 1) / FK;
  const int b_lo = part * g.kb_per, b_hi = min(nb, b_lo + g.kb_per);

  f32x16 acc[MI][NJ], low[MI][NJ];  // the sums of h h, and of the five smaller terms
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = low[i][j][e] = 0.0f;

  Tile<BM, NT, AK> ta;
  Tile<BN, NT, BK> tb;
  float rs[Tile<BM, NT, AK>::CH];
#pragma unroll
  for (int c = 0; c < Tile<BM, NT, AK>::CH; ++c) rs[c] = 0.0f;

  auto run = [&](const float *pa, int lda, int rows_per, long a_outer, const float *pb, int ldb, int K, int lo, int hi) {
    ta.init(pa, lda, m0, g.M, rows_per, a_outer);
    tb.init(pb, ldb, n0, g.N, 0, 0);
    // 16-byte pieces of a row, or (k-major) pairs of a k row, which end inside it (bdh_kmajor_row)
    const bool a_ok = AK ? ((lda & 1) == 0 && (g.M & 1) == 0 && (reinterpret_cast<uintptr_t>(pa) & 7) == 0)
                         : ((lda & 3) == 0 && (a_outer & 3) == 0 && K <= lda && (reinterpret_cast<uintptr_t>(pa) & 15) == 0);
    const bool b_ok = BK ? ((ldb & 1) == 0 && (g.N & 1) == 0 && (reinterpret_cast<uintptr_t>(pb) & 7) == 0)
                         : ((ldb & 3) == 0 && K <= ldb && (reinterpret_cast<uintptr_t>(pb) & 15) == 0);
    auto scaled = [&](int kb) {
      if (AK && EPI == GEMM_STORE && g.decay_state) {  // token k of K is decayed K - k times by the end
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          // (beyond K, where the operand is zero: 1, for the power of a steep decay would be infinite there)
          const float f = expf((float)max(K - (kb * FK + ta.k_off + q), 0) * ld);
#pragma unroll
          for (int c = 0; c < Tile<BM, NT, AK>::CH; ++c) ta.v[c][q] *= f;
        }
      }
      if (EPI == GEMM_NORM) {
#pragma unroll
        for (int c = 0; c < Tile<BM, NT, AK>::CH; ++c)
#pragma unroll
          for (int q = 0; q < 8; ++q) rs[c] += fabsf(ta.v[c][q]);
      }
    };
    auto multiply = [&](int buf) {
      const unsigned char *sa = s_a + buf * 3 * BM * 64, *sb = s_b + buf * 3 * BN * 64;
      // lane (r = lane % 32, half = lane / 32) feeds chunk 2 * step + half of its row
      const int r = lane & 31, half = lane >> 5;
#pragma unroll
      for (int step = 0; step < 2; ++step) {
        if (TURNS) __builtin_amdgcn_sched_barrier(0);  // one step's fragments at a time
        bf16x8 fa[3][MI], fb[3][NJ];
#pragma unroll
        for (int t = 0; t < 3; ++t) {
#pragma unroll
          for (int i = 0; i < MI; ++i)
            fa[t][i] = *reinterpret_cast<const bf16x8 *>(sa + t * BM * 64 + chunk_at(wm * (BM / WM) + i * 32 + r, 2 * step + half));
#pragma unroll
          for (int j = 0; j < NJ; ++j)
            fb[t][j] = *reinterpret_cast<const bf16x8 *>(sb + t * BN * 64 + chunk_at(wn * (BN / WN) + j * 32 + r, 2 * step + half));
        }
        constexpr int TA[6] = {2, 0, 1, 1, 0, 0}, TB[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
        for (int t = 0; t < 6; ++t)
#pragma unroll
          for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
              f32x16 &sum = t == 5 ? acc[i][j] : low[i][j];
              sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[TA[t]][i], fb[TB[t]][j], sum, 0, 0, 0);
            }
      }
    };
    if (a_ok && b_ok) {
      // from the last stage, the one that K may cut short, down: every load inside the loop then lies inside K, and the
      // loop is straight-line code (with a branch among them, loads are waited for where they are issued)
      ta.template load<TAIL>((hi - 1) * FK, K, lda);
      tb.template load<TAIL>((hi - 1) * FK, K, ldb);
      auto put = [&](int kb, int buf) {
        scaled(kb);
        ta.store(s_a + buf * 3 * BM * 64);
        tb.store(s_b + buf * 3 * BN * 64);
      };
      auto ask = [&](int kb) {
        ta.template load<IN>(kb * FK, K, lda);
        tb.template load<IN>(kb * FK, K, ldb);
      };
      if constexpr (TURNS) {
        __syncthreads();  // the fragment reads of an earlier pair of operands are done
        put(hi - 1, 0);
        if (hi - 1 > lo) ask(hi - 2);
        __syncthreads();
        int buf = 0;
        const bool first_half = wave < 4;
        for (int kb = hi - 1; kb > lo; --kb, buf ^= 1) {  // stage kb is in LDS, stage kb - 1 in registers or on its way there
          // the last of these asks for stage lo once more: what comes is not used
          if (!first_half) {
            put(kb - 1, buf ^ 1);
            ask(max(kb - 2, lo));
          }
          __builtin_amdgcn_sched_barrier(0);
          multiply(buf);
          __builtin_amdgcn_sched_barrier(0);
          if (first_half) {
            put(kb - 1, buf ^ 1);
            ask(max(kb - 2, lo));
          }
          __syncthreads();
        }
        multiply(buf);
      } else {
        for (int kb = hi - 1; kb > lo; --kb) {
          __syncthreads();  // the previous stage's fragment reads are done
          put(kb, 0);
          __syncthreads();
          ask(kb - 1);
          __builtin_amdgcn_sched_barrier(0);  // left alone, the scheduler sinks the loads behind the products
          multiply(0);
        }
        __syncthreads();
        put(lo, 0);
        __syncthreads();
        multiply(0);
      }
    } else {
      for (int kb = lo; kb < hi; ++kb) {
        ta.template load<CHECKED>(kb * FK, K, lda);
        tb.template load<CHECKED>(kb * FK, K, ldb);
        scaled(kb);
        __syncthreads();
        ta.store(s_a);
        tb.store(s_b);
        __syncthreads();
        multiply(0);
      }
    }
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          acc[i][j][e] += low[i][j][e];
          low[i][j][e] = 0.0f;
        }
  };
  // accumulator element e of lane l in a 32x32 tile: row = (e/4)*8 + (l/32)*4 + (e%4), col = l%32
  auto row_of = [&](int i, int e) { return m0 + wm * (BM / WM) + i * 32 + (e >> 2) * 8 + (lane >> 5) * 4 + (e & 3); };

  if (b_lo < min(b_hi, nb1))
    run(A, g.lda, g.rows_per, g.a_outer, B, g.ldb, K1, b_lo, min(b_hi, nb1));
  if (EPI == GEMM_STORE && g.decay_rows) {
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const float f = expf((float)row_of(i, e) * ld);
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j][e] *= f;
      }
  }
  if constexpr (!AK && BK && EPI == GEMM_STORE) {
    if (g.A2 && max(b_lo, nb1) < b_hi)
      run(g.A2 + s1 * g.a2_s1 + s2 * g.a2_s2, g.lda2, 0, 0, g.B2 + s1 * g.b2_s1 + s2 * g.b2_s2, g.ldb2, K2,
          max(b_lo, nb1) - nb1, b_hi - nb1);
  }

  if (EPI == GEMM_NORM) {  // four threads hold a row's chunks
#pragma unroll
    for (int c = 0; c < Tile<BM, NT, AK>::CH; ++c) {
      float t = rs[c];
      t += __shfl_xor(t, 1);
      t += __shfl_xor(t, 2);
      if ((tid & 3) == 0 && tid < Tile<BM, NT, AK>::USED) s_norm[(c * Tile<BM, NT, AK>::USED + tid) >> 2] = t;
    }
    __syncthreads();
  }
  if (g.ks > 1) {  // a part of the sums: [part][slice][M][N]
    float *P = C + (long)part * g.c_split + (long)slice * g.M * g.N;
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        const int col = n0 + wn * (BN / WN) + j * 32 + (lane & 31);
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int row = row_of(i, e);
          if (row < g.M && col < g.N) P[(long)row * g.N + col] = acc[i][j][e];
        }
      }
    return;
  }
  if (EPI == GEMM_STORE && (g.accumulate || g.decay_state)) {  // C in one piece: the launcher sees to it
    // C = C + acc or g^K C + acc: all of this wave's elements are asked for before the first is used.  (The L2's adder, one
    // no-return add per element, took 215 us where this takes 176: 12 slices of [8192 x 500] x [500 x 256].)
    float old[MI][NJ][16];
    auto place = [&](int i, int j, int e) {  // past the edge: the last row or column again
      return C + (long)min(row_of(i, e), g.M - 1) * g.ldc + min(n0 + wn * (BN / WN) + j * 32 + (lane & 31), g.N - 1);
    };
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) old[i][j][e] = *place(i, j, e);
    const float keep = g.decay_state ? expf((float)g.K * ld) : 1.0f;
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        const bool in = n0 + wn * (BN / WN) + j * 32 + (lane & 31) < g.N;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const float was = g.decay_state ? old[i][j][e] * keep : old[i][j][e];
          if (in && row_of(i, e) < g.M) *place(i, j, e) = was + acc[i][j][e];
        }
      }
    return;
  }
  if constexpr (EPI == GEMM_GATE) {
    const float *G = g.gate + s1 * g.c_s1 + s2 * g.c_s2;
    auto col_of = [&](int j) { return n0 + wn * (BN / WN) + j * 32 + (lane & 31); };
    float zero = 0.0f;  // ... while every sum of this lane is finite
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) zero = __builtin_fmaf(acc[i][j][e], 0.0f, zero);
    if (__any(zero != 0.0f)) {  // rare: all of the wavefront's elements again, eight rows at a time
#pragma unroll 1
      for (int q = 0; q < MI * 4; ++q) {
        const int row0 = row_of(q >> 2, (q & 3) * 4);
        const float *a[4], *b[NJ];
#pragma unroll
        for (int r = 0; r < 4; ++r) a[r] = row_of_a(g, A, min(row0 + r, g.M - 1));
#pragma unroll
        for (int j = 0; j < NJ; ++j) b[j] = B + min(col_of(j), g.N - 1);
        // A row that holds a NaN has sums that are NaN, whatever the weights.  Lanes 0 to 31 have rows row0 + r, the others rows
        // four further on: each half looks through its own.
        bool chain = false;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          bool nan = false;
          for (int k = lane & 31; k < g.K; k += 32) nan |= a[r][k] != a[r][k];
          const unsigned long long found = __ballot(nan);
          chain |= (found & 0xffffffffull) == 0 || (found >> 32) == 0;
        }
        float v[4][NJ];
        if (chain) {
          chains<4, NJ>(a, b, g.ldb, g.K, v);
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int j = 0; j < NJ; ++j) v[r][j] = NAN;
        }
        const int first = min(row0, g.M - 1);
        const RowPlaces places(g, first);
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
          for (int j = 0; j < NJ; ++j) {
            const long at = places.at(g, min(row0 + r, g.M - 1) - first) + col_of(j);
            if (row0 + r < g.M && col_of(j) < g.N) C[at] = gated(g, v[r][j], G[at]);
          }
      }
      return;
    }
    // the gates of a row of tiles are asked for before the first is used
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      long at[16];
      const int first = min(row_of(i, 0), g.M - 1);
      const RowPlaces places(g, first);
#pragma unroll
      for (int e = 0; e < 16; ++e) at[e] = places.at(g, min(row_of(i, e), g.M - 1) - first);
      float gate[NJ][16];
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e)
          gate[j][e] = __builtin_nontemporal_load(G + at[e] + min(col_of(j), g.N - 1));
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        const int col = col_of(j);
#pragma unroll
        for (int e = 0; e < 16; ++e)
          if (col < g.N && row_of(i, e) < g.M) __builtin_nontemporal_store(gated(g, acc[i][j][e], gate[j][e]), C + at[e] + col);
      }
    }
    return;
  }
  const float slope = (EPI == GEMM_SCORES && g.use_alibi) ? g.slopes[slice % g.heads] : 0.0f;
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    const RowPlaces places(g, row_of(i, 0));
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const int col = n0 + wn * (BN / WN) + j * 32 + (lane & 31);
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int row = row_of(i, e);
        if (row >= g.M) continue;
        float v = acc[i][j][e];
        if (EPI == GEMM_SCORES) {
          if (col >= g.ldc) continue;
          v = col < g.N ? score_value(g, v, row, col, ld, slope) : 0.0f;
          C[(long)row * g.ldc + col] = v;
        } else {
          if (col >= g.N) continue;
          if (EPI == GEMM_NORM) v = v / (s_norm[row - m0] + kRowNormEps);
          C[places.at(g, (e >> 2) * 8 + (e & 3)) + col] = v;
        }
      }
    }
  }
}

// 32 x 32 tile per workgroup, for products of few tiles and a short K: the four wavefronts share K, sixteen at a time in turn.
// An element then belongs to one lane, which loads it where it is fed to the matrix instruction, so nothing passes through LDS
// but the wavefronts' sums at the end, and four steps are on their way at a time.  What bounds it: a trip to memory or two and the
// launch; in the tiles above a stage is a chain of loads, conversions, two barriers and dependent products, about 1.2 us long
// when nothing else is on the CU (us, 64 x 64 | this, 4 slices of a prompt of 128 tokens, N = 256, d = 256: scores 14.8 | 7.8,
// readout 13.4 | 7.2, state 10.9 | 6.4, encoder 10.7 | 7.2).
template <bool AK, bool BK, int EPI>
__global__ __launch_bounds__(256, 2) void k_gemm_f32_small(GemmF32 g) {
  constexpr int TS = 32, U = 4;
  __shared__ float s_sum[4][16][64];
  __shared__ float s_norm[EPI == GEMM_NORM ? 4 : 1][TS];
  TileAt here;
  if (!here.find(g)) return;
  const int slice = here.slice, m0 = here.ti * TS, n0 = here.tj * TS;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 31, half = lane >> 5;
  const long s1 = slice / g.mod, s2 = slice % g.mod;
  const float *A = g.A + s1 * g.a_s1 + s2 * g.a_s2;
  const float *B = g.B + s1 * g.b_s1 + s2 * g.b_s2;
  float *C = g.C + s1 * g.c_s1 + s2 * g.c_s2;
  const float ld = (g.decay_rows || g.decay_state || g.decay_scores) ? g.log_decay[slice % g.heads] : 0.0f;
  int K1, K2;
  ends_of_k(g, EPI == GEMM_SCORES, m0, TS, n0, K1, K2);

  f32x16 acc = (f32x16)(0.0f), low = (f32x16)(0.0f);  // the sums of h h, and of the five smaller terms
  float rs = 0.0f;
  auto run = [&](const float *src_a, int lda, int rows_per, long a_outer, const float *src_b, int ldb, int K) {
    const int ar = min(m0 + r, g.M - 1), bc = min(n0 + r, g.N - 1);  // past the end: the last one again, not stored
    const float *pa = src_a + (AK ? (long)ar : rows_per > 0 ? (long)(ar / rows_per) * a_outer + (long)(ar % rows_per) * lda : (long)ar * lda);
    const float *pb = src_b + (BK ? (long)bc : (long)bc * ldb);
    const bool a_ok = (lda & 3) == 0 && (a_outer & 3) == 0 && (reinterpret_cast<uintptr_t>(src_a) & 15) == 0;
    const bool b_ok = (ldb & 3) == 0 && (reinterpret_cast<uintptr_t>(src_b) & 15) == 0;
    float a[U][8], b[U][8];
    auto eight = [&](float(&v)[8], const float *p, bool kmajor, int ld_, bool whole_pieces, int k) {
      if (kmajor) {
#pragma unroll
        for (int q = 0; q < 8; ++q) v[q] = p[(long)(k + q) * ld_];
      } else if (whole_pieces) {
        const float4 lo = *reinterpret_cast<const float4 *>(p + k), hi = *reinterpret_cast<const float4 *>(p + k + 4);
        v[0] = lo.x; v[1] = lo.y; v[2] = lo.z; v[3] = lo.w;
        v[4] = hi.x; v[5] = hi.y; v[6] = hi.z; v[7] = hi.w;
      } else {
#pragma unroll
        for (int q = 0; q < 8; ++q) v[q] = p[k + q];
      }
    };
    auto consume = [&](float(&va)[8], float(&vb)[8], int k) {
      if (AK && EPI == GEMM_STORE && g.decay_state) {  // token k of K is decayed K - k times by the end (beyond K: by 1)
#pragma unroll
        for (int q = 0; q < 8; ++q) va[q] *= expf((float)max(K - (k + q), 0) * ld);
      }
      if (EPI == GEMM_NORM) {
#pragma unroll
        for (int q = 0; q < 8; ++q) rs += fabsf(va[q]);
      }
      u32x4 fa[3], fb[3];
      split3(va, fa[0], fa[1], fa[2]);
      split3(vb, fb[0], fb[1], fb[2]);
      constexpr int TA[6] = {2, 0, 1, 1, 0, 0}, TB[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
      for (int t = 0; t < 6; ++t) {
        f32x16 &sum = t == 5 ? acc : low;
        sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, fa[TA[t]]), __builtin_bit_cast(bf16x8, fb[TB[t]]), sum, 0, 0, 0);
      }
    };
    const int full = K >> 4;  // whole steps of 16
    for (int s = wave; s < full; s += 4 * U) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int k = min(s + 4 * u, full - 1) * 16 + half * 8;  // (past the end: what comes is not used)
        eight(a[u], pa, AK, lda, a_ok, k);
        eight(b[u], pb, BK, ldb, b_ok, k);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (s + 4 * u < full) consume(a[u], b[u], (s + 4 * u) * 16 + half * 8);
    }
    if ((K & 15) && wave == (full & 3)) {  // what K leaves over, zeros beyond
      const int k = full * 16 + half * 8;
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const bool in = k + q < K;
        a[0][q] = in ? (AK ? pa[(long)(k + q) * lda] : pa[k + q]) : 0.0f;
        b[0][q] = in ? (BK ? pb[(long)(k + q) * ldb] : pb[k + q]) : 0.0f;
      }
      consume(a[0], b[0], k);
    }
    acc += low;
    low = (f32x16)(0.0f);
  };
  run(A, g.lda, g.rows_per, g.a_outer, B, g.ldb, K1);
  if (EPI == GEMM_STORE && g.decay_rows) {
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[e] *= expf((float)(m0 + (e >> 2) * 8 + half * 4 + (e & 3)) * ld);
  }
  if constexpr (!AK && BK && EPI == GEMM_STORE) {
    if (K2 > 0)
      run(g.A2 + s1 * g.a2_s1 + s2 * g.a2_s2, g.lda2, 0, 0, g.B2 + s1 * g.b2_s1 + s2 * g.b2_s2, g.ldb2, K2);
  }
#pragma unroll
  for (int e = 0; e < 16; ++e) s_sum[wave][e][lane] = acc[e];
  if (EPI == GEMM_NORM) {
    rs += __shfl_xor(rs, 32);
    if (half == 0) s_norm[wave][r] = rs;
  }
  __syncthreads();
  // wavefront w finishes rows 8 w .. 8 w + 7 of the tile: elements 4 w .. 4 w + 3 of the accumulators, summed in order
  const int col = n0 + r, row0 = m0 + wave * 8 + half * 4;
  const float slope = (EPI == GEMM_SCORES && g.use_alibi) ? g.slopes[slice % g.heads] : 0.0f;
  const bool reads_c = EPI == GEMM_STORE && (g.accumulate || g.decay_state);  // C in one piece: the launcher sees to it
  const float keep = g.decay_state ? expf((float)g.K * ld) : 1.0f;
  const float *G = EPI == GEMM_GATE ? g.gate + s1 * g.c_s1 + s2 * g.c_s2 : nullptr;
  const RowPlaces places(g, row0);
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int row = row0 + e, from = 4 * wave + e;
    if (row >= g.M || col >= (EPI == GEMM_SCORES ? g.ldc : g.N)) continue;
    float v = ((s_sum[0][from][lane] + s_sum[1][from][lane]) + s_sum[2][from][lane]) + s_sum[3][from][lane];
    const long at = places.at(g, e) + col;
    if (EPI == GEMM_SCORES) v = col < g.N ? score_value(g, v, row, col, ld, slope) : 0.0f;
    if (EPI == GEMM_NORM) {
      const int rr = row - m0;
      v = v / ((((s_norm[0][rr] + s_norm[1][rr]) + s_norm[2][rr]) + s_norm[3][rr]) + kRowNormEps);
    }
    if constexpr (EPI == GEMM_GATE) {
      if (!(fabsf(v) <= FLT_MAX)) {
        const float *a[1] = {row_of_a(g, A, row)}, *b[1] = {B + col};
        float again[1][1];
        chains<1, 1>(a, b, g.ldb, g.K, again);
        v = again[0][0];
      }
      v = gated(g, v, G[at]);
    }
    if (reads_c) v = (g.decay_state ? C[at] * keep : C[at]) + v;
    C[at] = v;
  }
}

template <int EPI>
void launch(hipStream_t st, const GemmF32 &g, bool ak, bool bk, int tile, unsigned grid) {
#define BDH_G(BM_, BN_, WM_, WN_, AK_, BK_) \
  hipLaunchKernelGGL((k_gemm_f32<BM_, BN_, WM_, WN_, AK_, BK_, EPI>), dim3(grid), dim3(WM_ * WN_ * 64), 0, st, g)
#define BDH_GT(AK_, BK_)                                     \
  do {                                                       \
    if (tile == 0) BDH_G(128, 128, 2, 2, AK_, BK_);          \
    else if (tile == 1) BDH_G(64, 64, 2, 2, AK_, BK_);       \
    else if (tile == 2) BDH_G(32, 128, 1, 4, AK_, BK_);      \
    else if (tile == 3) BDH_G(128, 256, 2, 4, AK_, BK_);     \
    else hipLaunchKernelGGL((k_gemm_f32_small<AK_, BK_, EPI>), dim3(grid), dim3(256), 0, st, g); \
  } while (0)
  if constexpr (EPI == GEMM_SCORES) {
    BDH_GT(false, false);
  } else if constexpr (EPI == GEMM_NORM || EPI == GEMM_GATE) {
    BDH_GT(false, true);
  } else {
    if (ak) BDH_GT(true, true);
    else BDH_GT(false, true);
  }
#undef BDH_GT
#undef BDH_G
}

constexpr int kTileM[5] = {128, 64, 32, 128, 32}, kTileN[5] = {128, 64, 128, 256, 32};

// scores over causal time blocks that end on tile edges: the tiles above the diagonal hold nothing, and a reader whose
// own row tiles are no larger never looks at them
bool lower_triangle(const GemmF32 &g, int tile) {
  return g.epilogue == GEMM_SCORES && !g.active && !g.sparse_pattern && kTileM[tile] == kTileN[tile] &&
         kTileM[tile] % g.block_size == 0 && kTileM[tile] % g.reader_rows == 0;
}

// The stages of a mean row tile, as a part of those of the last one: where K ends with the tile's last time block.  (32 slices
// of 511 tokens, d = 256: counted in full, 64 x 64 tiles looked no better than one 128 x 128 tile a CU; the readout 45 -> 30 us
// in them, and the scores that it reads, now left out above the diagonal of 64 x 64 tiles, 45 -> 32.)
double causal_share(const GemmF32 &g, int tile_rows) {
  if (!g.causal_k) return 1.0;
  const long all = (g.K + FK - 1) / FK + (g.K2 + FK - 1) / FK;
  long sum = 0, tiles = 0;
  for (int m = 0; m < g.M; m += tile_rows, ++tiles) {
    const int end = ((std::min(m + tile_rows, g.M) - 1) / g.block_size + 1) * g.block_size;
    sum += g.K2 > 0 ? (g.K + FK - 1) / FK + (std::min(g.K2, end) + FK - 1) / FK : (std::min(g.K, end) + FK - 1) / FK;
  }
  return all > 0 ? (double)sum / (double)(all * tiles) : 1.0;
}

}  // namespace

// Which tile and how many parts of K.  A CU that holds a few workgroups turns out a 32-deep stage of a 128 x 128, 64 x 64
// or 32 x 128 tile every `full` cycles; a workgroup alone on its CU takes `alone`, the memory round trip and the two
// barriers uncovered.  The last, partly filled round of workgroups counts like a whole one.  A 128 x 256 tile has its CU to
// itself: a stage takes `turn`, and nothing covers its first loads and its last stores, `turn_end` a tile (12 slices of
// [500 x 8192] x [8192 x 256] in 5 parts: 161 us, in 128 x 128 tiles and 8 parts 185; with a K of 500, [8192 x 500] x [500 x 256],
// 181 against 176; 32 slices of [511 x 511] x [511 x 256] 56 against 46).  More parts of K fill the
// chip where the tiles are few, at the price of writing and re-reading every part.  A 32 x 32 tile (k_gemm_f32_small) has no
// barriers: 750 a stage by itself, 500 where a CU has several, and half of what its last round leaves idle.  Whole calls with it
// over calls without: prompts of 16 to 256 tokens through 4 heads of 128 to 256 neurons 0.69 to 0.87, 8 heads of 256, d = 512,
// 0.76 to 0.92, 4 heads of 1024, 256 tokens 0.91; scoring 128 to 300 tokens 0.67 to 0.96; of 144 calls of 16 to 4088 tokens, up
// to 8192 neurons a head, none is slower by more than its runs differ, up to 2 %.  (With the last round counted as it is filled, 4 slices of [800 x
// 1024] x [1024 x 256], 3.1 rounds, took 28.0 us in 32 x 32 tiles where 64 x 64 tiles in two parts take 21.0 and 2.4 for their
// sum; counted as a whole one, 16 slices of a prompt's readout, 2.6 rounds, left them, and the call went from 446 to 473.)
GemmPlan bdh_gemm_f32_plan(const bdh_ctx *ctx, const GemmF32 &g, int max_split) {
  const double n_cu = ctx->n_cu > 0 ? ctx->n_cu : 256;
  constexpr double full[3] = {2600.0, 900.0, 900.0}, alone[3] = {3600.0, 2000.0, 2000.0};
  constexpr double turn = 3620.0, turn_end = 33000.0;
  const int nb = (g.K + FK - 1) / FK + (g.K2 + FK - 1) / FK;
  GemmPlan best;
  double best_t = 1e300;
  for (int t = 0; t < 5; ++t) {
    if (t == 2 && (g.epilogue == GEMM_SCORES || g.M > 96)) continue;
    const double mt = (g.M + kTileM[t] - 1) / kTileM[t], nt = (g.N + kTileN[t] - 1) / kTileN[t];
    const bool tri = lower_triangle(g, t);
    const double tiles = g.n_slices * (tri ? mt * (mt + 1) / 2 : mt * nt);
    const double share = causal_share(g, kTileM[t]);
    for (int ks = 1; ks <= (t == 4 ? 1 : max_split) && (ks == 1 || nb >= 4 * ks); ks = t == 3 ? ks + 1 : ks * 2) {
      const double per = (nb + ks - 1) / ks, mean = per * share;
      const double wgs = tiles * ks / n_cu;
      const double rounds = wgs <= 1.0 ? 1.0 : wgs;
      double cyc;
      if (t == 4) {
        cyc = std::max(mean * (rounds + std::ceil(rounds)) * 250.0, per * 750.0) + 3000.0;
      } else if (t == 3) {
        cyc = std::ceil(rounds) * (per * turn + turn_end);
      } else {
        cyc = std::max(mean * rounds * full[t], per * alone[t]) + 6000.0;
        if (wgs > 1.0) cyc += mean * full[t] * (std::ceil(wgs) - wgs) * 0.5;
      }
      if (ks > 1) cyc += 8000.0 + (double)g.n_slices * g.M * g.N * 4.0 * 2.0 * ks / 2000.0;  // bytes at about 5 TB/s
      if (cyc < best_t) {
        best_t = cyc;
        best.tile = t;
        best.ks = ks;
      }
    }
  }
  return best;
}

int bdh_gemm_f32_rows(const GemmPlan &plan) { return kTileM[plan.tile]; }

int bdh_launch_gemm_f32(bdh_ctx *ctx, GemmF32 g, bool a_kmajor, bool b_kmajor, const GemmPlan &plan, float *partial) {
  if ((g.accumulate || g.decay_state) && g.rows_per > 0)
    return bdh_fail(ctx, BDH_E_UNSUPPORTED, "a product that is added to what C holds takes C in one piece");
  g.block_shift = g.block_size > 0 && (g.block_size & (g.block_size - 1)) == 0 ? __builtin_ctz(g.block_size) : -1;
  g.mt = (g.M + kTileM[plan.tile] - 1) / kTileM[plan.tile];
  g.nt = (g.N + kTileN[plan.tile] - 1) / kTileN[plan.tile];
  g.tri = lower_triangle(g, plan.tile);
  const int nb = (g.K + FK - 1) / FK + (g.K2 + FK - 1) / FK;
  g.ks = plan.ks;
  g.kb_per = (nb + g.ks - 1) / g.ks;
  if (g.ks > 1) {
    g.C = partial;
    g.c_s1 = g.c_s2 = 0;
    g.c_split = (long)g.n_slices * g.M * g.N;
  }
  const long tiles = g.tri ? (long)g.mt * (g.mt + 1) / 2 : (long)g.mt * g.nt;
  const long total = (long)g.n_slices * g.ks * tiles;
  if (total + 8 > 0x7fffffffL || tiles > 0x7fffffL) return bdh_fail(ctx, BDH_E_SHAPE, "too many tiles");
  if (total == 0) return BDH_OK;
  const unsigned grid = (unsigned)(8 * ((total + 7) / 8));
  switch (g.epilogue) {
    case GEMM_SCORES: launch<GEMM_SCORES>(ctx->stream, g, a_kmajor, b_kmajor, plan.tile, grid); break;
    case GEMM_GATE: launch<GEMM_GATE>(ctx->stream, g, a_kmajor, b_kmajor, plan.tile, grid); break;
    case GEMM_NORM: launch<GEMM_NORM>(ctx->stream, g, a_kmajor, b_kmajor, plan.tile, grid); break;
    default: launch<GEMM_STORE>(ctx->stream, g, a_kmajor, b_kmajor, plan.tile, grid); break;
  }
  BDH_LAUNCH_CHECK(ctx, "k_gemm_f32");
  return BDH_OK;
}
