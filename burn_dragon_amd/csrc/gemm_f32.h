// Dense f32 products on the bf16 matrix cores: argument block and launcher (gemm_f32.hip), shared by the many-token
// forms of the state step, the all-tokens-at-once attention and the encoder E.
#pragma once

#include "bdh_internal.h"

// C[slice] = A[slice] . B[slice], slice = s1 * mod + s2.  Operand X of a slice starts at s1 * x_s1 + s2 * x_s2.
//   A  row-major (k contiguous):  A[m * lda + k];  k-major (a_kmajor): A[k * lda + m]
//   B  row-major (k contiguous):  B[n * ldb + k];  k-major (b_kmajor): B[k * ldb + n]
// Row-major A and C may be pieces of several sequences: row m lies at (m / rows_per) * x_outer + (m % rows_per) * ldx.
// A second pair (A2 row-major, B2 k-major, K2) continues the same sums: C = A . B + A2 . B2.
struct GemmF32 {
  const float *A = nullptr, *B = nullptr;
  float *C = nullptr;
  long a_s1 = 0, a_s2 = 0, b_s1 = 0, b_s2 = 0, c_s1 = 0, c_s2 = 0;
  int lda = 0, ldb = 0, ldc = 0;
  int M = 0, N = 0, K = 0;
  int n_slices = 1, mod = 1;
  int rows_per = 0;  // 0: one piece
  long a_outer = 0, c_outer = 0;
  const float *A2 = nullptr, *B2 = nullptr;
  long a2_s1 = 0, a2_s2 = 0, b2_s1 = 0, b2_s2 = 0;
  int lda2 = 0, ldb2 = 0, K2 = 0;
  // What is done with the sums.
  //   GEMM_STORE   C = acc, or C += acc (accumulate); with decay_rows the A . B part of row t is scaled by g^t; with
  //                decay_state token k of A is scaled by g^(K-k) and C = g^K C + acc.  The two that read C take it in one
  //                piece (rows_per == 0), others are refused.
  //   GEMM_SCORES  square, C zero above the diagonal of the block pattern, see the fields below
  //   GEMM_NORM    C = acc / (sum_k |A[m,k]| + 1e-6)
  //   GEMM_GATE    C = gate * max(acc - threshold, 0), the gate laid out as C
  int epilogue = 0;
  bool accumulate = false;
  bool decay_rows = false, decay_state = false, decay_scores = false;
  const float *gate = nullptr;
  float threshold = 0.0f;
  int heads = 1;              // head of a slice = slice % heads
  float log_decay[64] = {0};  // log g per head
  // scores of causal time blocks of block_size tokens: dense lower triangle of blocks, or the byte mask active[tb*tb];
  // tril(-1) on diagonal blocks, plus slope * (col - row) on every element of an active block
  int block_size = 1, tb = 0;
  int block_shift = -1;  // log2 of a block_size that is a power of two (filled in by the launcher), else -1
  const unsigned char *active = nullptr;
  bool use_alibi = false;
  float slopes[64] = {0};
  bool sparse_pattern = false;  // a byte mask will be given (for the plan)
  int reader_rows = 128;        // scores: the rows per tile of the product that reads them (it reads whole tiles)
  // k of the A . B sums (of A2 . B2 when there is a second pair) ends with the row tile's last time block: A is zero
  // beyond it and is not read there
  bool causal_k = false;
  // filled in by the launcher
  int mt = 0, nt = 0, ks = 1, kb_per = 0, tri = 0;
  long c_split = 0;
};
#if defined(__HIPCC__)
// The time block of token t >= 0.  (A division by a run-time number is some thirty instructions, and an epilogue asks for every
// element: 32 slices of [511 x 256] x [256 x 511] in 64 x 64 tiles 33.4 us with it, 29.6 with the shift.)
__device__ __forceinline__ int bdh_time_block(const GemmF32 &g, int t) {
  return g.block_shift >= 0 ? t >> g.block_shift : t / g.block_size;
}
#endif
constexpr int GEMM_STORE = 0, GEMM_SCORES = 1, GEMM_NORM = 2, GEMM_GATE = 3;

// How a product is cut: tile (0: 128 x 128, 1: 64 x 64, 2: 32 x 128, 3: 128 x 256, 4: 32 x 32 with K dealt to the wavefronts)
// and the number of parts of K.
struct GemmPlan {
  int tile = 0, ks = 1;
};
// max_split: the most parts of K the caller has room for (a part's sums are [n_slices][M][N] floats).
GemmPlan bdh_gemm_f32_plan(const bdh_ctx *ctx, const GemmF32 &g, int max_split);
int bdh_gemm_f32_rows(const GemmPlan &plan);  // rows of a tile
// partial: room for plan.ks parts of [n_slices][M][N] floats when plan.ks > 1 (C is then not written: the caller adds
// the parts up, in order); a scores product writes its parts without mask and decay.
int bdh_launch_gemm_f32(bdh_ctx *ctx, GemmF32 g, bool a_kmajor, bool b_kmajor, const GemmPlan &plan, float *partial);
