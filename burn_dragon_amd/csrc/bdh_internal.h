// Internal declarations shared by the translation units of libbdh_mi355x.so.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdarg>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <vector>

#include "../../include/bdh_mi355x.h"

struct bdh_ctx {
  int device = 0;
  hipStream_t stream = nullptr;
  // growable device workspace (partials, counters); owned by the context
  void *ws = nullptr;
  size_t ws_bytes = 0;
  // a second growable buffer for inputs a launcher converts before it calls a path that sizes ctx->ws itself
  void *stage = nullptr;
  size_t stage_bytes = 0;
  int n_cu = 0;
  int opt_step_split = -1;  // -1 choose by grid size, 0 / 1 force the 256- / 64-pair workgroup
  int opt_step_dense = -1;  // many-token state step as dense f32 products: -1 by dense_form_from, 0 never, 1 always
  int opt_decoder_mfma = 1;  // 0: the encoder E never takes the f32 matrix-core form
  int opt_model_one_launch = 1;  // small model's decode step in one launch: 1 when it pays, 2 whenever it fits, 0 never
  int opt_lowrank_row = 1;     // 0: relu_lowrank with one input row and a small matrix uses the column-per-thread kernel
  int opt_model_phase_batch = 1 << 30;  // two launches per layer for a decode step of at most this many sequences (0: never)
  int opt_lowrank_split = -1;  // D_y of a prompt on split-bf16 products: -1 by size, 0 / 1 never / always
  int opt_lowrank_gemm_rows = 64;  // relu_lowrank of 64 rows and more takes the f32 matrix cores from this many on (0: never)
  int opt_lowrank_mfma_rows = 2;  // relu_lowrank of fewer than 64 rows takes the f32 matrix cores from this many on (0: never)
  int opt_step_past_caches = -1;  // -1: by what passes between two visits of a row; 0 / 1: never / always
  int opt_step_dense_kernel = 1;  // 0: PoPE / eager ALiBi at d in {256,512} take the generic kernel
  int opt_decoder_splitk_rows = 24;  // decode-step encoder on the matrix cores from this many sequences on
  int opt_ws_max_mib = 0;   // the workspace never grows beyond this (0: no limit)
  int opt_fsa_path = -1;    // fused_state_aligned: -1 choose by T, 0 row kernel, 1 f32 matrix cores
  int opt_model_fused_rows = 1;  // 0: a one-sequence decode step never folds its reductions into the projections
  int opt_model_fused_kb = 256;  // rows of E per workgroup of the encoder's first stage in that form
  int opt_step_prompt_bf16 = 0;  // many-token state step on the bf16 matrix cores from this many tokens on (0: never)
  // time-block mask of the last sparse fused_state_aligned pattern (device) and the pattern it was built from
  void *fsa_mask = nullptr;
  size_t fsa_mask_bytes = 0;
  std::vector<int> fsa_mask_key;
  // latent block mask of the last relu_lowrank call that had one (device) and the bytes it was built from
  void *lat_mask = nullptr;
  size_t lat_mask_bytes = 0;
  std::vector<uint8_t> lat_mask_key;
  char err[512] = {0};
};

struct bdh_model {
  bdh_ctx *ctx = nullptr;
  bdh_model_config cfg{};
  bdh_model_weights w{};
  float *freqs = nullptr;   // device [N]
  float slopes[64] = {0};   // host, ALiBi only
  // activation scratch, grown on demand to the largest (B,T) seen
  void *act = nullptr;
  size_t act_bytes = 0;
  // scratch of the two-launch layer of a model that fits the one-launch step, at most 4 MiB of projection weights; sized at
  // creation for every batch that form is taken for: a decode step of such a model never allocates, and a captured one keeps
  // its buffer whatever runs later.  One buffer a model: its steps follow one another, captured ones too.
  float *phase_act = nullptr;
};

int bdh_fail(bdh_ctx *ctx, int status, const char *fmt, ...);

// model_phase.hip: a decode step in two launches per layer (T = 1, 128 <= d <= 512, N a multiple of 32)
bool bdh_model_phase_fits(const bdh_model *m);
bool bdh_model_phase_pays(const bdh_model *m, int B, int rho_dtype, bool lazy);
size_t bdh_model_phase_scratch_floats(const bdh_model *m, int B);
int bdh_launch_model_phases(bdh_model *m, const int64_t *tokens, int B, float *scratch, void *rho, int rho_dtype, int32_t *stamps,
                            int64_t position,
                            const int32_t *positions_dev, float **cur_final, float **dec_partial, int *G_out);
int bdh_launch_phase_head(bdh_model *m, int B, const float *cur, const float *dec_partial, int G, float *logits,
                          int64_t *next_tokens);
// projections.hip: cur[m,:] = LN(cur[m,:] + LN(sum_kb partial[kb][m][:]))
int bdh_launch_decoder_finalize(bdh_ctx *ctx, const float *partial, int KBN, int M, int d, float *cur);

// model_small.hip: the one-launch decode step of a small model (T = 1, f32 state)
bool bdh_model_small_fits(const bdh_model_config &c);
int bdh_model_one_launch_from(const bdh_model_config &c);  // sequences; 0: never
int bdh_launch_model_small(bdh_model *m, const int64_t *tokens, int B, void *rho, int rho_dtype, int32_t *stamps, int64_t position,
                           const int32_t *positions_dev, float *logits, int64_t *next_tokens);

// Grows ctx->ws to at least `bytes` (synchronises the stream before freeing the old one).
int bdh_ws_reserve(bdh_ctx *ctx, size_t bytes);
// The same for ctx->stage.
int bdh_stage_reserve(bdh_ctx *ctx, size_t bytes);

#define BDH_HIP_CHECK(ctx, call)                                                        \
  do {                                                                                  \
    hipError_t e_ = (call);                                                             \
    if (e_ != hipSuccess)                                                               \
      return bdh_fail((ctx), BDH_E_HIP, "%s failed: %s (%s:%d)", #call,                 \
                      hipGetErrorString(e_), __FILE__, __LINE__);                       \
  } while (0)

#define BDH_LAUNCH_CHECK(ctx, what)                                                     \
  do {                                                                                  \
    hipError_t e_ = hipGetLastError();                                                  \
    if (e_ != hipSuccess)                                                               \
      return bdh_fail((ctx), BDH_E_HIP, "launch of %s failed: %s", (what),              \
                      hipGetErrorString(e_));                                           \
  } while (0)

static inline size_t bdh_align_up(size_t v, size_t a) { return (v + a - 1) / a * a; }

// The log of the ROUNDED per-token decay factor expf(-slope) (src/model/attention.rs:181-186), for the forms that need powers
// of it.  Finite: a factor that rounds to zero (slopes above 103) still has the zeroth power 1, and 0 * -inf would be NaN.
static inline float bdh_log_decay(float slope) {
  const double l = log((double)expf(-slope));
  return l < -1e4 ? -1e4f : (float)l;
}
static inline bool bdh_aligned(const void *p, size_t a) {
  return (reinterpret_cast<uintptr_t>(p) % a) == 0;
}

// ---- launchers implemented in the kernel translation units --------------------------
struct StateStepParams {
  int B, h, T, N, d, rotary, rho_dtype;
  const float *x, *v, *freqs;
  int64_t position;
  const int32_t *positions_dev;
  const float *slopes_host;  // resolved (never null for ALiBi)
  void *rho;
  float *out;
  uint64_t *bitmask;
  int32_t *rows_touched;
  int32_t *stamps = nullptr;  // ALiBi only: [B,h,N] decay stamps of a lazily decayed state, or null
  // T = 1 on the RoPE kernels (d in {256, 512}) only: leave the readout as the per-workgroup partial sums
  // [B*h][S][d] in the context's workspace (the caller's next kernel adds them up): no second stage, `out` unused
  struct StepPartials *partials_out = nullptr;
  // bytes of all the states and weights that the caller's step walks before it comes back to this state; 0: not known
  size_t walked = 0;
};
struct StepPartials {
  const float *partial = nullptr;
  int S = 0;
};
int bdh_launch_state_steps(bdh_ctx *ctx, const StateStepParams &p);

// Variant used inside the fused model step: the readout is LayerNorm-ed on the fly
// (src/model/bdh.rs:359) when out_ln != nullptr.
int bdh_launch_state_steps_ln(bdh_ctx *ctx, const StateStepParams &p, float *out_ln);
// The same with the partials in a caller-given buffer (nothing is allocated; fails when they do not fit).
int bdh_launch_state_steps_in(bdh_ctx *ctx, const StateStepParams &p, float *out_ln, void *fixed, size_t fixed_bytes);
// The fixed scratch array of the allocation-free decode step: resolve its address on the context's device
// (that device must be current), read it back, and its size.
int bdh_step_scratch_resolve(bdh_ctx *ctx);
void *bdh_step_scratch_ptr(const bdh_ctx *ctx);
size_t bdh_step_scratch_bytes();
// The same T steps as four dense products per chunk on the f32 matrix cores (attention_parallel.hip):
// RoPE / PoPE, f32 state, no bitmask or row counts.
int bdh_launch_state_chunks_f32(bdh_ctx *ctx, const StateStepParams &p, float *out_ln);
// prefill.hip: the same T steps on the bf16 matrix cores (x, v and the scores rounded to bf16, f32 accumulation and
// f32 state; tolerance class 2e-2): any rotary, a lazily decayed state is brought up to date first; host position only.
int bdh_launch_state_prefill_bf16(bdh_ctx *ctx, const StateStepParams &p, float *out_ln);
// prefill.hip: fused_state_aligned (dense causal layout, row-normalised) on the bf16 matrix cores; tolerance class 2e-2
int bdh_launch_fsa_bf16(bdh_ctx *ctx, int B, int h, int T, int N, int dv, const float *query, const float *value,
                        const float *freqs, const float *alibi_slopes_host, int block_size, int rotary, float *out);
// rho <- the up-to-date state, stamps <- clock, for a lazily decayed ALiBi state
int bdh_launch_alibi_materialize(bdh_ctx *ctx, int B, int h, int N, int d, const float *slopes_host, int64_t clock,
                                 const int32_t *clocks_dev, void *rho, int rho_dtype, int32_t *stamps);

// state_deferred.hip: the decode step with logged updates (RoPE, T = 1).  out_ln != nullptr: the readout is also
// written LayerNorm-ed (src/model/bdh.rs:359).  The flush applies the pending steps to rho and empties the log.
int bdh_launch_state_step_deferred(bdh_ctx *ctx, bdh_state_log *log, const float *x, const float *v, const float *freqs,
                                   int64_t position, const int32_t *positions_dev, void *rho, float *out, float *out_ln,
                                   uint64_t *bitmask, int32_t *rows_touched);
int bdh_launch_state_flush(bdh_ctx *ctx, bdh_state_log *log, void *rho);

struct ReluLowrankParams {
  int B, h_in, T, d, h, N;
  const float *in, *weight, *bias;
  float threshold;
  int block_size;
  const uint8_t *active_blocks_host;
  int n_blocks;
  const float *gate;
  float *out;
  bool any_order = false;  // the caller does not need the bits of the k-sequential chain (gated calls only)
};
int bdh_launch_relu_lowrank(bdh_ctx *ctx, const ReluLowrankParams &p);
// a gated call in any order as split-bf16 products, and whether that is the faster form; csrc/attention_parallel.hip
int bdh_launch_relu_lowrank_split(bdh_ctx *ctx, const ReluLowrankParams &p);
bool bdh_relu_lowrank_split_pays(const bdh_ctx *ctx, const ReluLowrankParams &p);
// the same on the f32 matrix cores for many rows per (sequence, head); csrc/attention_parallel.hip
int bdh_launch_relu_lowrank_gemm(bdh_ctx *ctx, const ReluLowrankParams &p, const unsigned char *mask_dev);
// relu_lowrank for ONE input row per head whose values are made by the kernel itself from the partial sums an earlier
// kernel left (a decode step of one sequence: the two reductions of a layer whose inputs come from other CUs ride in
// front of the projection that consumes them, while its weights are on their way):
//   mode 1 (D_y, src/model/bdh.rs:359,370-381): row of head hh = LN(sum_g partial[hh][g][:]), g < S
//   mode 2 (D_x of the next layer, :436-441 then :346-350): row = LN(cur_old + LN(sum_kb dpart[kb][:])), kb < KBN,
//           shared by the heads; the workgroup (0, 0) also writes it to cur_new
//   mode 3 (D_x of the first layer, :319-322 then :346-350): row = LN(embed[tokens[0]]), written to cur_new too
struct ReluLowrankRowParams {
  int mode, h, N, d;
  const float *weight;
  float threshold;
  const float *gate;  // [h][N] or null
  float *out;         // [h][N]
  const float *partial;  // mode 1: [h][S][d]; mode 2: [KBN][d]
  int rows;              // S or KBN
  const float *cur_old;  // mode 2
  float *cur_new;        // modes 2 and 3
  const int64_t *tokens = nullptr;  // mode 3: device, the one token; partial = the embedding table, rows = V
};
int bdh_launch_relu_lowrank_row(bdh_ctx *ctx, const ReluLowrankRowParams &p);
// The first stage of the encoder for one row (M = 1): partial[kb][:] = sum over k-block kb of xy[k] E[k,:], KB rows
// per block; *KBN_out = number of blocks.  partial must hold KBN * d floats.
int bdh_launch_decoder_partial_row(bdh_ctx *ctx, int h, int N, int d, const float *xy, const float *decoder, int KB,
                                   float *partial, int *KBN_out);
// cur[m,:] = LN(cur[m,:] + LN(sum_kb partial[kb][m][:])) and, with head, the output head of the finished rows
int bdh_launch_decoder_finalize_head(bdh_ctx *ctx, const float *partial, int KBN, int M, int d, float *cur,
                                     const struct DecoderHead *head);
int bdh_launch_layer_norm(bdh_ctx *ctx, int64_t rows, int d, const float *in, float *out);
// the same for internal many-row use: statistics by wave reduction, not bit-identical to the index-order sums
int bdh_launch_layer_norm_rows(bdh_ctx *ctx, int64_t rows, int d, const float *in, float *out);

// embed gather + LN (src/model/bdh.rs:319-322); tokens validated on the device: an id
// outside [0,V) writes NaN rows (the reference would panic in the gather).
int bdh_launch_embed_ln(bdh_ctx *ctx, const int64_t *tokens, int64_t rows, int d, int V,
                        const float *embed, float *out);
// mlp = mixed . decoder with mixed[b*T+t, hh*N+n] = xy[b,hh,t,n]; cur = LN(cur + LN(mlp))
// (src/model/bdh.rs:383,436-441)
// The output head of the rows the decoder's second stage finishes, run in that same launch (the last layer of a
// model): logits[m,:] = cur[m,:] . lm_head and, optionally, the greedy token of each sequence's last row.
struct DecoderHead {
  const float *lm_head;  // [d][V]
  int T, V;
  float *logits;         // [M][V]
  int64_t *next_tokens;  // [B] or null
};
int bdh_launch_decoder_residual(bdh_ctx *ctx, int B, int T, int h, int N, int d,
                                const float *xy, const float *decoder, float *cur,
                                const DecoderHead *head = nullptr);
// logits = cur . lm_head (+ argmax of the last token per sequence) (src/model/bdh.rs:446-449)
// attention_parallel.hip: the encoder's terms [*rows_out][B*T][d] of prompts in the context's workspace, from products on
// the matrix cores (all of E is streamed, whatever is active)
int bdh_launch_decoder_partials_f32(bdh_ctx *ctx, int B, int T, int h, int N, int d, const float *xy, const float *decoder,
                                    int *rows_out);
int bdh_launch_lm_head(bdh_ctx *ctx, int B, int T, int d, int V, const float *cur,
                       const float *lm_head, float *logits, int64_t *next_tokens);
// positions[b] = min(positions[b] + delta, INT32_MAX): the device-side form of state.position += T
int bdh_launch_advance_positions(bdh_ctx *ctx, int32_t *positions_dev, int B, int delta);

// viz_taps.hip: out[h,N] = batch mean of the per-row mean |rho| (src/model/bdh.rs:411-419); with stamps the
// state is read through its pending ALiBi decay at clock (or clocks_dev[b] + clock_add)
int bdh_launch_rho_energy(bdh_ctx *ctx, int B, int h, int N, int d, const void *rho, int rho_dtype,
                          const int32_t *stamps, const float *slopes_host, int64_t clock, const int32_t *clocks_dev,
                          int clock_add, float *out);
// dst[hh, 0..cols) = src[hh * head_stride + offset + (0..cols)]
int bdh_launch_gather_head_rows(bdh_ctx *ctx, const float *src, int h, long head_stride, long offset, int cols,
                                float *dst);
int bdh_launch_fill_zero_f32(bdh_ctx *ctx, float *p, long n);

// Four adjacent elements of a state row, f32 or bf16 (raw 16-bit patterns; stores round to nearest even, NaN kept
// quiet): the element access of the decode forms that keep the state in either type.
__device__ __forceinline__ float4 bdh_rho_load4(const float *p) { return *reinterpret_cast<const float4 *>(p); }
__device__ __forceinline__ float4 bdh_rho_load4(const unsigned short *p) {
  const uint2 v = *reinterpret_cast<const uint2 *>(p);
  return make_float4(__uint_as_float(v.x << 16), __uint_as_float(v.x & 0xffff0000u), __uint_as_float(v.y << 16),
                     __uint_as_float(v.y & 0xffff0000u));
}
__device__ __forceinline__ unsigned int bdh_bf16_rne(float f) {
  unsigned int u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (u >> 16) | 0x40u;
  u += 0x7fffu + ((u >> 16) & 1u);
  return u >> 16;
}
__device__ __forceinline__ void bdh_rho_store4(float *p, float4 v) { *reinterpret_cast<float4 *>(p) = v; }
__device__ __forceinline__ void bdh_rho_store4(unsigned short *p, float4 v) {
  uint2 o;
  o.x = bdh_bf16_rne(v.x) | (bdh_bf16_rne(v.y) << 16);
  o.y = bdh_bf16_rne(v.z) | (bdh_bf16_rne(v.w) << 16);
  *reinterpret_cast<uint2 *>(p) = o;
}

// ---- sums over a wavefront ----------------------------------------------------------
template <int CTRL>
__device__ __forceinline__ float bdh_dpp(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}
// All lanes get the sum over the lanes l, l ^ 32, l ^ 16, l ^ 48: v + (its neighbour 32 away), then 16 away.
__device__ __forceinline__ float bdh_sum_over_rows(float v) {
  const unsigned int u = __float_as_uint(v);
  const auto a = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  const unsigned int w = __float_as_uint(v);
  const auto b = __builtin_amdgcn_permlane16_swap(w, w, false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}
// All lanes get the wave's sum: the bits of `for (o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o)` without its six trips
// through LDS.  (A rotation of a row of sixteen by four reaches the lane 4 away in either half: those are equal by then.)
__device__ __forceinline__ float bdh_wave_sum(float v) {
  v = bdh_sum_over_rows(v);
  v += bdh_dpp<0x128>(v);  // row rotated by 8
  v += bdh_dpp<0x124>(v);  // by 4
  v += bdh_dpp<0x4e>(v);   // lanes 2 apart
  v += bdh_dpp<0xb1>(v);   // neighbours
  return v;
}
// v / den for many v and one den, r = 1 / den rounded: one correction of v * r by its remainder gives the rounded quotient
// (P. Markstein, IBM J. Res. Dev. 34, 1990) in three operations instead of the ten of a division.  v and den are finite.
__device__ __forceinline__ float bdh_quotient(float v, float den, float r) {
  const float q = v * r;
  return __builtin_fmaf(__builtin_fmaf(-q, den, v), r, q);
}
// 0 + p[0] + p[step] + ... in index order (n the same for the wave), 16, 8 or 4 of the n values on their way at a time.
template <int U, typename V>
__device__ __forceinline__ void bdh_add_in_order(V &s, const V *p, long step) {
  V t[U];
#pragma unroll
  for (int u = 0; u < U; ++u) t[u] = p[u * step];
#pragma unroll
  for (int u = 0; u < U; ++u) s += t[u];
}
template <typename V>
__device__ __forceinline__ V bdh_sum_in_order(const V *p, long step, int n) {
  V s = V{};
  int g = 0;
  for (; g + 16 <= n; g += 16) bdh_add_in_order<16>(s, p + g * step, step);
  if (g + 8 <= n) { bdh_add_in_order<8>(s, p + g * step, step); g += 8; }
  if (g + 4 <= n) { bdh_add_in_order<4>(s, p + g * step, step); g += 4; }
  for (; g < n; ++g) s += p[g * step];
  return s;
}
