// A decode step (one token per sequence) of a mid-size model in TWO launches per layer instead of six.
// Kernel by kernel a layer of BDH::forward_with_state (src/model/bdh.rs:336-441) is D_x, state step, its second
// stage, D_y, encoder partials, encoder second stage; at a few sequences each of those is a launch latency plus a
// trip or two to memory.  The only points where a layer needs data from the whole sequence are the LayerNorm of
// a head's readout and the LayerNorm of the encoder output, so a workgroup that owns 64 (or 32) neurons of one head
// of one sequence can run everything between them on its own:
//   phase A: [previous layer's cur = LN(cur + LN(sum of encoder partials))]  D_x for its neurons, their state
//            rows (readout, update, decay), the readout partial of the workgroup;
//   phase B: LN(sum of the head's readout partials), D_y and the gate for its neurons, the encoder partial of
//            those rows of E.
// The sums over partials are redone by every workgroup that needs them (a few KiB from the L2).  All sums are taken in a
// fixed tree of their own (results agree with the kernel-by-kernel step to rounding, not bit for bit).
//
// What bounds it: latency.  Both phases ask for everything whose address does not depend on a result -- the partials, the
// weights, the state rows or the rows of E -- in the order in which it is needed, before they wait for any of it: one trip
// to memory per launch where one after the other takes three.  Weights come 16 bytes a lane, sixteen lanes per row of k,
// so a lane's part of a column's sum has d / (4 waves) terms and the parts meet over lanes and in LDS once; a chain over
// all of k, handed from wave to wave, took 2.0 us of phase A at d = 256 and 3.2 at 512.  Every wave redoes the LayerNorms
// on its own copy of the row: no barriers between their sums.  First start to last end of a launch, one sequence, d = 256,
// 1024 neurons: phase A 9.2 -> 4.3 us, phase B 5.7 -> 2.5; d = 512, 2048 neurons: 12.5 -> 6.6, 7.7 -> 3.5.  The 1.5 us from the
// end of one launch to the start of the next remain.
#include <algorithm>
#include <cfloat>

#include "bdh_internal.h"

namespace {

constexpr float kLnEps = 1e-5f;                    // src/model/bdh.rs:17
constexpr float kTwoPi = 6.28318530717958647692f;  // f32(2*PI), src/model/attention.rs:343

struct PhaseArgs {
  const int64_t *tokens;      // first layer only: [B] tokens, the layer's input is LN(embed[token]) (else null)
  const float *embed;         // [V][d]
  int V;
  const float *cur_in;        // [B][d] the layer's input before the pending encoder second stage (not the first layer)
  float *cur_out;             // [B][d] the layer's input, written by the first workgroup of a sequence
  const float *dec_partial;   // [G][B][d] encoder partials of the previous layer (not the first layer)
  float *x;                   // [B][h*N]
  float *attn_partial;        // [B][h][N / block][d]
  float *dec_partial_out;     // [G][B][d], G = h * N / block
  const float *enc, *enc_v, *dec, *freqs;
  void *rho;                  // this layer's state [B][h][Nq][d], f32 or bf16
  int32_t *stamps;            // this layer's stamps [B][h][N] or null
  const int32_t *pos_dev;
  long pos;
  int B, d, h, N, rotary;
  float thr;
  float decay[64], log_decay[64];
};

// The wave of the workgroup, in a scalar register: addresses that only depend on it cost the lanes nothing.
__device__ __forceinline__ int wave_id() { return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); }
// p[at / 4]: one base for the wave, a 32-bit byte offset per lane
template <typename V, typename T>
__device__ __forceinline__ V load_at(const T *p, unsigned int at) {
  return *reinterpret_cast<const V *>(reinterpret_cast<const char *>(p) + at);
}

// Four weights of a caller's array, which floats may begin at any address of theirs: one 16-byte load all the same.
__device__ __forceinline__ float4 load_weights(const float *p, unsigned int at) {
  typedef float Quad __attribute__((ext_vector_type(4), aligned(4)));
  const Quad q = load_at<Quad>(p, at);
  return make_float4(q.x, q.y, q.z, q.w);
}

// Orders a wave's own LDS writes and reads of other lanes' values for the compiler (the hardware runs them in order).
__device__ __forceinline__ void wave_lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// LayerNorm of a row held by one wave, column j * 64 + lane in v[j] (src/model/bdh.rs:86-89); zero beyond d.
template <int CJ>
__device__ __forceinline__ void wave_layer_norm(float (&v)[CJ], int d) {
  const int lane = threadIdx.x & 63;
  const float fd = (float)d, rd = 1.0f / fd;
  float s = 0.0f;
#pragma unroll
  for (int j = 0; j < CJ; ++j) s += j * 64 + lane < d ? v[j] : 0.0f;
  const float mean = bdh_quotient(bdh_wave_sum(s), fd, rd);
  float q = 0.0f;
#pragma unroll
  for (int j = 0; j < CJ; ++j) {
    const float c = j * 64 + lane < d ? v[j] - mean : 0.0f;
    v[j] = c;
    q += c * c;
  }
  // A variance beyond the floats is infinite and the row then zero, as the divisions have it: the remainder inf - inf of
  // either quotient must not come in.
  const float sum = bdh_wave_sum(q);
  const float den = sqrtf((sum <= FLT_MAX ? bdh_quotient(sum, fd, rd) : sum) + kLnEps), r = 1.0f / den;
  const float finite = fminf(den, FLT_MAX);
#pragma unroll
  for (int j = 0; j < CJ; ++j) v[j] = bdh_quotient(v[j], finite, r);
}

// How the NW waves of a workgroup share rows of d <= DC floats and the NB neurons of its block.
template <int DC, int NW, int NB>
struct Shape {
  static constexpr int NT = NW * 64;
  static constexpr int CJ = DC / 64;            // columns per lane where every wave holds the whole row
  static constexpr int RG = NT * 4 / DC;        // rows of partial sums that one 16-byte access of the workgroup covers
  static constexpr int PG = 64 / RG;            // ... and how many accesses 64 of them take
  static constexpr int LPW = NB / 4;            // lanes per row of a weight block, 16 bytes each
  static constexpr int KR = DC / NW / (64 / LPW);  // rows of a weight block per lane
  static constexpr int LPR = DC < 256 ? 32 : 64;  // lanes per state row (or row of E), 16 or 8 bytes each
  static constexpr int VPL = DC / (4 * LPR);    // pieces of a row per lane
  static constexpr int RPI = 64 / LPR;          // rows per access of a wave
  static constexpr int RU = NB / NW / RPI;      // accesses for a wave's share of NB rows
};

// The sum of `rows` <= 64 rows of d floats, the next one `stride` floats on: asked for by ask(), column j * 64 + lane of the
// sum in v[j] of every wave by collect(), which holds a barrier.
template <int DC, int NW>
struct RowSum {
  using S = Shape<DC, NW, 64>;
  float4 t[S::PG];
  __device__ __forceinline__ void ask(const float *__restrict__ src, long stride, int rows, int d) {
    const int rg = threadIdx.x / (DC / 4), c = threadIdx.x % (DC / 4) * 4;
    const unsigned int at = (c < d ? c : 0) * 4u, step = (unsigned int)stride * 4u;
#pragma unroll
    for (int i = 0; i < S::PG; ++i) {
      t[i] = make_float4(0.f, 0.f, 0.f, 0.f);
      if (i == 0 || i * S::RG < rows)  // uniform
        t[i] = load_at<float4>(src, at + min(i * S::RG + rg, rows - 1) * step);
    }
  }
  __device__ __forceinline__ void add(int rows, float4 *s_part) {  // this thread's part, [RG][DC]
    const int rg = threadIdx.x / (DC / 4);
    float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int i = 0; i < S::PG; ++i) {
      const bool in = i * S::RG + rg < rows;
      s.x += in ? t[i].x : 0.0f;
      s.y += in ? t[i].y : 0.0f;
      s.z += in ? t[i].z : 0.0f;
      s.w += in ? t[i].w : 0.0f;
    }
    s_part[threadIdx.x] = s;
  }
  __device__ __forceinline__ void collect(int rows, float4 *s_part, float (&v)[S::CJ]) {
    add(rows, s_part);
    __syncthreads();
    const float *f = reinterpret_cast<const float *>(s_part) + (threadIdx.x & 63);
#pragma unroll
    for (int j = 0; j < S::CJ; ++j) {
      v[j] = f[j * 64];
#pragma unroll
      for (int r = 1; r < S::RG; ++r) v[j] += f[r * DC + j * 64];
    }
  }
};

// row . w for NB columns of a weight matrix [d][N] (`weight` points at the first of them): ask() requests this wave's
// DC / NW rows of k, dot() returns the sum of column lane % NB in every wave (it holds a barrier).  s_row: the wave's own
// copy of the input row, zero beyond d.
template <int DC, int NW, int NB>
struct Project {
  using S = Shape<DC, NW, NB>;
  float4 w[S::KR];
  static __device__ __forceinline__ int first_k() { return wave_id() * (DC / NW) + (int)(threadIdx.x & 63) / S::LPW * S::KR; }
  __device__ __forceinline__ void ask(const float *__restrict__ weight, int d, int N) {
    const int k0 = first_k();
    unsigned int at = (min(k0, d - 1) * N + (threadIdx.x & (S::LPW - 1)) * 4) * 4u;
#pragma unroll
    for (int u = 0; u < S::KR; ++u) {
      w[u] = load_weights(weight, at);
      at += k0 + u < d - 1 ? N * 4u : 0u;  // not beyond the last row
    }
  }
  __device__ __forceinline__ float dot(const float *s_row, int d, float (*s_acc)[NB]) {
    const int lane = threadIdx.x & 63, k0 = first_k();
    if (d < DC) {  // what was asked for beyond the last row of k does not count
#pragma unroll
      for (int u = 0; u < S::KR; ++u)
        if (k0 + u >= d) w[u] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
    float r[S::KR];
#pragma unroll
    for (int u = 0; u < S::KR; ++u) r[u] = s_row[k0 + u];
    float p[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < S::KR; ++u) {
      p[0] = __builtin_fmaf(r[u], w[u].x, p[0]);
      p[1] = __builtin_fmaf(r[u], w[u].y, p[1]);
      p[2] = __builtin_fmaf(r[u], w[u].z, p[2]);
      p[3] = __builtin_fmaf(r[u], w[u].w, p[3]);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {  // over the lanes with the same columns: LPW apart
      if (S::LPW <= 4) p[e] += bdh_dpp<0x124>(p[e]);  // rotations of a row of sixteen by four and eight
      if (S::LPW <= 8) p[e] += bdh_dpp<0x128>(p[e]);
      p[e] = bdh_sum_over_rows(p[e]);
    }
    if (lane < S::LPW) *reinterpret_cast<float4 *>(&s_acc[wave_id()][lane * 4]) = make_float4(p[0], p[1], p[2], p[3]);
    __syncthreads();
    const int c = lane & (NB - 1);
    float s = s_acc[0][c];
#pragma unroll
    for (int w2 = 1; w2 < NW; ++w2) s += s_acc[w2][c];
    return s;
  }
};

// out[0..d) = the sum over the workgroup of the lanes' pieces of a row (Shape::VPL each; lanes of one wave that hold the
// same columns are added first).  Holds a barrier.
template <int DC, int NW>
__device__ __forceinline__ void write_row_sum(const float4 (&acc)[Shape<DC, NW, 64>::VPL], float (*s_red)[DC], int d,
                                              float *__restrict__ out) {
  using S = Shape<DC, NW, 64>;
  const int tid = threadIdx.x, lane = tid & 63, wave = wave_id();
#pragma unroll
  for (int j = 0; j < S::VPL; ++j) {
    float4 t = acc[j];
    if (S::RPI == 2) {
      t.x += __shfl_xor(t.x, 32);
      t.y += __shfl_xor(t.y, 32);
      t.z += __shfl_xor(t.z, 32);
      t.w += __shfl_xor(t.w, 32);
    }
    if (S::RPI == 1 || lane < S::LPR) *reinterpret_cast<float4 *>(&s_red[wave][(j * S::LPR + lane) * 4]) = t;
  }
  __syncthreads();
  for (int c = tid; c < d; c += S::NT) {
    float s = s_red[0][c];
#pragma unroll
    for (int w = 1; w < NW; ++w) s += s_red[w][c];
    out[c] = s;
  }
}

// A load through the scalar cache (the address is the same for the whole wave and nothing in this launch writes it).
template <typename T>
__device__ __forceinline__ T scalar_load(const T *p) {
  return *reinterpret_cast<const __attribute__((address_space(4))) T *>(reinterpret_cast<uintptr_t>(p));
}

// Four state elements as they are stored.
__device__ __forceinline__ float4 load_raw(const float *p) { return *reinterpret_cast<const float4 *>(p); }
__device__ __forceinline__ uint2 load_raw(const unsigned short *p) { return *reinterpret_cast<const uint2 *>(p); }
__device__ __forceinline__ float4 widen(float4 v) { return v; }
__device__ __forceinline__ float4 widen(uint2 v) {
  return make_float4(__uint_as_float(v.x << 16), __uint_as_float(v.x & 0xffff0000u), __uint_as_float(v.y << 16),
                     __uint_as_float(v.y & 0xffff0000u));
}

// ---- phase A ---------------------------------------------------------------------------------------------------
// AHEAD: all NB state rows are asked for before it is known which of them are visited (the launcher says when); otherwise
// the visited ones once they are.
// FIRST: the first layer, whose input is the LayerNorm of the embedding row.
template <int DC, int NW, int NB, typename RhoT, bool AHEAD, bool FIRST>
__global__ __launch_bounds__(NW * 64, AHEAD || DC == 512 ? 2 : 4) void k_layer_phase_a(PhaseArgs a) {
  using S = Shape<DC, NW, NB>;
  typedef decltype(load_raw((const RhoT *)nullptr)) Raw;
  __shared__ float4 s_part[S::NT];
  __shared__ __align__(16) float s_cur[NW][DC];  // every wave's own copy of the layer's input, zero beyond d
  __shared__ __align__(16) float s_acc[NW][NB];
  __shared__ unsigned char s_list[NW][NB];
  __shared__ __align__(16) float s_red[NW][DC];

  const int lane = threadIdx.x & 63, wave = wave_id();
  const int nblk = blockIdx.x, hh = blockIdx.y, b = blockIdx.z;
  const int d = a.d, h = a.h, N = a.N;
  const float dec = a.decay[hh], log_dec = a.log_decay[hh];
  // the kernel arguments in one go: fetched where each is used, they are eight waits one after the other
  asm volatile("" ::"s"(a.tokens), "s"(a.embed), "s"(a.cur_in), "s"(a.cur_out), "s"(a.dec_partial), "s"(a.x), "s"(a.attn_partial),
               "s"(a.enc), "s"(a.freqs), "s"(a.rho), "s"(a.stamps), "s"(a.pos_dev), "s"(a.pos), "s"(a.B), "s"(a.V), "s"(d),
               "s"(h), "s"(N), "s"(a.rotary), "s"(a.thr), "s"(dec), "s"(log_dec));
  const int nblk_n = N / NB;
  const int nl = lane & (NB - 1), n = nblk * NB + nl;  // this lane's neuron of the block and of the head
  const bool alibi = a.rotary == BDH_ALIBI, pope = a.rotary == BDH_POPE;
  const int Nq = pope ? 2 * N : N;
  RhoT *rho = static_cast<RhoT *>(a.rho) + ((long)b * h + hh) * (long)Nq * d;
  int32_t *st = a.stamps ? a.stamps + ((long)b * h + hh) * N : nullptr;
  const bool lazy = alibi && st != nullptr;

  // everything this launch reads, in the order of use
  float cur[S::CJ];
  RowSum<DC, NW> partials;
  bool bad = false;
  if constexpr (FIRST) {  // embedding row (src/model/bdh.rs:319-322); a bad token poisons the row
    const int64_t tok = scalar_load(a.tokens + b);
    bad = tok < 0 || tok >= a.V;
    const float *e = a.embed + (bad ? 0 : (long)tok * d);
#pragma unroll
    for (int j = 0; j < S::CJ; ++j) cur[j] = e[min(j * 64 + lane, d - 1)];
  } else {
    partials.ask(a.dec_partial + (long)b * d, (long)a.B * d, h * nblk_n, d);
#pragma unroll
    for (int j = 0; j < S::CJ; ++j) cur[j] = a.cur_in[(long)b * d + min(j * 64 + lane, d - 1)];
  }
  Project<DC, NW, NB> dx;
  dx.ask(a.enc + (long)hh * d * N + nblk * NB, d, N);
  const long pos = a.pos_dev ? (long)scalar_load(a.pos_dev + b) : a.pos;
  const float posf = (float)pos;
  const float freq = a.freqs[n];
  const int stamp = *(lazy ? st + n : reinterpret_cast<const int32_t *>(a.freqs + n));  // unused unless lazy: no branch
  const int sub = S::RPI == 2 ? lane >> 5 : 0, cl = lane & (S::LPR - 1);
  Raw rv[S::RU][S::VPL];
  // the row of slot u: row `base` of the head (the same for the wave), `more` (0 or, for half a wave, some) rows further on
  auto load_row = [&](int u, long base, int more) {
#pragma unroll
    for (int j = 0; j < S::VPL; ++j) {
      const int c = (j * S::LPR + cl) * 4;
      rv[u][j] = load_raw(rho + base * d + (more * d + (c < d ? c : 0)));
    }
  };
  // first row of slot u of this wave's share of the block when all are taken
  auto own_row = [&](int u) { return (wave * S::RU + u) * S::RPI; };
  if constexpr (AHEAD) {
#pragma unroll
    for (int u = 0; u < S::RU; ++u) load_row(u, nblk * NB + own_row(u), sub);
  }

  __builtin_amdgcn_sched_barrier(0);  // nothing is waited for before all of it is on its way

  // the layer's input: cur, after the pending second stage of the previous layer's encoder
  // (src/model/bdh.rs:383, 436-441: cur = LN(cur + LN(mixed . decoder)))
  if constexpr (FIRST) {
    if (bad) {
#pragma unroll
      for (int j = 0; j < S::CJ; ++j) cur[j] = __int_as_float(0x7fc00000);
    }
  } else {
    float mlp[S::CJ];
    partials.collect(h * nblk_n, s_part, mlp);
    wave_layer_norm<S::CJ>(mlp, d);
#pragma unroll
    for (int j = 0; j < S::CJ; ++j) cur[j] = cur[j] + mlp[j];
  }
  wave_layer_norm<S::CJ>(cur, d);
#pragma unroll
  for (int j = 0; j < S::CJ; ++j) s_cur[wave][j * 64 + lane] = j * 64 + lane < d ? cur[j] : 0.0f;
  if (hh == 0 && nblk == 0 && wave == 0) {
#pragma unroll
    for (int j = 0; j < S::CJ; ++j)
      if (j * 64 + lane < d) a.cur_out[(long)b * d + j * 64 + lane] = cur[j];
  }
  wave_lds_order();

  // x = relu(cur . encoder - thr) for the block's neurons (src/model/bdh.rs:337-351), the same in every wave
  float xn = dx.dot(s_cur[wave], d, s_acc);
  if (a.thr != 0.0f) xn = xn - a.thr;
  xn = xn > 0.0f ? xn : 0.0f;
  if (wave == 0 && lane < NB) a.x[((long)b * h + hh) * N + n] = xn;

  // the state rows of these neurons (src/model/bdh.rs:232-306): readout with the old rows, rank-1 update with
  // value = cur, ALiBi decay; only visited rows are touched
  float4 acc[S::VPL], vv[S::VPL];
#pragma unroll
  for (int j = 0; j < S::VPL; ++j) {
    acc[j] = make_float4(0.f, 0.f, 0.f, 0.f);
    vv[j] = *reinterpret_cast<const float4 *>(&s_cur[wave][(j * S::LPR + cl) * 4]);
  }
  for (int part = 0; part < (pope ? 2 : 1); ++part) {  // PoPE: real rows n, then imaginary rows N + n
    float q_l = 0.0f, scale_l = 1.0f;
    bool touch_l = false;
    if (alibi) {  // q = x (src/model/attention.rs:332-349)
      q_l = xn;
      touch_l = lazy ? (q_l != 0.0f) : true;
      if (lazy && touch_l) {
        const long k = pos - (long)stamp;
        if (k > 0) scale_l = expf((float)k * log_dec);
      }
    } else if (pope) {  // src/model/attention.rs:323-330
      const float mag = logf(expf(xn * 1.0f) + 1.0f) / 1.0f;
      const float raw = posf * freq;
      const float ph = (raw - floorf(raw)) * kTwoPi;
      q_l = part == 0 ? mag * cosf(ph) : mag * sinf(ph);
      touch_l = true;
    } else {  // RoPE (src/model/attention.rs:305-321)
      const float xo = bdh_dpp<0xb1>(xn);  // the other neuron of the pair
      touch_l = (xn != 0.0f) || (xo != 0.0f);
      if (touch_l) {
        const float raw = posf * freq;
        const float ph = (raw - floorf(raw)) * kTwoPi;
        float sn, cs;
        sincosf(ph, &sn, &cs);
        const float rot = (n & 1) ? xo : -xo;
        const float t0 = xn * cs, t1 = rot * sn;
        q_l = t0 + t1;
      }
    }
    const unsigned long long m = __ballot(touch_l && lane < NB);
    const long row_base = (long)(part * N + nblk * NB);
    int src[S::RU];  // the row of slot u, and whether it is visited
    bool ok[S::RU];
    if constexpr (AHEAD) {
#pragma unroll
      for (int u = 0; u < S::RU; ++u) {
        src[u] = own_row(u) + sub;
        ok[u] = S::RPI == 1 ? (m >> own_row(u)) & 1 : (m >> own_row(u) >> sub) & 1;
      }
    } else {  // every wave makes the same list of visited rows and takes every NW-th entry (pair of entries) of it
      const int count = __popcll(m);
      if (touch_l && lane < NB) s_list[wave][__popcll(m & ((1ull << lane) - 1ull))] = (unsigned char)lane;
      wave_lds_order();
#pragma unroll
      for (int u = 0; u < S::RU; ++u) {
        const int idx = (u * NW + wave) * S::RPI + sub;
        const int listed = s_list[wave][idx & (NB - 1)];  // read whether or not the slot is used: no branch
        ok[u] = idx < count;
        src[u] = ok[u] ? listed : 0;
        if (S::RPI == 1) src[u] = __builtin_amdgcn_readfirstlane(src[u]);
      }
#pragma unroll
      for (int u = 0; u < S::RU; ++u)
        if (u * NW * S::RPI < count)  // uniform
          load_row(u, row_base + (S::RPI == 1 ? src[u] : 0), S::RPI == 1 ? 0 : src[u]);
    }
#pragma unroll
    for (int u = 0; u < S::RU; ++u) {
      if (!AHEAD && u * NW * S::RPI >= __popcll(m)) break;
      float q_src, scale = 1.0f;
      if (S::RPI == 1) {
        q_src = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(q_l), src[u]));
        if (lazy) scale = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(scale_l), src[u]));
      } else {
        q_src = __shfl(q_l, src[u], 64);
        if (lazy) scale = __shfl(scale_l, src[u], 64);
      }
      if (S::RPI == 1 && !ok[u]) continue;  // uniform
      const float qn = ok[u] ? q_src : 0.0f;
      RhoT *row = rho + (row_base + (S::RPI == 1 ? src[u] : 0)) * d + (S::RPI == 1 ? 0 : src[u]) * d;
      Raw old[S::VPL];
#pragma unroll
      for (int j = 0; j < S::VPL; ++j) old[j] = rv[u][j];
      if (AHEAD && pope && part == 0) load_row(u, (long)N + nblk * NB + own_row(u), sub);  // its imaginary row
#pragma unroll
      for (int j = 0; j < S::VPL; ++j) {
        const int c = (j * S::LPR + cl) * 4;
        float4 e = widen(old[j]);
        if (!ok[u]) e = make_float4(0.f, 0.f, 0.f, 0.f);
        if (lazy) {
          e.x *= scale; e.y *= scale; e.z *= scale; e.w *= scale;
        }
        acc[j].x = __builtin_fmaf(e.x, qn, acc[j].x);
        acc[j].y = __builtin_fmaf(e.y, qn, acc[j].y);
        acc[j].z = __builtin_fmaf(e.z, qn, acc[j].z);
        acc[j].w = __builtin_fmaf(e.w, qn, acc[j].w);
        float t;
        t = qn * vv[j].x; e.x = e.x + t;
        t = qn * vv[j].y; e.y = e.y + t;
        t = qn * vv[j].z; e.z = e.z + t;
        t = qn * vv[j].w; e.w = e.w + t;
        if (alibi) {  // src/model/bdh.rs:299-301
          e.x *= dec; e.y *= dec; e.z *= dec; e.w *= dec;
        }
        if (ok[u] && c < d) bdh_rho_store4(row + c, e);
      }
    }
  }
  write_row_sum<DC, NW>(acc, s_red, d, a.attn_partial + (((long)b * h + hh) * nblk_n + nblk) * d);
  // behind the barrier in there: every wave has its stamps
  if (lazy && xn != 0.0f && wave == 0 && lane < NB) st[n] = (int32_t)min(pos + 1, 0x7fffffffL);
}

// ---- phase B ---------------------------------------------------------------------------------------------------
template <int DC, int NW, int NB>
__global__ __launch_bounds__(NW * 64, 2) void k_layer_phase_b(PhaseArgs a) {
  using S = Shape<DC, NW, NB>;
  __shared__ float4 s_part[S::NT];
  __shared__ __align__(16) float s_in[NW][DC];
  __shared__ __align__(16) float s_acc[NW][NB];
  __shared__ __align__(16) float s_red[NW][DC];

  const int lane = threadIdx.x & 63, wave = wave_id();
  const int nblk = blockIdx.x, hh = blockIdx.y, b = blockIdx.z;
  const int d = a.d, h = a.h, N = a.N;
  asm volatile("" ::"s"(a.attn_partial), "s"(a.x), "s"(a.enc_v), "s"(a.dec), "s"(a.dec_partial_out), "s"(a.B), "s"(d), "s"(h),
               "s"(N), "s"(a.thr));  // in one go, as above
  const int nblk_n = N / NB;

  // everything this launch reads, in the order of use: the readout partials of the head, its part of D_y, the gate, and
  // these NB rows of E
  RowSum<DC, NW> partials;
  partials.ask(a.attn_partial + ((long)b * h + hh) * nblk_n * d, d, nblk_n, d);
  Project<DC, NW, NB> dy;
  dy.ask(a.enc_v + (long)hh * d * N + nblk * NB, d, N);
  const float gate = a.x[((long)b * h + hh) * N + nblk * NB + (lane & (NB - 1))];
  const int sub = S::RPI == 2 ? lane >> 5 : 0, cl = lane & (S::LPR - 1);
  float4 ev[S::RU][S::VPL];
#pragma unroll
  for (int u = 0; u < S::RU; ++u) {
    const float *e = a.dec + ((long)hh * N + nblk * NB + (wave * S::RU + u) * S::RPI) * d;
#pragma unroll
    for (int j = 0; j < S::VPL; ++j) {
      const int c = (j * S::LPR + cl) * 4;
      ev[u][j] = load_weights(e, (sub * d + (c < d ? c : 0)) * 4u);
    }
  }

  __builtin_amdgcn_sched_barrier(0);

  // LayerNorm of the head's readout (src/model/bdh.rs:359)
  {
    float at[S::CJ];
    partials.collect(nblk_n, s_part, at);
    wave_layer_norm<S::CJ>(at, d);
#pragma unroll
    for (int j = 0; j < S::CJ; ++j) s_in[wave][j * 64 + lane] = j * 64 + lane < d ? at[j] : 0.0f;
    wave_lds_order();
  }
  // xy = x * relu(LN(attn) . encoder_v - thr) for the block's neurons (src/model/bdh.rs:361-381), the same in every wave
  float y = dy.dot(s_in[wave], d, s_acc);
  if (a.thr != 0.0f) y = y - a.thr;
  const float xy = gate * (y > 0.0f ? y : 0.0f);

  // encoder partial of these rows of E (src/model/bdh.rs:383)
  float4 acc[S::VPL];
#pragma unroll
  for (int j = 0; j < S::VPL; ++j) acc[j] = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
  for (int u = 0; u < S::RU; ++u) {
    const int r = (wave * S::RU + u) * S::RPI + sub;
    const float q = S::RPI == 1 ? __int_as_float(__builtin_amdgcn_readlane(__float_as_int(xy), r)) : __shfl(xy, r, 64);
#pragma unroll
    for (int j = 0; j < S::VPL; ++j) {
      acc[j].x = __builtin_fmaf(q, ev[u][j].x, acc[j].x);
      acc[j].y = __builtin_fmaf(q, ev[u][j].y, acc[j].y);
      acc[j].z = __builtin_fmaf(q, ev[u][j].z, acc[j].z);
      acc[j].w = __builtin_fmaf(q, ev[u][j].w, acc[j].w);
    }
  }
  write_row_sum<DC, NW>(acc, s_red, d, a.dec_partial_out + ((long)(hh * nblk_n + nblk) * a.B + b) * d);
}

// ---- head -----------------------------------------------------------------------------------------------------
// The last layer's pending second stage, then the logits and the greedy token (src/model/bdh.rs:436-449): one
// workgroup of 16 waves per sequence.  logits[v] = sum_k cur[k] * lm_head[k][v]: a thread takes NC adjacent columns (the last
// thread of a row may take some of its neighbour's again, alike) and one of GK spans of k, in one fmaf chain per column whose
// first AHEAD rows are asked for before the LayerNorms (wave 0 makes those); the spans of a wave are added in its registers,
// the others in order; the lowest index wins ties.  What bounds it: the launch, one trip to memory, and for the larger
// vocabularies that one CU fetches all of lm_head, 64 bytes a cycle.  d = 128, V = 69, one sequence: 7.2 us with a column a
// thread, half of the threads idle, rows worked on as 512 wide whatever d, and spans of k in whole waves; 5.1 here.
template <int DC, int NC>
__global__ __launch_bounds__(1024) void k_phase_head(const float *__restrict__ cur_in, const float *__restrict__ dec_partial,
                                                     int G, int B, int d, const float *__restrict__ lm_head, int V,
                                                     float *__restrict__ logits, int64_t *__restrict__ next) {
  using S = Shape<DC, 16, 64>;
  constexpr int AHEAD = 16;
  typedef float Cols __attribute__((ext_vector_type(NC), aligned(4)));
  __shared__ float s_cur[DC];
  __shared__ float4 s_part[1024];
  __shared__ float s_grp[1024 * NC];
  __shared__ float s_best[16];
  __shared__ int s_arg[16];
  const int tid = threadIdx.x, lane = tid & 63, wave = wave_id();
  const int b = blockIdx.x;
  RowSum<DC, 16> partials;
  partials.ask(dec_partial + (long)b * d, (long)B * d, G, d);
  float cur[S::CJ];
#pragma unroll
  for (int j = 0; j < S::CJ; ++j) cur[j] = wave == 0 ? cur_in[(long)b * d + min(j * 64 + lane, d - 1)] : 0.0f;
  const int per_row = (V + NC - 1) / NC;  // threads per row of lm_head
  const int span = per_row <= 16 ? 16 : per_row <= 32 ? 32 : (per_row + 63) & ~63, GK = 1024 / span;
  const int g = tid / span, c = min((tid - g * span) * NC, V - NC);
  const int per = (d + GK - 1) / GK;
  const bool busy = g < GK && tid - g * span < per_row;
  const int k0 = min(d, g * per), k1 = busy ? min(d, k0 + per) : k0;
  const float *wp = lm_head + (busy ? c : 0);
  Cols wv[AHEAD];
#pragma unroll
  for (int u0 = 0; u0 < AHEAD; u0 += 4) {
    if (u0 < per) {  // uniform
#pragma unroll
      for (int u = 0; u < 4; ++u) wv[u0 + u] = *reinterpret_cast<const Cols *>(wp + (long)min(k0 + u0 + u, d - 1) * V);
    }
  }
  __builtin_amdgcn_sched_barrier(0);

  partials.add(G, s_part);
  __syncthreads();
  if (tid < DC) {
    const float *f = reinterpret_cast<const float *>(s_part) + tid;
    float v = f[0];
#pragma unroll
    for (int r = 1; r < S::RG; ++r) v += f[r * DC];
    s_cur[tid] = v;
  }
  __syncthreads();
  if (wave == 0) {
    float mlp[S::CJ];
#pragma unroll
    for (int j = 0; j < S::CJ; ++j) mlp[j] = s_cur[j * 64 + lane];
    wave_layer_norm<S::CJ>(mlp, d);
#pragma unroll
    for (int j = 0; j < S::CJ; ++j) cur[j] = cur[j] + mlp[j];
    wave_layer_norm<S::CJ>(cur, d);
#pragma unroll
    for (int j = 0; j < S::CJ; ++j) s_cur[j * 64 + lane] = cur[j];
  }
  __syncthreads();
  Cols acc = 0.0f;
  if (busy) {
    auto add4 = [&](int k, const Cols *w) {  // a row past the span counts as zero
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const bool in = k + u < k1;
        acc = __builtin_elementwise_fma(Cols(s_cur[in ? k + u : 0]), in ? w[u] : Cols(0.0f), acc);
      }
    };
#pragma unroll
    for (int u0 = 0; u0 < AHEAD; u0 += 4)
      if (u0 < per) add4(k0 + u0, wv + u0);
    for (int k = k0 + AHEAD; k < k0 + per; k += 16) {  // narrow vocabularies and long rows only
#pragma unroll
      for (int u = 0; u < 16; ++u) wv[u] = *reinterpret_cast<const Cols *>(wp + (long)min(k + u, d - 1) * V);
#pragma unroll
      for (int u = 0; u < 16; u += 4) add4(k + u, wv + u);
    }
  }
  // the spans of one wave
#pragma unroll
  for (int e = 0; e < NC; ++e) {
    if (span == 16) acc[e] = bdh_sum_over_rows(acc[e]);
    else if (span == 32) acc[e] += __shfl_xor(acc[e], 32);
  }
  const int rows = min(GK, 16);
  if (busy && (span >= 64 || lane < span)) {
#pragma unroll
    for (int e = 0; e < NC; ++e) s_grp[(span >= 64 ? g : wave) * span * NC + c + e] = acc[e];
  }
  __syncthreads();
  float best = -INFINITY;
  int arg = 0x7fffffff;
  if (tid < V) {
    float v = s_grp[tid];
    for (int r = 1; r < rows; ++r) v += s_grp[r * span * NC + tid];
    logits[(long)b * V + tid] = v;
    if (v > best) {
      best = v;
      arg = tid;
    }
  }
  if (!next) return;  // uniform
  for (int o = 32; o > 0; o >>= 1) {
    const float ob = __shfl_xor(best, o);
    const int oa = __shfl_xor(arg, o);
    if (ob > best || (ob == best && oa < arg)) {
      best = ob;
      arg = oa;
    }
  }
  if (lane == 0) {
    s_best[wave] = best;
    s_arg[wave] = arg;
  }
  __syncthreads();
  if (tid == 0) {
    for (int w = 1; w * 64 < V; ++w)  // the waves that hold columns
      if (s_best[w] > best || (s_best[w] == best && s_arg[w] < arg)) {
        best = s_best[w];
        arg = s_arg[w];
      }
    next[b] = arg == 0x7fffffff ? 0 : arg;
  }
}

// The same without the greedy token, which is all that needs a sequence's logits in one place: a workgroup per 64 columns,
// which redoes the second stage as phase A does.  Bound by its launch and one trip to memory (d = 256, V = 256, one sequence:
// 3.5 us, 6.3 where one CU fetched all 256 KiB of lm_head).
template <int DC, int NW>
__global__ __launch_bounds__(NW * 64, 2) void k_phase_logits(const float *__restrict__ cur_in,
                                                             const float *__restrict__ dec_partial, int G, int B, int d,
                                                             const float *__restrict__ lm_head, int V,
                                                             float *__restrict__ logits) {
  using S = Shape<DC, NW, 64>;
  __shared__ float4 s_part[S::NT];
  __shared__ __align__(16) float s_cur[NW][DC];
  __shared__ __align__(16) float s_acc[NW][64];
  const int lane = threadIdx.x & 63, wave = wave_id(), b = blockIdx.y;
  const int base = min((int)blockIdx.x * 64, V - 64);  // the last block may make some of its neighbour's columns again, alike

  RowSum<DC, NW> partials;
  partials.ask(dec_partial + (long)b * d, (long)B * d, G, d);
  float cur[S::CJ];
#pragma unroll
  for (int j = 0; j < S::CJ; ++j) cur[j] = cur_in[(long)b * d + min(j * 64 + lane, d - 1)];
  Project<DC, NW, 64> head;
  head.ask(lm_head + base, d, V);
  __builtin_amdgcn_sched_barrier(0);

  float mlp[S::CJ];
  partials.collect(G, s_part, mlp);
  wave_layer_norm<S::CJ>(mlp, d);
#pragma unroll
  for (int j = 0; j < S::CJ; ++j) cur[j] = cur[j] + mlp[j];
  wave_layer_norm<S::CJ>(cur, d);
#pragma unroll
  for (int j = 0; j < S::CJ; ++j) s_cur[wave][j * 64 + lane] = j * 64 + lane < d ? cur[j] : 0.0f;
  wave_lds_order();
  const float v = head.dot(s_cur[wave], d, s_acc);
  if (wave == 0) logits[(long)b * V + base + lane] = v;
}

// The two launches of a layer.
template <int DC, int NW, int NB, typename RhoT, bool AHEAD>
void launch_phase_a(hipStream_t stream, dim3 grid, bool first, const PhaseArgs &a) {
  if (first) hipLaunchKernelGGL((k_layer_phase_a<DC, NW, NB, RhoT, AHEAD, true>), grid, dim3(NW * 64), 0, stream, a);
  else hipLaunchKernelGGL((k_layer_phase_a<DC, NW, NB, RhoT, AHEAD, false>), grid, dim3(NW * 64), 0, stream, a);
}
template <int DC, int NW, int NB>
void launch_layer(hipStream_t stream, dim3 grid, int rho_dtype, bool ahead, bool first, const PhaseArgs &a) {
  if (rho_dtype == BDH_BF16) {
    if (ahead) launch_phase_a<DC, NW, NB, unsigned short, true>(stream, grid, first, a);
    else launch_phase_a<DC, NW, NB, unsigned short, false>(stream, grid, first, a);
  } else {
    if (ahead) launch_phase_a<DC, NW, NB, float, true>(stream, grid, first, a);
    else launch_phase_a<DC, NW, NB, float, false>(stream, grid, first, a);
  }
  hipLaunchKernelGGL((k_layer_phase_b<DC, NW, NB>), grid, dim3(NW * 64), 0, stream, a);
}

}  // namespace

bool bdh_model_phase_fits(const bdh_model *m) {
  const bdh_model_config &c = m->cfg;
  if (c.rotary != BDH_ROPE && c.rotary != BDH_ALIBI && c.rotary != BDH_POPE) return false;
  if (c.n_embd < 128 || c.n_embd > 512 || (c.n_embd & 3) != 0) return false;
  if (c.latent < 32 || (c.latent & 31) != 0) return false;  // whole blocks of 64 or 32 neurons
  if (c.n_head < 1 || c.n_head > 64 || c.n_layer < 1) return false;
  // every workgroup of a sequence sums the partials of all the others: only while those are few
  return (long)c.n_head * (c.latent / ((c.latent & 63) == 0 ? 64 : 32)) <= 64;
}

// Neurons of a workgroup's block.  A head whose N is no multiple of 64 takes 32.  For the others: fewer neurons share the
// bytes that a CU has to fetch among more CUs and make more partials, which every workgroup adds up: 32 while those blocks
// number at most 64 and every workgroup has a CU to itself, 64 otherwise (us a step, 32 | 64: 4 layers of 1024 neurons, d =
// 256, 1 sequence 46 | 52, 8 sequences (256 workgroups) 52 | 56, 16 sequences 66 | 61; 8 layers of 2048, d = 512, 1 sequence
// 114 | 131, 4 sequences 134 | 146, 8 sequences 223 | 172).
static int block_neurons(const bdh_ctx *ctx, const bdh_model_config &c, int B) {
  const long n_cu = ctx->n_cu > 0 ? ctx->n_cu : 256, blocks = (long)c.n_head * c.latent / 32;
  return (c.latent & 63) != 0 || (blocks <= 64 && blocks * B <= n_cu) ? 32 : 64;
}

// Whether the two-launch layer is the fastest form of a decode step of B sequences: while batch x weights of a layer (every
// workgroup streams its share once per sequence) stay below a bound in MiB from measurement.  The other forms leave out more of
// what inactive neurons do not need, so each line was looked for with half of the neurons firing and with a twentieth (one
// figure below where every state row is visited whatever fires: PoPE, and ALiBi not lazily decayed).  Time of the other form
// over that of two launches, half | a twentieth, at so many MiB.  Kernel by kernel:
//   f32, d = 256 RoPE 288: 1.02 | 0.92, 336: 0.99 | 0.83; ALiBi 384: 1.06; PoPE 384: 0.94 to 1.07.  d = 512 RoPE 288: 1.05 | 1.01, 320: 0.95 | 0.84.
//     A row between 256 and 512 columns is work for 512: d = 384 RoPE 216: 1.13 | 0.98, 288: 0.98 | 0.82
//   bf16, d = 256 and 512 (for which the state step has fast kernels) RoPE 192: 1.00 to 1.14 | 0.98 to 1.26, 224: 0.90 to 0.95 | 0.89 to
//     0.98; ALiBi 224: 0.98 to 1.05, 256: 0.97; lazily decayed 288: 1.28 to 1.81 | 1.07 to 1.34, 381: 1.50 | 0.95, d = 512 576: 1.70 | 1.05.
//     Other d: d = 192 RoPE 250: 1.44 | 0.93, ALiBi 284: 1.38, PoPE 284: 2.2; d = 384 RoPE 256: 1.23 | 0.97
//   d = 128, 384: f32 1.11 | 1.02, bf16 1.71 | 1.15; lazily decayed bf16 480: 1.83 | 1.1
//   an odd number of 32-neuron blocks per head, which are not taken two at a time: f32 RoPE 144: 1.39 | 1.26, 160: 1.01 | 0.85; bf16
//     162: 1.36 | 0.94; PoPE and ALiBi 192: 1.2 to 1.5
// One launch for the whole step, where that is the other form: a CU spends it on its sequence's w MiB a layer, and takes the
// next sequence when it has done one.  w = 0.19 RoPE 48: 1.05 | 1.12, 96 (512 sequences) 1.41 | 1.56; w = 0.38 64: 1.01 | 1.05, 80: 0.99 | 0.98;
//   w = 0.75 80: 1.15 | 1.09, 96: 1.10 | 1.08, 112: 0.96 | 0.93; w = 1.1 96: 1.12 | 1.04, 112: 1.00 | 0.93; w = 1.7 135: 1.22 | 1.06, 162: 1.01 | 0.90,
//   PoPE 236: 1.08; w = 3 225: 1.37 | 1.31; odd blocks w = 0.28 45: 1.06 | 1.07, w = 0.84 64: 1.08 | 0.99, 80: 0.96 | 0.86
bool bdh_model_phase_pays(const bdh_model *m, int B, int rho_dtype, bool lazy) {
  const bdh_model_config &c = m->cfg;
  const int d = c.n_embd;
  const double w = sizeof(float) * 3.0 * c.n_head * c.latent * d / (1 << 20), mib = w * B;
  const bool bf16 = rho_dtype == BDH_BF16, odd = (c.latent & 63) != 0;
  const bool pope = c.rotary == BDH_POPE, eager = c.rotary == BDH_ALIBI && !lazy;
  double kernels;
  if (odd) kernels = bf16 || pope || eager ? 192 : 144;
  else if (d <= 128) kernels = bf16 && lazy ? 480 : 384;
  else if (!bf16) kernels = pope ? 384 : d > 256 ? d * 9 / 16 : eager ? 384 : 288;
  else if (lazy) kernels = d == 256 ? 380 : d == 512 ? 576 : d > 256 ? d * 9 / 16 : 256;
  else if (d == 256 || d == 512) kernels = eager ? 224 : 192;
  else kernels = pope || eager ? 288 : 256;
  if (B > 65535 || mib > kernels) return false;
  const int from_one = bdh_model_one_launch_from(c), n_cu = m->ctx->n_cu > 0 ? m->ctx->n_cu : 256;
  if (from_one == 0 || B < from_one) return true;
  const double one = pope || eager ? 20 + 110 * w : std::max(36 + 60 * w, std::min(44 + 70 * w, 96.0));
  return mib <= (odd ? 0.71 : 1.0) * one * ((B + n_cu - 1) / n_cu);
}

size_t bdh_model_phase_scratch_floats(const bdh_model *m, int B) {
  const bdh_model_config &c = m->cfg;
  const size_t d = c.n_embd, cols = (size_t)c.n_head * c.latent, G = cols / block_neurons(m->ctx, c, B);
  // cur ping-pong | x | readout partials | encoder partials
  return 2 * bdh_align_up((size_t)B * d, 64) + bdh_align_up((size_t)B * cols, 64) + bdh_align_up((size_t)B * G * d, 64) +
         bdh_align_up(G * (size_t)B * d, 64);
}

// On return cur_final points at the buffer holding the last layer's input and dec_partial at its encoder partials
// [G][B][d]: the caller runs the encoder's second stage and the head.
int bdh_launch_model_phases(bdh_model *m, const int64_t *tokens, int B, float *scratch, void *rho, int rho_dtype,
                            int32_t *stamps, int64_t position,
                            const int32_t *positions_dev, float **cur_final, float **dec_partial, int *G_out) {
  bdh_ctx *ctx = m->ctx;
  const bdh_model_config &c = m->cfg;
  if (!bdh_model_phase_fits(m)) return bdh_fail(ctx, BDH_E_SHAPE, "model does not fit the two-launch layer");
  const int d = c.n_embd, h = c.n_head, N = c.latent, L = c.n_layer;
  const int nb = block_neurons(ctx, c, B);
  const size_t cols = (size_t)h * N, G = cols / nb;
  if (B > 65535) return bdh_fail(ctx, BDH_E_SHAPE, "grid too large");
  const dim3 grid((unsigned)(N / nb), (unsigned)h, (unsigned)B);
  float *cur[2] = {scratch, scratch + bdh_align_up((size_t)B * d, 64)};
  float *x = cur[1] + bdh_align_up((size_t)B * d, 64);
  float *attn_partial = x + bdh_align_up((size_t)B * cols, 64);
  float *dpart = attn_partial + bdh_align_up((size_t)B * G * d, 64);
  const size_t Nq = c.rotary == BDH_POPE ? 2 * (size_t)N : (size_t)N;
  PhaseArgs a{};
  a.x = x;
  a.attn_partial = attn_partial;
  a.dec_partial_out = dpart;
  a.enc = m->w.encoder;
  a.enc_v = m->w.encoder_v;
  a.dec = m->w.decoder;
  a.freqs = m->freqs;
  a.pos_dev = positions_dev;
  a.pos = (long)position;
  a.B = B;
  a.d = d;
  a.h = h;
  a.N = N;
  a.rotary = c.rotary;
  a.thr = c.relu_threshold;
  if (c.rotary == BDH_ALIBI)
    for (int i = 0; i < h; ++i) {
      a.decay[i] = expf(-m->slopes[i]);                 // src/model/attention.rs:181-186
      a.log_decay[i] = (float)log((double)a.decay[i]);  // of the rounded factor, as the lazy state step
    }
  // Phase A asks for all state rows ahead where every row is visited anyway, and where the rows are bf16 and short: half the
  // bytes, so the rows that were asked for in vain cost less than the trip (us a step, ahead | visited rows only: d = 256,
  // 64 blocks, RoPE, 16 sequences bf16 199 | 211, f32 256 | 255; 128 neurons per head, d = 128, f32 44 | 39; PoPE 42 | 43).
  const bool dense = c.rotary == BDH_POPE || (c.rotary == BDH_ALIBI && !stamps);
  const bool ahead = dense || (rho_dtype == BDH_BF16 && (nb == 32 || (d > 128 && d <= 256)));
  int in = 0;  // cur[in] is the layer's input; a layer with a pending second stage writes cur[in ^ 1]
  a.embed = m->w.embed;
  a.V = c.vocab;
  for (int l = 0; l < L; ++l) {
    a.tokens = l == 0 ? tokens : nullptr;  // the first layer makes its own input and leaves it in cur[0]
    a.cur_in = cur[in];
    a.cur_out = l == 0 ? cur[0] : cur[in ^ 1];
    a.dec_partial = l > 0 ? dpart : nullptr;
    a.rho = static_cast<char *>(rho) + (size_t)l * B * h * Nq * d * (rho_dtype == BDH_BF16 ? 2 : 4);
    a.stamps = stamps ? stamps + (size_t)l * B * h * N : nullptr;
#define BDH_PHASE(DC_, NW_)                                                                              \
  do {                                                                                                   \
    if (nb == 64) launch_layer<DC_, NW_, 64>(ctx->stream, grid, rho_dtype, ahead, l == 0, a);            \
    else launch_layer<DC_, NW_, 32>(ctx->stream, grid, rho_dtype, ahead, l == 0, a);                     \
  } while (0)
    if (d <= 128) BDH_PHASE(128, 4); else if (d <= 256) BDH_PHASE(256, 8); else BDH_PHASE(512, 8);
#undef BDH_PHASE
    BDH_LAUNCH_CHECK(ctx, "k_layer_phase_a/b");
    if (l > 0) in ^= 1;  // phase A has applied the pending second stage: the layer's input is now cur[in ^ 1]
  }
  *cur_final = cur[in];
  *dec_partial = dpart;
  *G_out = (int)G;
  return BDH_OK;
}

// The last layer's second stage and the output head in one launch (V <= 1024).
int bdh_launch_phase_head(bdh_model *m, int B, const float *cur, const float *dec_partial, int G, float *logits,
                          int64_t *next_tokens) {
  bdh_ctx *ctx = m->ctx;
  const bdh_model_config &c = m->cfg;
  if (c.vocab > 1024 || c.n_embd > 512) return bdh_fail(ctx, BDH_E_SHAPE, "head kernel needs V <= 1024 and d <= 512");
  // Without a greedy token 64 columns a workgroup: one CU need not fetch all of lm_head (3.5 us where one workgroup takes
  // 6.3, V = 256).  Fewer columns than that leave a block's accesses beyond the row.
  if (!next_tokens && c.vocab >= 64 && G <= 64 && B <= 65535) {
    const dim3 grid((unsigned)((c.vocab + 63) / 64), (unsigned)B);
#define BDH_LOGITS(DC_, NW_)                                                                                               \
  hipLaunchKernelGGL((k_phase_logits<DC_, NW_>), grid, dim3(NW_ * 64), 0, ctx->stream, cur, dec_partial, G, B, c.n_embd,   \
                     m->w.lm_head, c.vocab, logits)
    if (c.n_embd <= 128) BDH_LOGITS(128, 4); else if (c.n_embd <= 256) BDH_LOGITS(256, 8); else BDH_LOGITS(512, 8);
#undef BDH_LOGITS
    BDH_LAUNCH_CHECK(ctx, "k_phase_logits");
    return BDH_OK;
  }
#define BDH_HEAD(DC_, NC_)                                                                                                 \
  hipLaunchKernelGGL((k_phase_head<DC_, NC_>), dim3((unsigned)B), dim3(1024), 0, ctx->stream, cur, dec_partial, G, B,      \
                     c.n_embd, m->w.lm_head, c.vocab, logits, next_tokens)
#define BDH_HEAD_OF(NC_)                                                                                                   \
  do {                                                                                                                     \
    if (c.n_embd <= 128) BDH_HEAD(128, NC_); else if (c.n_embd <= 256) BDH_HEAD(256, NC_); else BDH_HEAD(512, NC_);        \
  } while (0)
  if (c.vocab >= 4) BDH_HEAD_OF(4); else BDH_HEAD_OF(1);
#undef BDH_HEAD_OF
#undef BDH_HEAD
  BDH_LAUNCH_CHECK(ctx, "k_phase_head");
  return BDH_OK;
}
