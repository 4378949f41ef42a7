// The recurrences over matrix states that a prompt brings, sixteen tokens at a time on the 32-bit matrix cores: the gated
// delta rule (a decay per head or per key channel), gated linear attention and the matrix memory of an mLSTM layer
// (formulas at their token-by-token kernels in sequence_ops.hip, which serve decode steps, 32-bit models and other sizes).
//
// With S the state that enters a chunk, d_t the decay of token t (a number or a vector over key channels), cp_t the product
// of the chunk's decays up to and with t, and E_ts the product of those behind s up to and with t, the recurrence unrolls to
//   u = T (V - Kt S),   Kt_t = cp_t k_t,   T = (1 + diag(beta) A)^-1 diag(beta),   A_ts = k_t . (E_ts k_s) for s < t
//   O = Qt S + P u,     Qt_t = cp_t q_t,   P_ts = q_t . (E_ts k_s) for s <= t
//   S <- cp_C S + Kh^T u,   Kh_s = E_Cs k_s                                       (C: the chunk's last token)
// without the delta u is V (rows weighted with what is taken of them go into P and Kh).  Decays are multiplied, never
// divided by or taken as differences of sums of logarithms, so every factor is as exact as in the token-by-token walk and
// nothing can overflow.  Everything is 32-bit.
//
//   * chunk_prepare_kernel, a block a (chunk, head): Kt, Qt, Kh^T, P, T and cp_C into a workspace, all chunks side by side;
//   * chunk_walk_kernel, a block of four waves a (request, head, 16 columns of S): the chunks in order.  A wave keeps dk / 4
//     rows of S as accumulators of its MFMAs, whose layout is that of the operand of the products with S (step i of an
//     MFMA takes rows 4 g + i), so S never leaves its registers; the waves' parts of Kt S and Qt S meet in LDS behind the
//     one barrier of a chunk, then every wave forms u for itself, again operand for operand in registers.  A chunk's
//     operands are asked for two chunks ahead.  A chunk with values that are not finite takes its two triangular products row
//     by row (causal_product): a token's infinity reaches itself and later ones alone, as in the walk.  (The look at every
//     chunk's values costs the delta rules 1 to 2%: 2,048 tokens 240 -> 242 us in all, 4 x 3,000 1,532 -> 1,561.)
// What bounds it: the walk, a chain of one chunk behind the other, about 1.7 us each, of which 16 + 4 + 8 MFMAs of 32 cycles are
// 0.4; the rest is the way through LDS, the barrier and the operands' loads.  A prompt of 2,048 tokens with 32 heads of 128 takes
// 40 + 219 us with the rule of a decay per head (token by token 1,242, 16 columns a block), eight prompts of 1,804 tokens 63 + 137 us
// with a decay per channel (816) and 24 + 32 + 143 us as matrix memory (634).  Against 64 bits the states of 32 heads (rows of
// 40 to 600 tokens, all four kinds) are 0.90 to 1.01 times as far as the walk's; of two heads alone up to 1.27 times, by chance.
// The workspace grows with the rows: a step's tokens are taken in windows (the state goes through memory between them), and it
// holds a slot for every 16 tokens of a window and one more for every row of the step.  The caller bounds it, or walks.
#include "common.h"
#include "recurrence.h"

namespace {

constexpr int kChunk = 16;
enum : int { kRuleHead = 0, kRuleChannel = 1, kRulePlain = 2, kRuleMemory = 3 };

__device__ __forceinline__ float sigmoid_c(float z) { return 1.0f / (1.0f + expf(-z)); }
__device__ __forceinline__ float softplus_c(float z) { return fmaxf(z, 0.f) + log1pf(expf(-fabsf(z))); }
__device__ __forceinline__ float log_sigmoid_c(float z) { return fminf(z, 0.f) - log1pf(expf(-fabsf(z))); }

// A product of decays with what its roundings lose, so that sixteen factors are rounded once.
struct Product {
  float hi = 1.f, lo = 0.f;
  __device__ __forceinline__ void times(float d) {
    const float p = hi * d;
    lo = fmaf(lo, d, fmaf(hi, d, -p));
    hi = p;
  }
  __device__ __forceinline__ float value() const { return hi + lo; }
};

// The sum over the 16 lanes of a row of lanes, by moves within the row; every lane gets the same bits.
__device__ __forceinline__ float sum_of_sixteen_lanes(float v) {
  v = sum_of_eight_lanes(v);
  return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x140, 0xf, 0xf, false));
}

// Floats of a (chunk, head) in the workspace, and where its parts begin.
template <int DK>
struct Part {
  static constexpr int kKt = 0, kQt = kChunk * DK, kKh = 2 * kChunk * DK, kLast = 3 * kChunk * DK, kP = kLast + DK, kT = kP + kChunk * kChunk;
  static constexpr int kFloats = kT + kChunk * kChunk;
};

struct ChunkArgs {
  const bf16_t* q;       // rows of tokens: queries at q + h_k * dk, keys at k, values at v + h * dv
  const bf16_t* k;
  const bf16_t* v;
  int stride;            // elements from a token's row to the next
  const bf16_t* proj;    // pre-activations of beta (b_off + h) and of a decay per head (a_off + h)
  int proj_stride, b_off, a_off;
  const float* A_log;
  const float* dt_bias;
  const float* a_ch;     // pre-activations of a decay per channel [token][a_stride]
  int a_stride;
  float plain_rate;
  float* gates;          // matrix memory: [token of the window][H][3]: log keep, log take, maximum
  int i_off, f_off;      // matrix memory: columns of the gates' pre-activations behind q
  const float* i_bias;
  const float* f_bias;
  float cap;
  float* state;
  long long state_stride;
  const int32_t* qo_indptr;
  const int32_t* slot_ids;
  int rows;
  int H, G, dv;
  int w0, w1;            // the window of tokens
  float* ws;
  float* o_raw;          // [token][H][dv]
  float* den;            // matrix memory: [token][H]
};

// Tokens of a row inside the window, counted from the window's start, and the row's first slot of the workspace: rows need
// ceil(length / 16) slots each, and floor(start / 16) + row leaves room for them.
__device__ __forceinline__ int in_window(int t, const ChunkArgs& g) { return min(max(t, g.w0), g.w1) - g.w0; }
__device__ __forceinline__ int first_slot(int row, const ChunkArgs& g) { return in_window(g.qo_indptr[row], g) / kChunk + row; }

// ----------------------------------------------------------------------------- matrix memory: maxima
// m_t = max(f_t + m_(t-1), i_t): a wave takes 64 tokens of a (request, head) at a time, a lane the gates of one; then all
// lanes walk the chain of additions and comparisons, token after token as the kernels for single tokens do.  (Scanned over
// the lanes in six steps, sums of forget gates that later cancel cost the maximum three digits.)
__device__ __forceinline__ float lane_value(float v, int lane) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane)); }
__global__ void __launch_bounds__(256) memory_gates_kernel(const ChunkArgs g, int dk) {
  const int h = blockIdx.x * 4 + threadIdx.x / kWave, lane = threadIdx.x % kWave;
  const int row = blockIdx.y;
  if (h >= g.H) return;
  const int start = in_window(g.qo_indptr[row], g), end = in_window(g.qo_indptr[row + 1], g);
  const int W = g.dv + 1;
  float m = g.state[(long long)g.slot_ids[row] * g.state_stride + (size_t)g.H * W * dk + (size_t)h * W];
  for (int t0 = start; t0 < end; t0 += kWave) {
    const int t = t0 + lane;
    const bool in = t < end;
    const bf16_t* at = g.q + (size_t)(g.w0 + min(t, end - 1)) * g.stride;
    const float gi = g.cap * tanhf((to_f32(at[g.i_off + h]) + g.i_bias[h]) / g.cap);
    const float gf = log_sigmoid_c(g.cap * tanhf((to_f32(at[g.f_off + h]) + g.f_bias[h]) / g.cap));
    // (past the row's end: nothing kept of the forget gate's, nothing from the input gate)
    const float f = in ? gf : 0.f, i = in ? gi : -INFINITY;
    float mt = m, before = m;
#pragma unroll
    for (int l = 0; l < kWave; ++l) {
      const float entered = m;
      m = fmaxf(lane_value(f, l) + m, lane_value(i, l));
      if (lane == l) {
        mt = m;
        before = entered;
      }
    }
    if (in) {
      float* to = g.gates + ((size_t)t * g.H + h) * 3;
      to[0] = gf + before - mt;
      to[1] = gi - mt;
      to[2] = mt;
    }
  }
}

// ----------------------------------------------------------------------------- a chunk by itself
template <int DK, int RULE>
__global__ void __launch_bounds__(256) chunk_prepare_kernel(const ChunkArgs g) {
  constexpr bool kChannel = RULE == kRuleChannel || RULE == kRulePlain, kDelta = RULE == kRuleHead || RULE == kRuleChannel;
  constexpr int kPitch = DK + 4, kPer = DK / 16;  // channels of a thread
  static_assert(kPer % 4 == 0, "whole float4s");
  using P = Part<DK>;
  __shared__ __attribute__((aligned(16))) float k_l[kChunk][kPitch];
  __shared__ __attribute__((aligned(16))) float q_l[kChunk][kPitch];
  __shared__ __attribute__((aligned(16))) float d_l[kChannel ? kChunk : 1][kPitch];  // decays
  __shared__ float dec_l[kChunk], take_l[kChunk], beta_l[kChunk];
  __shared__ float a_l[kChunk][kChunk + 1];  // beta_t A_ts
  const int tid = threadIdx.x, lane = tid % kWave;
  const int slot = blockIdx.x, h = blockIdx.y;
  int row = -1;  // the last row whose first slot is not beyond this one
  for (int r0 = 0; r0 < g.rows; r0 += kWave) {
    const bool at_or_before = r0 + lane < g.rows && first_slot(min(r0 + lane, g.rows - 1), g) <= slot;
    const int n = __popcll(__ballot(at_or_before));
    row += n;
    if (n < kWave) break;
  }
  if (row < 0) return;
  const int start = in_window(g.qo_indptr[row], g), end = in_window(g.qo_indptr[row + 1], g);
  const int t0 = start + (slot - first_slot(row, g)) * kChunk;
  if (t0 >= end) return;
  const int nt = min(kChunk, end - t0);
  float* out = g.ws + ((size_t)slot * g.H + h) * P::kFloats;

  // keys and queries, scaled; 16 threads a token; tokens past the row's end are zeros that decay nothing
  {
    const int t = tid / 16, d0 = (tid % 16) * kPer;
    const size_t at = (size_t)(g.w0 + t0 + min(t, nt - 1)) * g.stride + (h / (g.H / g.G)) * DK + d0;
    float kk[kPer], qq[kPer], k2 = 0.f, q2 = 0.f;
#pragma unroll
    for (int u = 0; u < kPer; u += 4) {
      const Four<bf16_t> k4 = *reinterpret_cast<const Four<bf16_t>*>(g.k + at + u), q4 = *reinterpret_cast<const Four<bf16_t>*>(g.q + at + u);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        kk[u + e] = to_f32(k4.e[e]);
        qq[u + e] = to_f32(q4.e[e]);
        k2 = fmaf(kk[u + e], kk[u + e], k2);
        q2 = fmaf(qq[u + e], qq[u + e], q2);
      }
    }
    float ks = 1.f, qs = 1.0f / sqrtf((float)DK);
    if constexpr (kDelta) {
      ks = 1.0f / sqrtf(sum_of_sixteen_lanes(k2) + 1e-6f);
      qs /= sqrtf(sum_of_sixteen_lanes(q2) + 1e-6f);
    }
    if (t >= nt) ks = qs = 0.f;
#pragma unroll
    for (int u = 0; u < kPer; u += 4) {
      *reinterpret_cast<float4*>(&k_l[t][d0 + u]) = t < nt ? float4{kk[u] * ks, kk[u + 1] * ks, kk[u + 2] * ks, kk[u + 3] * ks} : float4{0.f, 0.f, 0.f, 0.f};
      *reinterpret_cast<float4*>(&q_l[t][d0 + u]) = t < nt ? float4{qq[u] * qs, qq[u + 1] * qs, qq[u + 2] * qs, qq[u + 3] * qs} : float4{0.f, 0.f, 0.f, 0.f};
    }
  }
  if (tid < kChunk) {
    const bool in = tid < nt;
    const size_t t = (size_t)t0 + min(tid, nt - 1);
    if constexpr (kDelta) beta_l[tid] = in ? sigmoid_c(to_f32(g.proj[(g.w0 + t) * g.proj_stride + g.b_off + h])) : 0.f;
    if constexpr (RULE == kRuleHead)
      dec_l[tid] = in ? expf(-expf(g.A_log[h]) * softplus_c(to_f32(g.proj[(g.w0 + t) * g.proj_stride + g.a_off + h]) + g.dt_bias[h])) : 1.f;
    if constexpr (RULE == kRuleMemory) {
      dec_l[tid] = in ? expf(g.gates[(t * g.H + h) * 3]) : 1.f;
      take_l[tid] = in ? expf(g.gates[(t * g.H + h) * 3 + 1]) : 0.f;
    }
  }
  if constexpr (kChannel) {
    const float rate = RULE == kRulePlain ? 0.f : -expf(g.A_log[h]);
    for (int e = tid; e < kChunk * DK; e += 256) {
      const int t = e / DK, d = e % DK;
      const float pre = g.a_ch[(size_t)(g.w0 + t0 + min(t, nt - 1)) * g.a_stride + h * DK + d] + g.dt_bias[h * DK + d];
      const float dec = RULE == kRulePlain ? expf(g.plain_rate * log_sigmoid_c(pre)) : expf(rate * softplus_c(pre));
      d_l[t][d] = t < nt ? dec : 1.f;
    }
  }
  __syncthreads();

  // A and P: thread (s, piece of the channels) carries w = E_ts k_s along t; the 16 pieces are neighbouring lanes
  {
    const int s = tid / kWave + 4 * (lane / 16), d0 = (lane % 16) * kPer;  // (a wave's four s are spread, so that waves do alike)
    float w[kPer], scale = 1.f;
#pragma unroll
    for (int u = 0; u < kPer; ++u) w[u] = k_l[s][d0 + u];
    if constexpr (RULE == kRuleMemory) scale = take_l[s];
    float p_mine = 0.f, a_mine = 0.f;  // of t = lane % 16
#pragma unroll 4
    for (int t = 0; t < kChunk; ++t) {
      const bool behind = t > s;
      float ks = 0.f, qs = 0.f;
      if constexpr (!kChannel) scale *= behind ? dec_l[t] : 1.f;
#pragma unroll
      for (int u = 0; u < kPer; u += 4) {
        const float4 q4 = *reinterpret_cast<const float4*>(&q_l[t][d0 + u]);
        const float qv[4] = {q4.x, q4.y, q4.z, q4.w};
        float kv[4] = {0.f, 0.f, 0.f, 0.f}, dv[4] = {1.f, 1.f, 1.f, 1.f};
        if constexpr (kDelta) {
          const float4 k4 = *reinterpret_cast<const float4*>(&k_l[t][d0 + u]);
          kv[0] = k4.x; kv[1] = k4.y; kv[2] = k4.z; kv[3] = k4.w;
        }
        if constexpr (kChannel) {
          const float4 d4 = *reinterpret_cast<const float4*>(&d_l[t][d0 + u]);
          dv[0] = d4.x; dv[1] = d4.y; dv[2] = d4.z; dv[3] = d4.w;
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if constexpr (kChannel) w[u + e] *= behind ? dv[e] : 1.f;
          if constexpr (kDelta) ks = fmaf(kv[e], w[u + e], ks);
          qs = fmaf(qv[e], w[u + e], qs);
        }
      }
      qs = sum_of_sixteen_lanes(qs) * scale;
      if constexpr (kDelta) ks = sum_of_sixteen_lanes(ks) * scale;
      if (lane % 16 == t) {
        p_mine = t >= s ? qs : 0.f;
        a_mine = behind ? ks : 0.f;
      }
    }
    const int t = lane % 16;
    out[P::kP + t * kChunk + s] = p_mine;
    if constexpr (kDelta) a_l[t][s] = beta_l[t] * a_mine;
  }
  // Kt, Qt and cp_C: a thread walks its channel's decays; Kh^T the other way round
  if (tid < DK) {
    Product cp;
#pragma unroll
    for (int t = 0; t < kChunk; ++t) {
      cp.times(kChannel ? d_l[kChannel ? t : 0][tid] : dec_l[t]);
      if constexpr (kDelta) out[P::kKt + t * DK + tid] = cp.value() * k_l[t][tid];
      out[P::kQt + t * DK + tid] = cp.value() * q_l[t][tid];
    }
    out[P::kLast + tid] = cp.value();
  } else if (tid < 2 * DK) {
    const int d = tid - DK;
    Product cp;
    float kh[kChunk];
#pragma unroll
    for (int s = kChunk - 1; s >= 0; --s) {
      kh[s] = cp.value() * (RULE == kRuleMemory ? take_l[s] : 1.f) * k_l[s][d];
      cp.times(kChannel ? d_l[kChannel ? s : 0][d] : dec_l[s]);
    }
#pragma unroll
    for (int s = 0; s < kChunk; s += 4) *reinterpret_cast<float4*>(out + P::kKh + d * kChunk + s) = float4{kh[s], kh[s + 1], kh[s + 2], kh[s + 3]};
  }
  if constexpr (kDelta) {
    __syncthreads();
    if (tid < kChunk) {  // column tid of T by forward substitution
      float x[kChunk];
#pragma unroll
      for (int t = 0; t < kChunk; ++t) {
        float v = t == tid ? beta_l[t] : 0.f;
#pragma unroll
        for (int s = 0; s < t; ++s) v = fmaf(-a_l[t][s], x[s], v);
        x[t] = v;
        out[P::kT + t * kChunk + tid] = v;
      }
    }
  }
}

// ----------------------------------------------------------------------------- the chunks in order
__device__ __forceinline__ bool finite(float v) { return fabsf(v) < INFINITY; }
__device__ __forceinline__ bool all_finite(const f32x4_t& v) { return finite(v[0]) & finite(v[1]) & finite(v[2]) & finite(v[3]); }

// acc + L x as four MFMAs give it (step i takes the rows 4 g + i in ascending order), for L zero above its diagonal, but row t
// over the rows s <= t alone: the zeros above the diagonal times a later token's infinity would be NaN.  Operands and result
// lie as the MFMAs have them: lane 16 g + r holds L[r][4 g ..+ 3], and of x, acc and the result rows 4 g ..+ 3 of column r.  What
// is not finite in an earlier row (with `own` in row t itself too) makes the result NaN, as infinities of both signs do that
// a walk adds up channel by channel.
__device__ __forceinline__ f32x4_t causal_product(const f32x4_t& l, const f32x4_t& x, f32x4_t acc, bool own, int lane) {
  const int n16 = lane % 16, g4 = lane / 16;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll 1
    for (int g = 0; g < 4; ++g) {
      const int s = 4 * g + i;
      const float xs = __shfl(x[i], 16 * g + n16, kWave);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int t = 4 * g4 + j;
        const float ls = __shfl(l[i], 16 * g + t, kWave);
        if (s <= t) acc[j] = finite(xs) || (s == t && !own) ? fmaf(ls, xs, acc[j]) : NAN;
      }
    }
  return acc;
}

template <int DK, int RULE>
__global__ void __launch_bounds__(256, 2) chunk_walk_kernel(const ChunkArgs g, int column_groups) {
  constexpr bool kDelta = RULE == kRuleHead || RULE == kRuleChannel, kMemory = RULE == kRuleMemory;
  constexpr int KT = DK / 64;  // 16-row tiles of S a wave holds
  using P = Part<DK>;
  __shared__ __attribute__((aligned(16))) f32x4_t parts[2][4][kDelta ? 2 : 1][kWave];
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  const int n16 = lane % 16, g4 = lane / 16;
  // blocks go to the eight XCDs in turn: with heads in eights all column groups of a head share an XCD, whose L2 then holds
  // what they all read
  int h, cg;
  if (g.H % 8 == 0) {
    const int j = blockIdx.x / 8;
    cg = j % column_groups;
    h = blockIdx.x % 8 + 8 * (j / column_groups);
  } else {
    h = blockIdx.x / column_groups;
    cg = blockIdx.x % column_groups;
  }
  const int row = blockIdx.y;
  const int start = in_window(g.qo_indptr[row], g), end = in_window(g.qo_indptr[row + 1], g);
  if (start >= end) return;
  const int chunks = (end - start + kChunk - 1) / kChunk;
  const int W = g.dv + (kMemory ? 1 : 0);  // columns of S (the memory's normaliser is one more)
  const int col = cg * 16 + n16;
  const bool live = col < W;
  float* st = g.state + (long long)g.slot_ids[row] * g.state_stride;
  float* column = st + ((size_t)h * W + min(col, W - 1)) * DK + wave * KT * 16 + 4 * g4;
  f32x4_t S[KT];
#pragma unroll
  for (int x = 0; x < KT; ++x) S[x] = *reinterpret_cast<const f32x4_t*>(column + 16 * x);

  struct Operands {
    f32x4_t kt[kDelta ? KT : 1], qt[KT], kh[KT], last[KT], t, p;
    bf16_t v[4];
  };
  const float* chunk0 = g.ws + ((size_t)first_slot(row, g) * g.H + h) * P::kFloats;
  const bf16_t* values = g.v + (size_t)h * g.dv + min(col, g.dv - 1);
  auto load = [&](Operands& o, int c_raw) {
    const int c = min(c_raw, chunks - 1);
    const float* at = chunk0 + (size_t)c * g.H * P::kFloats;
#pragma unroll
    for (int x = 0; x < KT; ++x) {
      const int tile = (wave * KT + x) * 16;
      if constexpr (kDelta) o.kt[x] = *reinterpret_cast<const f32x4_t*>(at + P::kKt + n16 * DK + tile + 4 * g4);
      o.qt[x] = *reinterpret_cast<const f32x4_t*>(at + P::kQt + n16 * DK + tile + 4 * g4);
      o.kh[x] = *reinterpret_cast<const f32x4_t*>(at + P::kKh + (tile + n16) * kChunk + 4 * g4);
      o.last[x] = *reinterpret_cast<const f32x4_t*>(at + P::kLast + tile + 4 * g4);
    }
    if constexpr (kDelta) o.t = *reinterpret_cast<const f32x4_t*>(at + P::kT + n16 * kChunk + 4 * g4);
    o.p = *reinterpret_cast<const f32x4_t*>(at + P::kP + n16 * kChunk + 4 * g4);
#pragma unroll
    for (int i = 0; i < 4; ++i) o.v[i] = values[(size_t)(g.w0 + min(start + c * kChunk + 4 * g4 + i, end - 1)) * g.stride];
  };
  auto step = [&](const Operands& o, int c) {
    const int t0 = start + c * kChunk;
    const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
    f32x4_t pk = zero, pq = zero;
#pragma unroll
    for (int x = 0; x < KT; ++x)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if constexpr (kDelta) pk = mfma_f32(o.kt[x][i], S[x][i], pk);
        pq = mfma_f32(o.qt[x][i], S[x][i], pq);
      }
    // (two sets: a wave that is a chunk ahead writes the other one, and cannot be two ahead)
    parts[c & 1][wave][0][lane] = pq;
    if constexpr (kDelta) parts[c & 1][wave][1][lane] = pk;
    __syncthreads();
    f32x4_t u;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const bool in = t0 + 4 * g4 + i < end;
      u[i] = in ? (kMemory && col == g.dv ? 1.f : to_f32(o.v[i])) : 0.f;
    }
    if constexpr (kDelta) {
      f32x4_t ks = parts[c & 1][0][1][lane];
#pragma unroll
      for (int w = 1; w < 4; ++w) ks += parts[c & 1][w][1][lane];
      const f32x4_t r = u - ks;
      const bool odd = __ballot(!all_finite(r)) != 0;  // (of all lanes: every wave has the same r)
      u = zero;
#pragma unroll
      for (int i = 0; i < 4; ++i) u = mfma_f32(o.t[i], r[i], u);
#pragma unroll
      for (int x = 0; x < KT; ++x) S[x] *= o.last[x];  // (before the branch: while the MFMAs run)
      if (odd) u = causal_product(o.t, r, zero, false, lane);
    } else {
#pragma unroll
      for (int x = 0; x < KT; ++x) S[x] *= o.last[x];
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int x = 0; x < KT; ++x) S[x] = mfma_f32(o.kh[x][i], u[i], S[x]);
    if (wave == (c & 3)) {  // the waves take turns with the results
      f32x4_t out = parts[c & 1][0][0][lane];
#pragma unroll
      for (int w = 1; w < 4; ++w) out += parts[c & 1][w][0][lane];
      const f32x4_t before = out;
#pragma unroll
      for (int i = 0; i < 4; ++i) out = mfma_f32(o.p[i], u[i], out);
      if (__ballot(!all_finite(out))) out = causal_product(o.p, u, before, kMemory, lane);  // (its walk reads the state that has the token; the others add q . k u)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int t = t0 + 4 * g4 + i;
        if (t >= end || !live) continue;
        if (kMemory && col == g.dv)
          g.den[(size_t)(g.w0 + t) * g.H + h] = fmaxf(fabsf(out[i]), expf(-g.gates[((size_t)t * g.H + h) * 3 + 2])) + 1e-6f;
        else
          g.o_raw[((size_t)(g.w0 + t) * g.H + h) * g.dv + col] = out[i];
      }
    }
  };
  Operands a, b;
  load(a, 0);
  load(b, 1);
  for (int c = 0; c < chunks; c += 2) {
    step(a, c);
    load(a, c + 2);
    if (c + 1 < chunks) {
      step(b, c + 1);
      load(b, c + 3);
    }
  }
  if (live) {
#pragma unroll
    for (int x = 0; x < KT; ++x) *reinterpret_cast<f32x4_t*>(column + 16 * x) = S[x];
    if (kMemory && wave == 0 && g4 == 0) st[(size_t)g.H * W * DK + (size_t)h * W + col] = g.gates[((size_t)(end - 1) * g.H + h) * 3 + 2];
  }
}

// Tokens a window holds: what keeps the workspace of 32 heads of 128 channels near 110 MB, which the memory-side cache holds.
constexpr int kWindow = 2048;

template <int DK, int RULE>
int run_chunks(ChunkArgs g, int t_first, int t_last, hipStream_t stream) {
  const int W = g.dv + (RULE == kRuleMemory ? 1 : 0);
  const int column_groups = (W + 15) / 16;
  for (int w0 = t_first; w0 < t_last; w0 += kWindow) {
    g.w0 = w0;
    g.w1 = w0 + kWindow < t_last ? w0 + kWindow : t_last;
    const int slots = (g.w1 - w0) / kChunk + g.rows;
    if (RULE == kRuleMemory) memory_gates_kernel<<<dim3((g.H + 3) / 4, g.rows), 256, 0, stream>>>(g, DK);
    chunk_prepare_kernel<DK, RULE><<<dim3(slots, g.H), 256, 0, stream>>>(g);
    chunk_walk_kernel<DK, RULE><<<dim3(g.H * column_groups, g.rows), 256, 0, stream>>>(g, column_groups);
  }
  return tl_check_launch("delta_chunks");
}

}  // namespace

// Which calls the chunks take: keys of 64 or 128 channels, rows and offsets that let four channels be read at once, a
// workspace that holds a window.  ``floats`` of workspace are there, of which tl_chunk_floats tells the need.
TL_EXPORT long long tl_chunk_floats(int n_tokens, int rows, int H, int dk, int memory) {
  if (dk != 64 && dk != 128) return 0;
  const long long window = n_tokens < kWindow ? n_tokens : kWindow;
  const long long slots = window / kChunk + rows;
  return slots * H * (dk == 64 ? Part<64>::kFloats : Part<128>::kFloats) + (memory ? 3LL * window * H : 0);
}

static bool aligned_rows(const void* p, int stride) { return (uintptr_t)p % 8 == 0 && stride % 4 == 0; }

// The delta rule (plain_rate 0; a_ch null: a decay per head) or gated linear attention over the tokens t_first .. t_last of the
// rows of qo_indptr.  Returns 1 when the sizes or alignments are not taken (nothing launched).
int tl_delta_chunks(const void* qkv, int stride, const void* proj, int proj_stride, int b_off, int a_off, const float* A_log, const float* dt_bias,
                    float* state, long long state_stride, const int32_t* qo_indptr, const int32_t* slot_ids, float* o_raw, int t_first, int t_last,
                    int rows, int H, int G, int dk, int dv, const float* a_ch, int a_stride, float plain_rate, float* ws, long long floats,
                    hipStream_t stream) {
  if (ws == nullptr || (dk != 64 && dk != 128) || tl_chunk_floats(t_last - t_first, rows, H, dk, 0) > floats || !aligned_rows(qkv, stride) ||
      (uintptr_t)state % 16 || state_stride % 4 || (uintptr_t)ws % 16)
    return 1;
  ChunkArgs g = {};
  g.q = (const bf16_t*)qkv;
  g.k = g.q + (size_t)G * dk;
  g.v = g.k + (size_t)G * dk;
  g.stride = stride;
  g.proj = (const bf16_t*)proj;
  g.proj_stride = proj_stride; g.b_off = b_off; g.a_off = a_off;
  g.A_log = A_log; g.dt_bias = dt_bias; g.a_ch = a_ch; g.a_stride = a_stride; g.plain_rate = plain_rate;
  g.state = state; g.state_stride = state_stride; g.qo_indptr = qo_indptr; g.slot_ids = slot_ids; g.rows = rows;
  g.H = H; g.G = G; g.dv = dv; g.ws = ws; g.o_raw = o_raw;
#define TL_CHUNKS(DK)                                                                     \
  do {                                                                                    \
    if (plain_rate > 0.f) return run_chunks<DK, kRulePlain>(g, t_first, t_last, stream);  \
    if (a_ch) return run_chunks<DK, kRuleChannel>(g, t_first, t_last, stream);            \
    return run_chunks<DK, kRuleHead>(g, t_first, t_last, stream);                         \
  } while (0)
  if (dk == 64) TL_CHUNKS(64);
  TL_CHUNKS(128);
#undef TL_CHUNKS
}

// The matrix memory; offsets are columns of proj.  Returns 1 when the sizes or alignments are not taken.
int tl_memory_chunks(const void* proj, int stride, int q_off, int k_off, int v_off, int i_off, int f_off, const float* i_bias, const float* f_bias,
                     float cap, float* state, long long state_stride, const int32_t* qo_indptr, const int32_t* slot_ids, float* o_raw, float* den,
                     int t_first, int t_last, int rows, int H, int dk, int dv, float* ws, long long floats, hipStream_t stream) {
  const bf16_t* p = (const bf16_t*)proj;
  if (ws == nullptr || (dk != 64 && dk != 128) || tl_chunk_floats(t_last - t_first, rows, H, dk, 1) > floats || !aligned_rows(p + q_off, stride) ||
      !aligned_rows(p + k_off, stride) || (uintptr_t)state % 16 || state_stride % 4 || (uintptr_t)ws % 16)
    return 1;
  ChunkArgs g = {};
  g.q = p + q_off; g.k = p + k_off; g.v = p + v_off;
  g.stride = stride;
  g.i_off = i_off - q_off; g.f_off = f_off - q_off; g.i_bias = i_bias; g.f_bias = f_bias; g.cap = cap;
  g.state = state; g.state_stride = state_stride; g.qo_indptr = qo_indptr; g.slot_ids = slot_ids; g.rows = rows;
  g.H = H; g.G = H; g.dv = dv; g.ws = ws; g.o_raw = o_raw; g.den = den;
  g.gates = ws + tl_chunk_floats(t_last - t_first, rows, H, dk, 0);
  return dk == 64 ? run_chunks<64, kRuleMemory>(g, t_first, t_last, stream) : run_chunks<128, kRuleMemory>(g, t_first, t_last, stream);
}
