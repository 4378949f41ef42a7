// The products of routed experts over their gathered rows, bfloat16 inputs, 32-bit sums: for every expert e,
// C[r, n] = rows[r] . W[e][n] for its rows offsets[e] .. offsets[e + 1], or (GLU) mid[r, n] = silu(rows[r] . Wgate[e][n]) *
// (rows[r] . Wup[e][n]), rounded once or as dense layers round (gated, below).  How many rows an expert got is known on the device only, so one launch covers all
// experts: a block finds its tile from the offsets, and blocks beyond the last tile end at once.  Nothing is read back, and
// the launch depends on the step's shape alone (it can be recorded).
//
//   * A block of four waves takes BM rows of one expert and BN rows of its matrix; K is walked in steps of 64.  A step's
//     rows lie in LDS as in memory, 128 bytes a row, 16-byte piece p of row r at slot p ^ (r % 8): the eight lanes that are
//     served together read eight different slots.  Everything is fetched by global_load_lds, kStages - 1 steps ahead.
//   * C^T by MFMA 16x16x32 (first operand W): a lane holds four neighbouring columns of a row.  Operands of one half of a
//     step are read while the other half is multiplied; the one barrier a step stands between the two halves, so that
//     neither the wait for LDS nor that for the barrier leaves the matrix cores idle.
//   * GLU: a wave's rows of W are half gate rows, half up rows of the same columns, so the gate meets its up product in
//     registers.
//   * Tiles by the rows an expert has on average: 128 x 128 for prompts (bound by LDS reads and the matrix cores, which take
//     about the same time; two blocks a CU fill each other's gaps) and 128 x 256 for long ones (below), 16, 32 or 64 rows for decode steps and short prompts
//     (bound by reading W: many blocks with several steps in flight).
//   * Blocks go to the eight XCDs in turn.  All row tiles of one (expert, column tile) go to the same XCD one after the
//     other, so W is read from memory once and met again in that XCD's L2; an expert's column tiles are spread over all XCDs.
// 8 experts, pairs spread by chance, gated + plain product, us (the kernels for other widths, or a library product per expert, the
// activation in a kernel of its own and a wait of the host, which these took the place of): 4,096 x 3,584, 16 pairs 79 + 40 (116 +
// 46; the bytes of W at 6.1 TB/s: 77 + 38), 128 pairs 83 + 44 (159 + 94), 4,096 pairs 294 + 181 (650 in all); 2,048 x 2,048, 16
// pairs 28 + 16 (38 + 22), 128 pairs 28 + 17 (45 + 25), 4,096 pairs 106 + 81 (441).
#include <type_traits>

#include "common.h"

namespace {

typedef __bf16 bf16x8_e __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4_e __attribute__((ext_vector_type(4)));
typedef float float4_e __attribute__((ext_vector_type(4)));

constexpr int kStepE = 64;    // k per step: 8 pieces of 16 bytes a row
constexpr int kXcds = 8;

// silu(gate) * up of four columns.  rounded: the two products and the activation are rounded to bfloat16 on the way, as dense
// layers' are (silu_mul of a product stored in bfloat16); otherwise the result alone is.
__device__ __forceinline__ bf16x4_e gated(const float4_e& gate, const float4_e& up, bool rounded) {
  bf16x4_e out;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float g = rounded ? (float)(__bf16)gate[i] : gate[i], u = rounded ? (float)(__bf16)up[i] : up[i];
    const float act = g / (1.0f + expf(-g));
    out[i] = (__bf16)((rounded ? (float)(__bf16)act : act) * u);
  }
  return out;
}

template <int BM, int BN, int WAVES_M, int kStages, bool GLU>
struct ExpertTile {
  static constexpr int kWavesN = 4 / WAVES_M;
  static constexpr int WM = BM / WAVES_M, WN = BN / kWavesN;
  static constexpr int MT = WM / 16, NT = WN / 16;
  static constexpr int kColumns = GLU ? BN / 2 : BN;           // output columns of a block
  static constexpr int kALoads = BM >= 32 ? BM / 32 : 1;       // load instructions of a wave per step: 8 rows each
  static constexpr int kWLoads = BN / 32;
  static constexpr int kStage = (BM + BN) * kStepE;            // elements of one buffer
  static constexpr int kLdsBytes = kStages * kStage * 2;
  static constexpr int kPending = (kStages - 2) * (kALoads + kWLoads);
  static_assert(kPending < 64, "vmcnt has six bits");
  // s_waitcnt that leaves the loads of the kStages - 2 latest steps outstanding
  static constexpr int kWait = (kPending & 0xF) | (0x7 << 4) | (0xF << 8) | ((kPending >> 4) << 14);
};

// Which tile a block takes: XCD x walks, expert after expert, its column tiles n = x, x + 8, ... (the start shifted from expert
// to expert, so that a number of tiles that is no multiple of 8 evens out), the row tiles of each side by side.  False: none.
struct Tile { int e, n_tile, r0, hi; };
template <int BM>
__device__ __forceinline__ bool find_tile(const int32_t* __restrict__ offsets, int n_experts, int n_tiles, int lane, Tile& t) {
  const int per_xcd = (n_tiles + kXcds - 1) / kXcds;
  const int x = blockIdx.x % kXcds;
  int j = blockIdx.x / kXcds;  // place among this XCD's tiles
  int e = -1, m_tiles = 0;
  for (int e0 = 0; e0 < n_experts; e0 += kWave) {
    const int mine = e0 + lane < n_experts ? (offsets[e0 + lane + 1] - offsets[e0 + lane] + BM - 1) / BM : 0;
    int sum = mine;  // row tiles up to and with this expert
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
      const int before = __shfl_up(sum, off, kWave);
      if (lane >= off) sum += before;
    }
    const unsigned long long beyond = __ballot(sum * per_xcd > j);
    if (beyond) {
      const int l = __ffsll(beyond) - 1;
      e = e0 + l;
      m_tiles = __shfl(mine, l, kWave);
      j -= (__shfl(sum, l, kWave) - m_tiles) * per_xcd;
      break;
    }
    j -= __shfl(sum, kWave - 1, kWave) * per_xcd;
  }
  if (e < 0) return false;
  t.e = __builtin_amdgcn_readfirstlane(e);
  t.n_tile = __builtin_amdgcn_readfirstlane((j / m_tiles) * kXcds + (x + t.e * (n_tiles % kXcds)) % kXcds);
  if (t.n_tile >= n_tiles) return false;
  t.hi = offsets[t.e + 1];
  t.r0 = __builtin_amdgcn_readfirstlane(offsets[t.e] + (j % m_tiles) * BM);
  return true;
}

template <int BM, int BN, int WAVES_M, int kStages, bool GLU>
__global__ void __launch_bounds__(256)
expert_tile_kernel(const bf16_t* __restrict__ rows, const bf16_t* __restrict__ w, const int32_t* __restrict__ offsets, int n_experts,
                   bf16_t* __restrict__ mid, float* __restrict__ y, int K, int N, bool rounded) {
  using S = ExpertTile<BM, BN, WAVES_M, kStages, GLU>;
  constexpr int MT = S::MT, NT = S::NT;
  extern __shared__ __attribute__((aligned(16))) bf16_t lds_e[];
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  const int n16 = lane % 16, g4 = lane / 16;

  Tile tile;
  if (!find_tile<BM>(offsets, n_experts, (N + S::kColumns - 1) / S::kColumns, lane, tile)) return;
  const int e = tile.e, n_tile = tile.n_tile, r0 = tile.r0, hi = tile.hi;
  const int n0 = n_tile * S::kColumns;
  const bf16_t* we = w + (size_t)e * (GLU ? 2 : 1) * N * K;

  // what this lane fetches: rows past the expert's last repeat it, columns past N likewise; neither result is stored
  const int q8 = lane / 8, piece = 8 * ((lane % 8) ^ q8);
  const bf16_t* asrc[S::kALoads];
  const int a_first = BM >= 32 ? wave * S::kALoads * 8 : (wave % (BM / 8)) * 8;  // (16 rows: two waves fetch what the others fetch too)
#pragma unroll
  for (int i = 0; i < S::kALoads; ++i) asrc[i] = rows + (size_t)min(r0 + a_first + 8 * i + q8, hi - 1) * K + piece;
  const bf16_t* wsrc[S::kWLoads];
#pragma unroll
  for (int i = 0; i < S::kWLoads; ++i) {
    const int r = (wave * S::kWLoads + i) * 8 + q8;  // row of the buffer
    int row;
    if constexpr (GLU) {
      const int in = r % S::WN, half = in / (S::WN / 2);
      row = half * N + min(n0 + (r / S::WN) * (S::WN / 2) + in % (S::WN / 2), N - 1);
    } else {
      row = min(n0 + r, N - 1);
    }
    wsrc[i] = we + (size_t)row * K + piece;
  }
  const uint32_t base = (uint32_t)(uintptr_t)lds_e;
  const uint32_t a_at = __builtin_amdgcn_readfirstlane(base + a_first * kStepE * 2);
  const uint32_t w_at = __builtin_amdgcn_readfirstlane(base + (BM + wave * S::kWLoads * 8) * kStepE * 2);
  auto issue = [&](int step, int buffer) {
#pragma unroll
    for (int i = 0; i < S::kALoads; ++i) load_to_lds(asrc[i] + step * kStepE, a_at + (buffer * S::kStage + i * 8 * kStepE) * 2);
#pragma unroll
    for (int i = 0; i < S::kWLoads; ++i) load_to_lds(wsrc[i] + step * kStepE, w_at + (buffer * S::kStage + i * 8 * kStepE) * 2);
  };

  float4_e acc[NT][MT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int c = 0; c < MT; ++c) acc[t][c] = float4_e{0.f, 0.f, 0.f, 0.f};

  const int am = (wave % WAVES_M) * S::WM, wn = wave / WAVES_M;
  const int at[2] = {n16 * kStepE + 8 * (g4 ^ (n16 % 8)), n16 * kStepE + 8 * ((4 + g4) ^ (n16 % 8))};
  bf16x8_e wop[2][NT], aop[2][MT];
  auto operands = [&](int buffer, int half) {
    const bf16_t* as = lds_e + buffer * S::kStage + am * kStepE + at[half];
    const bf16_t* ws = lds_e + buffer * S::kStage + (BM + wn * S::WN) * kStepE + at[half];
#pragma unroll
    for (int c = 0; c < MT; ++c) aop[half][c] = *reinterpret_cast<const bf16x8_e*>(as + c * 16 * kStepE);
#pragma unroll
    for (int t = 0; t < NT; ++t) wop[half][t] = *reinterpret_cast<const bf16x8_e*>(ws + t * 16 * kStepE);
  };
  auto multiply = [&](int half) {
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int c = 0; c < MT; ++c) acc[t][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wop[half][t], aop[half][c], acc[t][c], 0, 0, 0);
  };

  // all loads are unconditional (past the end the last step is fetched again and never used), so that a wave's count of
  // outstanding loads is the same in every trip
  const int steps = K / kStepE;
  // rows of W lie a power of two apart, so blocks that walk K in step would all press on the same memory channels at once:
  // the column tiles start their walks at different steps and wrap around (the row tiles of one at the same step: they share
  // W in L2, and a row's sums do not depend on where it lies).  Eight experts of 2,048 x 2,048, gated + plain product, in step | like
  // this: 48 pairs 35.3 + 19.2 us | 27.5 + 16.5, 256 pairs 37.1 + 22.7 | 29.3 + 22.0; of 4,096 x 3,584 92.0 + 42.8 | 81.6 + 42.6 and
  // 94.1 + 48.8 | 89.3 + 50.6.  With 128 rows a tile blocks lose what they share of the rows (4,096 pairs 315 + 202 | 345 + 212).
  const int rot = BM <= 64 ? (n_tile * 5 + e * 3) % steps : 0;
  auto step_of = [&](int i) { return i + rot < steps ? i + rot : i + rot - steps; };
#pragma unroll
  for (int s = 0; s < kStages - 1; ++s) issue(step_of(min(s, steps - 1)), s);
  __builtin_amdgcn_s_waitcnt(S::kWait);
  __syncthreads();
  operands(0, 0);
  int buffer = 0;
  for (int i = 0; i < steps; ++i) {
    // (everybody passed the barrier below after reading the last of step i - 1, whose buffer is filled again here)
    issue(step_of(min(i + kStages - 1, steps - 1)), buffer == 0 ? kStages - 1 : buffer - 1);
    operands(buffer, 1);
    __builtin_amdgcn_sched_barrier(0);
    multiply(0);
    __builtin_amdgcn_sched_barrier(0);
    buffer = buffer + 1 == kStages ? 0 : buffer + 1;
    __builtin_amdgcn_s_waitcnt(S::kWait);  // this wave's loads of step i + 1 have landed; after the barrier everybody's have
    __syncthreads();
    operands(buffer, 0);
    __builtin_amdgcn_sched_barrier(0);
    multiply(1);
    __builtin_amdgcn_sched_barrier(0);
  }
  __builtin_amdgcn_s_waitcnt(0);  // the last, unused fetches must not land after the block has gone

  // acc[t][c][i]: row r0 + am + 16 c + n16, W row 16 t + 4 g4 + i of the wave's
#pragma unroll
  for (int c = 0; c < MT; ++c) {
    const int r = r0 + am + 16 * c + n16;
    if (r >= hi) continue;
    if constexpr (GLU) {
#pragma unroll
      for (int t = 0; t < NT / 2; ++t) {
        const int n = n0 + wn * (S::WN / 2) + 16 * t + 4 * g4;
        if (n >= N) continue;  // (N is a multiple of 4)
        *reinterpret_cast<bf16x4_e*>(mid + (size_t)r * N + n) = gated(acc[t][c], acc[t + NT / 2][c], rounded);
      }
    } else {
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const int n = n0 + wn * S::WN + 16 * t + 4 * g4;
        if (n < N) *reinterpret_cast<float4_e*>(y + (size_t)r * N + n) = acc[t][c];
      }
    }
  }
}

template <int BM, int BN, int WAVES_M, int kStages, bool GLU>
int launch_expert_tiles(const void* rows, const void* w, const int32_t* offsets, int n_experts, void* mid, float* y, int K, int N, int pairs,
                        bool rounded, hipStream_t stream) {
  using S = ExpertTile<BM, BN, WAVES_M, kStages, GLU>;
  const auto kernel = expert_tile_kernel<BM, BN, WAVES_M, kStages, GLU>;
  if (S::kLdsBytes > 48 * 1024) {
    hipError_t err = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, S::kLdsBytes);
    if (err != hipSuccess) return tl_fail(TL_ERR_HIP, "expert products: %s", hipGetErrorString(err));
  }
  const int n_tiles = (N + S::kColumns - 1) / S::kColumns;
  const int per_xcd = (n_tiles + kXcds - 1) / kXcds;
  const int most = (pairs < n_experts ? pairs : n_experts) + pairs / BM;  // row tiles there can be
  kernel<<<dim3((unsigned)(kXcds * per_xcd) * most), 256, S::kLdsBytes, stream>>>((const bf16_t*)rows, (const bf16_t*)w, offsets, n_experts,
                                                                               (bf16_t*)mid, y, K, N, rounded);
  return tl_check_launch("expert_tiles");
}

// The same with 128 x 256 tiles, for prompts: a wave takes 64 x 128 of it, so that it reads three quarters of the LDS bytes an
// MFMA that 64 x 64 reads.  K in steps of 32 (64 bytes a row, piece p at slot p ^ (r / 2 % 4)), three buffers of 24 KB, so that
// two blocks share a CU; a step's operands are read while the step before is multiplied, one barrier a step.
constexpr int kWideM = 128, kWideN = 256, kWideStep = 32, kWideStage = (kWideM + kWideN) * kWideStep;  // (elements)
template <bool GLU>
__global__ void __launch_bounds__(256, 2)
expert_wide_tile_kernel(const bf16_t* __restrict__ rows, const bf16_t* __restrict__ w, const int32_t* __restrict__ offsets, int n_experts,
                        bf16_t* __restrict__ mid, float* __restrict__ y, int K, int N, bool rounded) {
  constexpr int kColumns = GLU ? kWideN / 2 : kWideN, WM = 64, WN = 128, MT = WM / 16, NT = WN / 16, kLoads = 6;
  extern __shared__ __attribute__((aligned(16))) bf16_t lds_e[];
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  const int n16 = lane % 16, g4 = lane / 16;
  Tile tile;
  if (!find_tile<kWideM>(offsets, n_experts, (N + kColumns - 1) / kColumns, lane, tile)) return;
  const int e = tile.e, r0 = tile.r0, hi = tile.hi;
  const int n0 = tile.n_tile * kColumns;
  const bf16_t* we = w + (size_t)e * (GLU ? 2 : 1) * N * K;

  // instruction j of the wave fills 16 rows of the buffer: two of rows, four of W
  const int r16 = lane / 4, piece = 8 * ((lane % 4) ^ (r16 / 2 % 4));
  const bf16_t* src[kLoads];
#pragma unroll
  for (int j = 0; j < 2; ++j) src[j] = rows + (size_t)min(r0 + (wave * 2 + j) * 16 + r16, hi - 1) * K + piece;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int r = (wave * 4 + j) * 16 + r16;
    int row;
    if constexpr (GLU) {
      const int in = r % WN, half = in / (WN / 2);
      row = half * N + min(n0 + (r / WN) * (WN / 2) + in % (WN / 2), N - 1);
    } else {
      row = min(n0 + r, N - 1);
    }
    src[2 + j] = we + (size_t)row * K + piece;
  }
  const uint32_t base = (uint32_t)(uintptr_t)lds_e;
  const uint32_t a_at = __builtin_amdgcn_readfirstlane(base + wave * 2 * 1024);
  const uint32_t w_at = __builtin_amdgcn_readfirstlane(base + kWideM * kWideStep * 2 + wave * 4 * 1024);
  auto issue = [&](int step, int buffer) {
#pragma unroll
    for (int j = 0; j < 2; ++j) load_to_lds(src[j] + step * kWideStep, a_at + buffer * kWideStage * 2 + j * 1024);
#pragma unroll
    for (int j = 0; j < 4; ++j) load_to_lds(src[2 + j] + step * kWideStep, w_at + buffer * kWideStage * 2 + j * 1024);
  };
  float4_e acc[NT][MT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int c = 0; c < MT; ++c) acc[t][c] = float4_e{0.f, 0.f, 0.f, 0.f};
  const int am = (wave % 2) * WM, wn = wave / 2;
  const int at = n16 * kWideStep + 8 * (g4 ^ (n16 / 2 % 4));
  bf16x8_e wop[2][NT], aop[2][MT];
  auto operands = [&](auto set, int buffer) {
    const bf16_t* as = lds_e + buffer * kWideStage + am * kWideStep + at;
    const bf16_t* ws = lds_e + buffer * kWideStage + (kWideM + wn * WN) * kWideStep + at;
#pragma unroll
    for (int c = 0; c < MT; ++c) aop[set][c] = *reinterpret_cast<const bf16x8_e*>(as + c * 16 * kWideStep);
#pragma unroll
    for (int t = 0; t < NT; ++t) wop[set][t] = *reinterpret_cast<const bf16x8_e*>(ws + t * 16 * kWideStep);
  };
  auto multiply = [&](auto set) {
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int c = 0; c < MT; ++c) acc[t][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wop[set][t], aop[set][c], acc[t][c], 0, 0, 0);
  };
  // s_waitcnt: loads of all but the `steps` latest steps have landed; LDS reads too where `lds` is 0
  constexpr auto wait = [](int steps, int lds) { return (steps * kLoads & 0xF) | (0x7 << 4) | (lds << 8) | (steps * kLoads >> 4 << 14); };
  const int steps = K / kWideStep;  // (even: K is a multiple of 64)
  int b = 0;                        // buffer of step i
  // (loads are unconditional, as above)
  auto pass = [&](int i, auto set, auto next) {
    // this wave's operands of step i are in registers and its loads of step i + 1 in LDS; after the barrier everybody's are, and
    // the buffer of step i is free
    __builtin_amdgcn_s_waitcnt(wait(1, 0));
    __syncthreads();
    issue(min(i + 3, steps - 1), b);
    b = b == 2 ? 0 : b + 1;
    operands(next, b);
    __builtin_amdgcn_sched_barrier(0);
    multiply(set);
    __builtin_amdgcn_sched_barrier(0);
  };
  using Zero = std::integral_constant<int, 0>;
  using One = std::integral_constant<int, 1>;
#pragma unroll
  for (int s = 0; s < 3; ++s) issue(min(s, steps - 1), s);
  __builtin_amdgcn_s_waitcnt(wait(2, 0xF));
  __syncthreads();
  operands(Zero(), 0);
  for (int i = 0; i < steps; i += 2) {
    pass(i, Zero(), One());
    pass(i + 1, One(), Zero());
  }
  __builtin_amdgcn_s_waitcnt(0);  // the last, unused fetches must not land after the block has gone

  // acc[t][c][i]: row r0 + am + 16 c + n16, W row 16 t + 4 g4 + i of the wave's
#pragma unroll
  for (int c = 0; c < MT; ++c) {
    const int r = r0 + am + 16 * c + n16;
    if (r >= hi) continue;
    if constexpr (GLU) {
#pragma unroll
      for (int t = 0; t < NT / 2; ++t) {
        const int n = n0 + wn * (WN / 2) + 16 * t + 4 * g4;
        if (n >= N) continue;  // (N is a multiple of 4)
        *reinterpret_cast<bf16x4_e*>(mid + (size_t)r * N + n) = gated(acc[t][c], acc[t + NT / 2][c], rounded);
      }
    } else {
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const int n = n0 + wn * WN + 16 * t + 4 * g4;
        if (n < N) *reinterpret_cast<float4_e*>(y + (size_t)r * N + n) = acc[t][c];
      }
    }
  }
}

template <bool GLU>
int launch_expert_wide(const void* rows, const void* w, const int32_t* offsets, int n_experts, void* mid, float* y, int K, int N, int pairs,
                       bool rounded, hipStream_t stream) {
  constexpr int kLds = 3 * kWideStage * 2, kColumns = GLU ? kWideN / 2 : kWideN;
  const auto kernel = expert_wide_tile_kernel<GLU>;
  hipError_t err = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
  if (err != hipSuccess) return tl_fail(TL_ERR_HIP, "expert products: %s", hipGetErrorString(err));
  const int per_xcd = ((N + kColumns - 1) / kColumns + kXcds - 1) / kXcds;
  const int most = (pairs < n_experts ? pairs : n_experts) + pairs / kWideM;  // row tiles there can be
  kernel<<<dim3((unsigned)(kXcds * per_xcd) * most), 256, kLds, stream>>>((const bf16_t*)rows, (const bf16_t*)w, offsets, n_experts, (bf16_t*)mid, y,
                                                                        K, N, rounded);
  return tl_check_launch("expert_wide_tiles");
}

}  // namespace

// What the kernels take: K a multiple of a step, columns in fours, rows and weights on 16-byte boundaries (K in 64s keeps every row
// there), results on those of their stores.
bool tl_expert_tiles_fit(const void* rows, const void* w, const void* mid, const float* y, int K, int N) {
  return K % kStepE == 0 && N % 4 == 0 && ((uintptr_t)rows | (uintptr_t)w | (uintptr_t)y) % 16 == 0 && (uintptr_t)mid % 8 == 0;
}

// mid != null: the gated product (w [E, 2 N, K], gate rows then up rows; rounded: as dense layers do), otherwise y = the plain one
// (w [E, N, K]).
//
// Which tile: by the rows an expert has on average (`pairs` counts those of outputs that are no experts too).  Measured at 8
// experts, pairs spread by chance, gated + plain product in us, tiles of 16 | 32 | 64 | 128 rows | 128 x 256:
//   4,096 x 3,584: 16 pairs 81 + 42 | 80 + 42 | 82 + 42; 128 pairs 91 + 48 | 83 + 43 | 83 + 43 | 103 + 67; 256 pairs 113 + 64 | 94 + 54 |
//   90 + 46 | 104 + 66; 1,024 pairs 171 + 107 (32) | 146 + 86 | 160 + 75 | 152 + 81; 2,424 pairs 238 + 137 (64) | 230 + 135 | 228 + 127;
//   4,096 pairs 374 + 215 (64) | 313 + 200 | 287 + 180.
//   2,048 x 2,048: 16 pairs 28 + 16 | 27 + 16 | 28 + 24; 256 pairs 39 + 25 | 35 + 22 | 29 + 25 | 46 + 37; 1,024 pairs 59 + 37 (32) | 50 + 35
//   | 50 + 41 | 51 + 44; 2,424 pairs 77 + 49 (64) | 81 + 46 | 75 + 45; 4,096 pairs 120 + 72 (64) | 118 + 81 | 106 + 66.
// 128 x 256 tiles where they are more than five for four CUs; with fewer the CUs that get none weigh more (4,096 x 1,024, 512 to
// 2,424 pairs, gated: 72 to 77 with 128 rows, 79 to 83 with these), though not everywhere: 288 of them for the plain product
// of 4,096 pairs of 2,048 x 2,048 take 66, and 128 x 128, which the rule takes, 81.
int tl_expert_tiles(const void* rows, const void* w, const int32_t* offsets, int n_experts, void* mid, float* y, int K, int N, int pairs,
                    bool rounded, hipStream_t stream) {
  const double mean = (double)pairs / n_experts;
  // (the large tiles there will be, every expert's last one half empty)
  const double large = (pairs / (double)kWideM + 0.5 * n_experts) * ((N + (mid ? kWideN / 2 : kWideN) - 1) / (mid ? kWideN / 2 : kWideN));
  if (mean > 256 && large > 1.25 * tl_device_facts().compute_units)
    return mid ? launch_expert_wide<true>(rows, w, offsets, n_experts, mid, y, K, N, pairs, rounded, stream)
               : launch_expert_wide<false>(rows, w, offsets, n_experts, mid, y, K, N, pairs, rounded, stream);
#define TL_TILES(BM, BN, WM, ST, GLU) return launch_expert_tiles<BM, BN, WM, ST, GLU>(rows, w, offsets, n_experts, mid, y, K, N, pairs, rounded, stream)
  if (mid) {
    if (mean <= 12) TL_TILES(16, 128, 1, 4, true);
    if (mean <= 24) TL_TILES(32, 128, 1, 4, true);
    if (mean <= 256) TL_TILES(64, 128, 1, 3, true);
    TL_TILES(128, 128, 2, 2, true);
  }
  if (mean <= 12) TL_TILES(16, 64, 1, 4, false);
  if (mean <= 48) TL_TILES(32, 64, 1, 4, false);
  if (mean <= 128) TL_TILES(64, 128, 1, 3, false);
  TL_TILES(128, 128, 2, 2, false);
#undef TL_TILES
}
