// C[M, N] = A[M, K] * W[N, K]^T in true 32-bit: float inputs, every product and sum rounded to float, no
// reduced-precision mode.  An output element is the sum over groups of 16 products: a group's products are chained by
// fused multiply-adds from k ascending, starting from zero, and its sum joins the running sum, groups in ascending order.
// (The rounding error of a long sum grows with the number of additions to one accumulator: this way there are K / 16 + 16
// of them instead of K.)  So a value depends neither on M nor on where the row sits in the batch, whichever kernel
// computes it: tiles on the matrix cores for prompts, a wave per four columns for up to 16 rows.
#include "common.h"
#include "recurrence.h"  // mfma_f32

namespace {

constexpr int BK = 16;  // products that are added among themselves before they join the running sum

// ----------------------------------------------------------------------------- prompts
// v_mfma_f32_16x16x4_f32 computes an element as four fused multiply-adds chained from depth 0 up, each rounded to float
// (checked against fmaf bit for bit over a million groups of 16, values of 2^-30 to 2^30 and denormal ones): four of them
// from a zero accumulator are a group.  It does 143 to 155 TFLOP/s here where fused multiply-adds issued from registers
// reach 113, needs a fraction of the LDS reads, and a few chains a wave keep a SIMD busy.  What bounds it: the running sums'
// additions and the LDS reads take turns with the MFMAs (an addition an MFMA alone: 127 of 143 with two waves a SIMD).
//   * a block of four waves takes a BM x BN tile of C, a wave a WM x WN piece of it; K is walked in steps of 32 or 64;
//   * the step's rows of A and W lie in LDS as they are in memory, 128 or 256 bytes a row; 16-byte piece p of row r at slot
//     p ^ (r / 2 % 8) or p ^ (r % 16), so that the 16 rows x 4 words that a wave's operand read takes fall on all 64 banks;
//   * with 16-byte rows (kVec) the pieces go straight to LDS (global_load_lds), kStages - 1 steps ahead; otherwise they
//     pass through registers element by element, one step ahead;
//   * rows past M and N repeat the last row (their results are not stored), elements past K are zeros: a chain that goes
//     on with zeros keeps its bits.
// C^T tiles (W the first operand): a lane holds four neighbouring columns of a row of C.
// 562 rows of the 1B shape's qkv, o, gate/up and down matrices: 434 us on average for all but gate/up and 758 for that with
// tiles of plain fused multiply-adds before, 95 + 73 + 388 + 266 now; 2,048 rows of the 8B shape's gate/up: 4.0 ms, 120 TFLOP/s.
__device__ __attribute__((aligned(16))) const float kZeroPiece[4] = {0.f, 0.f, 0.f, 0.f};

template <int BM, int BN, int WM, int WN, int kStepF, int kStages, bool kVec>
__global__ void __launch_bounds__(256, 2)  // (two waves a SIMD: with 256 registers the compiler keeps sums out of the accumulation registers)
gemm_f32_tile_kernel(const float* __restrict__ A, int lda, const float* __restrict__ W, int ldw, float* __restrict__ C, int ldc, int M,
                     int N, int K) {
  static_assert((BM / WM) * (BN / WN) == 4, "four waves");
  constexpr int MT = WM / 16, NT = WN / 16;
  constexpr int kRowPieces = kStepF / 4;
  constexpr int kTurn = 64 / kStepF;             // rows that lie on the 64 banks side by side
  constexpr int kStage = (BM + BN) * kStepF;     // floats of one buffer: rows of A, then rows of W
  constexpr int kLoads = (BM + BN) * kRowPieces / 256;  // load instructions of a wave per step: a KB each
  constexpr int kPending = (kStages - 2) * kLoads;
  static_assert(kPending < 64, "vmcnt has six bits");
  // s_waitcnt that leaves the loads of the kStages - 2 latest steps outstanding
  constexpr int kWaitOldest = (kPending & 0xF) | (0x7 << 4) | (0xF << 8) | ((kPending >> 4) << 14);
  extern __shared__ __attribute__((aligned(16))) float tiles[];
  const int tid = threadIdx.x;
  const int wave = tid / kWave, lane = tid % kWave;
  const int n16 = lane % 16, g4 = lane / 16;
  // consecutive blocks share their columns: the tile of W is read from memory once for all of them
  const unsigned row_tiles = (unsigned)(M + BM - 1) / BM;
  const int m0 = (int)(blockIdx.x % row_tiles) * BM, n0 = (int)(blockIdx.x / row_tiles) * BN;
  const int wm = (wave % (BM / WM)) * WM, wn = (wave / (BM / WM)) * WN;
  const int steps = (K + kStepF - 1) / kStepF;

  // row r of a buffer: row of A, or of W behind them; a clamped row of memory
  auto row_of = [&](int r) { return r < BM ? A + (size_t)min(m0 + r, M - 1) * lda : W + (size_t)min(n0 + r - BM, N - 1) * ldw; };

  // -- aligned rows: instruction j of the wave fills buffer rows 8 (wave kLoads + j) ... + 7, a lane one slot of one row
  const float* src[kLoads];
  const uint32_t lds_base = (uint32_t)(uintptr_t)tiles;
  const uint32_t at0 = __builtin_amdgcn_readfirstlane(lds_base + wave * kLoads * 1024);
  int piece[kLoads];
  if constexpr (kVec) {
#pragma unroll
    for (int j = 0; j < kLoads; ++j) {
      const int r = (64 / kRowPieces) * (wave * kLoads + j) + lane / kRowPieces;
      piece[j] = 4 * ((lane % kRowPieces) ^ (r / kTurn % kRowPieces));
      src[j] = row_of(r);
    }
  }
  auto issue = [&](int step, int buffer) {
#pragma unroll
    for (int j = 0; j < kLoads; ++j) {
      const int k = step * kStepF + piece[j];
      load_to_lds(k < K ? src[j] + k : kZeroPiece, at0 + buffer * kStage * (int)sizeof(float) + j * 1024);
    }
  };
  // -- other rows: a thread moves pieces tid, tid + 256, ... of the buffer
  constexpr int kMoves = (BM + BN) * kRowPieces / 256;
  float held[kMoves][4];
  auto fetch = [&](int step) {
#pragma unroll
    for (int j = 0; j < kMoves; ++j) {
      const int r = (tid + 256 * j) / kRowPieces, k = step * kStepF + 4 * (tid % kRowPieces);
      const float* row = row_of(r);
#pragma unroll
      for (int e = 0; e < 4; ++e) held[j][e] = k + e < K ? row[k + e] : 0.f;
    }
  };
  auto put = [&](int buffer) {
#pragma unroll
    for (int j = 0; j < kMoves; ++j) {
      const int r = (tid + 256 * j) / kRowPieces;
      *reinterpret_cast<float4*>(tiles + buffer * kStage + r * kStepF + 4 * ((tid % kRowPieces) ^ (r / kTurn % kRowPieces))) =
          float4{held[j][0], held[j][1], held[j][2], held[j][3]};
    }
  };

  f32x4_t acc[NT][MT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int c = 0; c < MT; ++c) acc[t][c] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  // word offsets of the lane's operands within 16 rows: piece p of row n16, depth g4 of its four
  int word[kRowPieces];
#pragma unroll
  for (int p = 0; p < kRowPieces; ++p) word[p] = n16 * kStepF + 4 * (p ^ (n16 / kTurn % kRowPieces)) + g4;
  auto multiply = [&](int buffer) {
    const float* as = tiles + buffer * kStage + wm * kStepF;
    const float* ws = tiles + buffer * kStage + (BM + wn) * kStepF;
    constexpr int kGroups = kStepF / BK;
    if constexpr (MT * NT == 1) {
      // one tile: the step's groups are the chains that run side by side
      float w[kRowPieces], a[kRowPieces];
#pragma unroll
      for (int p = 0; p < kRowPieces; ++p) {
        w[p] = ws[word[p]];
        a[p] = as[word[p]];
      }
      f32x4_t part[kGroups];
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int g = 0; g < kGroups; ++g) part[g] = mfma_f32(w[4 * g + s], a[4 * g + s], s == 0 ? f32x4_t{0.f, 0.f, 0.f, 0.f} : part[g]);
#pragma unroll
      for (int g = 0; g < kGroups; ++g)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[0][0][i] += part[g][i];
    } else {
      // a row of MT tiles at a time: its chains run side by side, and between its MFMAs stand the additions of the row
      // before it, so that the matrix core does not wait for them; operands of the next group are read during this one
      float w[2][4][NT], a[2][4][MT];
      auto operands = [&](int g) {
#pragma unroll
        for (int s = 0; s < 4; ++s) {
#pragma unroll
          for (int t = 0; t < NT; ++t) w[g & 1][s][t] = ws[t * 16 * kStepF + word[4 * g + s]];
#pragma unroll
          for (int c = 0; c < MT; ++c) a[g & 1][s][c] = as[c * 16 * kStepF + word[4 * g + s]];
        }
      };
      f32x4_t part[2][MT];
      operands(0);
#pragma unroll
      for (int u = 0; u <= kGroups * NT; ++u) {
        const int g = u / NT, t = u % NT;
        if (t == 0 && g + 1 < kGroups) operands(g + 1);
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          // (the order as written: left to itself the compiler starts all rows at once and spills)
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int c = 0; c < MT; ++c) {
            if (u < kGroups * NT) part[u & 1][c] = mfma_f32(w[g & 1][s][t], a[g & 1][s][c], s == 0 ? f32x4_t{0.f, 0.f, 0.f, 0.f} : part[u & 1][c]);
            if (u > 0) acc[(u - 1) % NT][c][s] += part[(u - 1) & 1][c][s];
          }
        }
      }
    }
  };

  if constexpr (kVec) {
    // all loads are unconditional (past the end the last step is fetched again and never used), so that a wave's count of
    // outstanding loads is the same in every trip
#pragma unroll
    for (int s = 0; s < kStages - 1; ++s) issue(min(s, steps - 1), s);
    int buffer = 0;
    for (int i = 0; i < steps; ++i) {
      // this wave's loads of step i have landed; after the barrier everybody's have, and everybody has finished with
      // step i - 1, whose buffer the next loads overwrite
      __builtin_amdgcn_s_waitcnt(kWaitOldest);
      __syncthreads();
      issue(min(i + kStages - 1, steps - 1), buffer == 0 ? kStages - 1 : buffer - 1);
      multiply(buffer);
      buffer = buffer + 1 == kStages ? 0 : buffer + 1;
    }
    __builtin_amdgcn_s_waitcnt(0);  // the last, unused fetches must not land after the block has gone
  } else {
    fetch(0);
    put(0);
    __syncthreads();
    for (int i = 0; i < steps; ++i) {
      if (i + 1 < steps) fetch(i + 1);
      multiply(i & 1);
      if (i + 1 < steps) put((i + 1) & 1);
      __syncthreads();
    }
  }

  // acc[t][c][i] = C[m0 + wm + 16 c + n16][n0 + wn + 16 t + 4 g4 + i]
  const bool whole = ldc % 4 == 0 && (uintptr_t)C % 16 == 0;
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int c = 0; c < MT; ++c) {
      const int m = m0 + wm + 16 * c + n16, n = n0 + wn + 16 * t + 4 * g4;
      if (m >= M) continue;
      float* dst = C + (size_t)m * ldc + n;
      if (whole && n + 4 <= N) {
        *reinterpret_cast<f32x4_t*>(dst) = acc[t][c];
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (n + i < N) dst[i] = acc[t][c][i];
      }
    }
}

// ----------------------------------------------------------------------------- few rows (decode steps)
// The kernel above gives a block 32 rows of A and more; a decode step has one to sixteen, and what counts is reading W
// from everywhere at once.  This kernel computes the very same arithmetic for every output element (groups
// of 16 products, chained by fused multiply-adds from k ascending, each group's sum added to the
// running sum in the order of the groups), so its results are the same bits, but spreads the groups
// of an element over the lanes of a wave:
//   * a block of 4 waves takes 16 columns of the result, 4 per wave, and all rows (at most MR);
//   * K is walked in rounds of 1,024 = 64 groups: lane j computes group j of the round for its wave's
//     4 columns and every row (W: the wave reads a column's 4 KB of the round 1 KB per instruction and
//     turns it through a piece of LDS of its own, so that lane j holds elements 16 j .. 16 j + 15;
//     A: the round's slice of every row lies in LDS, loaded once per block, transposed so that the 64
//     lanes read 64 consecutive words); what the next round needs travels from memory into registers
//     while this round is multiplied;
//   * the groups' sums then have to join the running sums in the order of the groups: they go through
//     LDS, transposed, and lane p of the wave adds the 64 sums of (column, row) pair p one after the other.
constexpr int kRowsCols = 4;               // columns per wave
constexpr int kRowsWaves = 4;              // waves per block
constexpr int kRound = 64 * BK;            // k per round
constexpr int kPad = 65;                   // row stride of transposed tables in LDS (odd: no bank conflicts)
constexpr int kTurned = kRound + kRound / 4;  // a column's round of W in LDS: four words of padding behind every group

template <int MR, bool kVec>
__global__ void __launch_bounds__(kRowsWaves * kWave)
gemm_f32_rows_kernel(const float* __restrict__ A, int lda, const float* __restrict__ W, int ldw,
                     float* __restrict__ C, int ldc, int M, int N, int K) {
  constexpr int kPairs = kRowsCols * MR;   // (column, row) pairs of a wave: at most 64
  constexpr int kWaveRegion = kPairs * kPad > kTurned ? kPairs * kPad : kTurned;
  extern __shared__ float lds[];
  float* xs = lds;                                          // [MR][BK][kPad]: element u of group j of row m at (m * BK + u) * kPad + j
  float* ps = lds + MR * BK * kPad;                         // [waves][kWaveRegion]: a wave's own piece
  const int tid = threadIdx.x;
  const int wave = tid / kWave;
  const int lane = tid % kWave;
  float* my_ps = ps + wave * kWaveRegion;                   // [kPairs][kPad] sums, or a column's round of W being turned
  const int n0 = (blockIdx.x * kRowsWaves + wave) * kRowsCols;

  float acc = 0.f;  // lane p < kPairs: running sum of pair p = (column p / MR, row p % MR)

  // What a round needs from memory is asked for a round ahead and waits in registers while the round
  // before it is multiplied.  Thread t moves elements 4 t .. 4 t + 3 of every row's slice of A; lane l
  // moves, of each of the wave's four columns of W, elements 256 q + 4 l .. + 3 for q = 0 .. 3 (the wave
  // reads 1 KB on end per instruction).
  // Two kernels (kVec): with rows of A and W on 16-byte boundaries and K a multiple of 4 everything is
  // fetched sixteen bytes a lane, otherwise element by element (one kernel with both forms under a branch
  // came out of the compiler with the element-wise loads for both).  Rows past M and elements past K are
  // read from a valid place (the row's last elements) and replaced by zeros when the round begins:
  // nothing here looks at a loaded value, or the wave would wait for each load in turn.
  float a_next[MR][4];
  float w_next[kRowsCols][BK];
  auto fetch = [&](int k0) {
    const int ka = k0 + 4 * tid;
#pragma unroll
    for (int m = 0; m < MR; ++m) {
      const float* arow = A + (size_t)(m < M ? m : 0) * lda;
      if constexpr (kVec) {
        const float4 v = *reinterpret_cast<const float4*>(arow + min(ka, K - 4));
        a_next[m][0] = v.x; a_next[m][1] = v.y; a_next[m][2] = v.z; a_next[m][3] = v.w;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) a_next[m][e] = arow[min(ka + e, K - 1)];
      }
    }
#pragma unroll
    for (int c = 0; c < kRowsCols; ++c) {
      const int n = n0 + c;
      const float* wrow = W + (size_t)(n < N ? n : N - 1) * ldw;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int k = k0 + 256 * q + 4 * lane;
        if constexpr (kVec) {
          const float4 v = *reinterpret_cast<const float4*>(wrow + min(k, K - 4));
          w_next[c][4 * q] = v.x; w_next[c][4 * q + 1] = v.y; w_next[c][4 * q + 2] = v.z; w_next[c][4 * q + 3] = v.w;
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) w_next[c][4 * q + e] = wrow[min(k + e, K - 1)];
        }
      }
    }
  };

  fetch(0);
  for (int k0 = 0; k0 < K; k0 += kRound) {
    __syncthreads();  // everybody has finished with the slice of the round before
#pragma unroll
    for (int m = 0; m < MR; ++m)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int kk = 4 * tid + e;
        xs[(m * BK + kk % BK) * kPad + kk / BK] = (m < M && k0 + kk < K) ? a_next[m][e] : 0.f;
      }
    // the wave turns its columns of W through its own piece of LDS (free: the sums of the round before
    // have been added): lane j gets group j, elements 16 j .. 16 j + 15 of the round.  A wave's LDS
    // instructions are carried out in their order, so no barrier stands between the writes and the reads.
    float w[kRowsCols][BK];
#pragma unroll
    for (int c = 0; c < kRowsCols; ++c) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int kk = 256 * q + 4 * lane;
        const int left = K - (k0 + kk);  // elements of the row from here on: past them, zeros
        *reinterpret_cast<float4*>(my_ps + kk + 4 * (kk / BK)) =
            float4{left > 0 ? w_next[c][4 * q] : 0.f, left > 1 ? w_next[c][4 * q + 1] : 0.f,
                   left > 2 ? w_next[c][4 * q + 2] : 0.f, left > 3 ? w_next[c][4 * q + 3] : 0.f};
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int u = 0; u < BK; u += 4) {
        const float4 v = *reinterpret_cast<const float4*>(my_ps + (BK + 4) * lane + u);
        w[c][u] = v.x; w[c][u + 1] = v.y; w[c][u + 2] = v.z; w[c][u + 3] = v.w;
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
    // (asked for as soon as the registers are free, before the barrier: the fewer cycles a wave has no
    // load under way, the better; with two blocks a CU nobody else fills the gap)
    if (k0 + kRound < K) fetch(k0 + kRound);
    __syncthreads();
    float part[kRowsCols][MR];
#pragma unroll
    for (int c = 0; c < kRowsCols; ++c)
#pragma unroll
      for (int m = 0; m < MR; ++m) part[c][m] = 0.f;
#pragma unroll
    for (int u = 0; u < BK; ++u) {
#pragma unroll
      for (int m = 0; m < MR; ++m) {
        const float a = xs[(m * BK + u) * kPad + lane];
#pragma unroll
        for (int c = 0; c < kRowsCols; ++c) part[c][m] = fmaf(a, w[c][u], part[c][m]);
      }
    }
    // the sums of this lane's group, transposed: pair p's 64 sums lie side by side
#pragma unroll
    for (int c = 0; c < kRowsCols; ++c)
#pragma unroll
      for (int m = 0; m < MR; ++m) my_ps[(c * MR + m) * kPad + lane] = part[c][m];
    __syncthreads();
    if (lane < kPairs) {
      const float* mine = my_ps + lane * kPad;
      const int groups = min(64, (K - k0 + BK - 1) / BK);  // groups of this round that exist
      if (groups == 64) {
        // all 64 sums are asked for before the first is added (a loop would wait for LDS 64 times in a row)
        float sums[64];
#pragma unroll
        for (int g = 0; g < 64; ++g) sums[g] = mine[g];
#pragma unroll
        for (int g = 0; g < 64; ++g) acc += sums[g];
      } else {
        for (int g = 0; g < groups; ++g) acc += mine[g];
      }
    }
  }
  if (lane < kPairs) {
    const int n = n0 + lane / MR, m = lane % MR;
    if (n < N && m < M) C[(size_t)m * ldc + n] = acc;
  }
}

template <int BM, int WM, int kStepF, int kStages, bool kVec>
int launch_tile(const float* A, int lda, const float* W, int ldw, float* C, int ldc, int M, int N, int K, hipStream_t stream) {
  constexpr size_t kLds = (size_t)kStages * (2 * BM) * kStepF * sizeof(float);
  const size_t grid = ((size_t)M + BM - 1) / BM * (((size_t)N + BM - 1) / BM);  // (one dimension: the others end at 65,535 tiles)
  TL_REQUIRE(grid * 256 < (1ull << 32), "gemm_f32: %d x %d exceeds the grid limit of one launch", M, N);
  if (kLds > 48 * 1024) {
    hipError_t e = hipFuncSetAttribute((const void*)gemm_f32_tile_kernel<BM, BM, WM, WM, kStepF, kStages, kVec>,
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLds);
    if (e != hipSuccess) return tl_fail(TL_ERR_HIP, "gemm_f32: %s", hipGetErrorString(e));
  }
  gemm_f32_tile_kernel<BM, BM, WM, WM, kStepF, kStages, kVec><<<dim3((unsigned)grid), 256, kLds, stream>>>(A, lda, W, ldw, C, ldc, M, N, K);
  return tl_check_launch("gemm_f32_tile");
}

// Which tile: 128 x 128, 64 x 64 or 32 x 32.  A launch takes as long as the fullest CU, so its time is about fixed + per x
// (blocks of the fullest CU); with K = 2,048 measured 30 + 141 us for the large tile (16,384 columns of 2,048 rows: 1,160 us,
// 118 TFLOP/s), 20 + 39 for the middle one (562 rows of them: 387 against 545 and 461 for the others) and 10 + 12 for the
// small one (2,048 columns of 562 rows: 73 against 94 and 181).  The same figures decide for every K (both parts of a tile's
// time shrink with it): 17 to 2,048 rows of matrices of 64 x 64 to 4,096 x 14,336, 192 products, none slower than by the tiles of
// plain fused multiply-adds before.
int launch_tiles(const float* A, int lda, const float* W, int ldw, float* C, int ldc, int M, int N, int K, hipStream_t stream) {
  const bool vec = K % 4 == 0 && lda % 4 == 0 && ldw % 4 == 0 && ((uintptr_t)A % 16) == 0 && ((uintptr_t)W % 16) == 0;
  const size_t cus = (size_t)tl_device_facts().compute_units;
  auto cost = [&](int tile, double fixed, double per) {
    const size_t blocks = (size_t)((M + tile - 1) / tile) * ((N + tile - 1) / tile);
    return fixed + per * (double)((blocks + cus - 1) / cus);
  };
  const double large = cost(128, 30.0, 141.0), middle = cost(64, 20.0, 39.0), small = cost(32, 10.0, 12.1);
  if (!vec)  // (the large tile's rows would not fit into registers on their way)
    return middle <= small ? launch_tile<64, 32, 32, 2, false>(A, lda, W, ldw, C, ldc, M, N, K, stream)
                           : launch_tile<32, 16, 64, 2, false>(A, lda, W, ldw, C, ldc, M, N, K, stream);
  if (large <= middle && large <= small) return launch_tile<128, 64, 32, 2, true>(A, lda, W, ldw, C, ldc, M, N, K, stream);
  if (middle <= small) return launch_tile<64, 32, 32, 3, true>(A, lda, W, ldw, C, ldc, M, N, K, stream);
  return launch_tile<32, 16, 64, 3, true>(A, lda, W, ldw, C, ldc, M, N, K, stream);
}

}  // namespace

TL_EXPORT int tl_gemm_f32(const float* A, int lda, const float* W, int ldw, float* C, int ldc, int M, int N,
                          int K, hipStream_t stream) {
  TL_REQUIRE(M >= 0 && N > 0 && K > 0, "gemm_f32: bad sizes M=%d N=%d K=%d", M, N, K);
  TL_REQUIRE(lda >= K && ldw >= K && ldc >= N, "gemm_f32: leading dimensions too small");
  if (M == 0) return TL_OK;
  if (M <= 16) {
    // decode steps: the same sums, spread over a wave (see above)
    const unsigned blocks = (N + kRowsWaves * kRowsCols - 1) / (kRowsWaves * kRowsCols);
    const bool vec = K % 4 == 0 && lda % 4 == 0 && ldw % 4 == 0 && ((uintptr_t)A % 16) == 0 && ((uintptr_t)W % 16) == 0;
#define TL_ROWS_LAUNCH(MR)                                                                               \
  do {                                                                                                   \
    const size_t region = (size_t)kRowsCols * MR * kPad > (size_t)kTurned ? (size_t)kRowsCols * MR * kPad : (size_t)kTurned; \
    const size_t lds = ((size_t)MR * BK * kPad + (size_t)kRowsWaves * region) * sizeof(float);               \
    if (lds > 48 * 1024) {                                                                               \
      hipError_t e = hipFuncSetAttribute(vec ? (const void*)gemm_f32_rows_kernel<MR, true>               \
                                             : (const void*)gemm_f32_rows_kernel<MR, false>,             \
                                         hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);          \
      if (e != hipSuccess) return tl_fail(TL_ERR_HIP, "gemm_f32: %s", hipGetErrorString(e));             \
    }                                                                                                    \
    if (vec)                                                                                             \
      gemm_f32_rows_kernel<MR, true><<<blocks, kRowsWaves * kWave, lds, stream>>>(A, lda, W, ldw, C, ldc, M, N, K); \
    else                                                                                                 \
      gemm_f32_rows_kernel<MR, false><<<blocks, kRowsWaves * kWave, lds, stream>>>(A, lda, W, ldw, C, ldc, M, N, K); \
  } while (0)
    if (M == 1) TL_ROWS_LAUNCH(1);
    else if (M == 2) TL_ROWS_LAUNCH(2);
    else if (M <= 4) TL_ROWS_LAUNCH(4);
    else if (M <= 8) TL_ROWS_LAUNCH(8);
    else TL_ROWS_LAUNCH(16);
#undef TL_ROWS_LAUNCH
    return tl_check_launch("gemm_f32_rows");
  }
  return launch_tiles(A, lda, W, ldw, C, ldc, M, N, K, stream);
}
