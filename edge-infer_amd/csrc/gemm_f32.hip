// True float32 matrix product C[M, N] = A[M, K] . W[N, K]^T for the 32-bit path:
// float32 inputs, float32 fused multiply-adds, no reduced-precision matrix mode.
// W is a checkpoint matrix in its stored [out, in] layout (the reference multiplies
// the same bytes through cublasGemmEx with OP_T, operators/src/cuda/execution.cu:299-324).
//
// The order of an output's sum depends on K alone, so a row's result does not depend on which other
// rows are in the batch, on where the operands lie, nor on which of the kernels below computed it:
// matrix-core kernels for K in fours (few rows, many rows, very many outputs), and one of plain multiply-adds, k in
// ascending order, for every other size.
#include "common.h"

namespace {

constexpr int BM = 64, BN = 64, BK = 16, TM = 4, TN = 4;      // (sizes that are no multiple of 4)

__global__ void __launch_bounds__(256)
gemm_f32_kernel(const float* __restrict__ A, const float* __restrict__ W, float* __restrict__ C,
                int M, int N, int K, long long lda, long long ldw, long long ldc) {
  __shared__ float As[BK][BM + 4];
  __shared__ float Ws[BK][BN + 4];
  const int t = threadIdx.x;
  const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
  const int ty = t / 16, tx = t % 16;
  float acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = 0.f;

  const int lrow = t / 4, lk = (t % 4) * 4;
  for (int k0 = 0; k0 < K; k0 += BK) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int k = k0 + lk + e;
      const int am = m0 + lrow, wn = n0 + lrow;
      As[lk + e][lrow] = (am < M && k < K) ? A[static_cast<size_t>(am) * lda + k] : 0.f;
      Ws[lk + e][lrow] = (wn < N && k < K) ? W[static_cast<size_t>(wn) * ldw + k] : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < BK; ++k) {
      float a[TM], w[TN];
#pragma unroll
      for (int i = 0; i < TM; ++i) a[i] = As[k][ty * TM + i];
#pragma unroll
      for (int j = 0; j < TN; ++j) w[j] = Ws[k][tx * TN + j];
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = fmaf(a[i], w[j], acc[i][j]);
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int m = m0 + ty * TM + i;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int n = n0 + tx * TN + j;
      if (n < N) C[static_cast<size_t>(m) * ldc + n] = acc[i][j];
    }
  }
}

// K in fours (every real model): float32 matrix products, v_mfma_f32_16x16x4_f32, whose
// operands and sums are IEEE float32 like those of a fused multiply-add, at twice the rate of
// v_fma_f32 (packed float32 instructions are not used).  Operands go from global memory straight
// into the lanes that multiply them: lane (i = lane % 16, g = lane / 16) reads the four
// neighbouring values k0 + 4 g .. + 3 of row i, and product s of a step of 16 takes the values
// k0 + 4 g + s of the four lane groups, so one 16-byte load feeds four products.
//
// The sum of an output is cut into kSegs pieces of K, each a chain of products from zero, added as
// a tree, ((c0 + c1) + (c2 + c3)) + ((c4 + c5) + (c6 + c7)).  The pieces depend on K alone and
// the kernels below add them the same way, so a row gives the same bits in each of them, whatever
// other rows there are.
typedef float f32x4 __attribute__((ext_vector_type(4)));
// four neighbouring floats that begin anywhere: one load all the same (global loads of 16 bytes want
// 4-byte alignment), slower only by the cache lines it touches
typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));
constexpr int kSegs = 8, kStep = 16, kFewRowTiles = 4;

__host__ __device__ inline int steps_a_segment(int K) {
  return ((K + kStep - 1) / kStep + kSegs - 1) / kSegs;
}

// The chain of one piece of K for RT x CT tiles of 16 x 16 outputs: rows of A from the pointers
// `a` (one a tile, at the lane's own row and k offset), rows of W from `w`.  The operands of the
// next step are on their way while this one is multiplied.
template <int RT, int CT>
__device__ __forceinline__ void chain(const float* const (&a)[RT], const float* const (&w)[CT], int first,
                                      int last, int k_lane, int K, f32x4 (&acc)[RT][CT]) {
  const f32x4 zero = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int j = 0; j < CT; ++j) acc[i][j] = zero;
  if (first >= last) return;
  f32x4 ax[2][RT], wx[2][CT];
  // (a step beyond the last one is the last one again: asked for, never multiplied)
  auto fetch = [&](int step, f32x4 (&ad)[RT], f32x4 (&wd)[CT]) {
    const int k = min(step, last - 1) * kStep;
    if (k + kStep <= K) {
#pragma unroll
      for (int j = 0; j < CT; ++j) wd[j] = *reinterpret_cast<const f32x4_any*>(w[j] + k);
#pragma unroll
      for (int i = 0; i < RT; ++i) ad[i] = *reinterpret_cast<const f32x4_any*>(a[i] + k);
    } else {                                 // K's own end: the lanes beyond it bring zeros
      const bool live = k + k_lane < K;
#pragma unroll
      for (int j = 0; j < CT; ++j) wd[j] = live ? *reinterpret_cast<const f32x4_any*>(w[j] + k) : zero;
#pragma unroll
      for (int i = 0; i < RT; ++i) ad[i] = live ? *reinterpret_cast<const f32x4_any*>(a[i] + k) : zero;
    }
  };
  auto multiply = [&](const f32x4 (&ad)[RT], const f32x4 (&wd)[CT]) {
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < CT; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(wd[j][s], ad[i][s], acc[i][j], 0, 0, 0);
  };
  fetch(first, ax[0], wx[0]);
  for (int step = first; step < last; step += 2) {
    fetch(step + 1, ax[1], wx[1]);
    multiply(ax[0], wx[0]);
    if (step + 1 < last) {
      fetch(step + 2, ax[0], wx[0]);
      multiply(ax[1], wx[1]);
    }
  }
}

// Many rows: a block of four waves makes 16 RT x 16 CT outputs, every wave all of them for two
// neighbouring pieces of K, the first of which waits in LDS for the second.  No operand goes
// through LDS: a wave's step reads 1 KB a tile row or column for 4 RT CT products of 32 cycles.  What
// bounds it are those loads, whose neighbouring lanes are different rows: 16 bytes a cycle and unit,
// as long as the products of the four waves take.  4 x 4 tiles take 292 registers, a block a unit;
// bound to 256, two blocks fit, but read over each other's cache lines (2,048 rows, 4,096 x 4,096: 665 us
// against 770; 451 rows, 6,144 x 1,024: 76 against 99).
template <int RT, int CT>
__global__ void __launch_bounds__(256)
gemm_f32_tile_kernel(const float* __restrict__ A, const float* __restrict__ W, float* __restrict__ C,
                     int M, int N, int K, long long lda, long long ldw, long long ldc, int col_tiles) {
  __shared__ f32x4 parts[kSegs / 2][RT * CT][EI_WAVE];
  const int lane = threadIdx.x % EI_WAVE, wave = threadIdx.x / EI_WAVE;
  const int i16 = lane % 16, g = lane / 16;
  // Blocks go to the eight dies in turn.  Of few row tiles, those that share a column tile follow
  // each other on one die, whose L2 then serves W to all but the first (192 x 16,000 x 1,024:
  // 80.8 -> 77.0 us); of many, the column tiles come first, which keeps a die's share of both
  // operands small.
  const int row_tiles = (M + 16 * RT - 1) / (16 * RT);
  int row_tile, col_tile;
  if (row_tiles <= kFewRowTiles) {
    const int die = blockIdx.x % 8, there = blockIdx.x / 8;
    row_tile = there % row_tiles;
    col_tile = there / row_tiles * 8 + die;
    if (col_tile >= col_tiles) return;
  } else {
    row_tile = blockIdx.x / col_tiles;
    col_tile = blockIdx.x % col_tiles;
  }
  const int m0 = row_tile * 16 * RT, n0 = col_tile * 16 * CT;
  const float* a[RT];
  const float* w[CT];
#pragma unroll
  for (int i = 0; i < RT; ++i)      // (rows beyond the last: that row again, never stored)
    a[i] = A + static_cast<size_t>(min(m0 + 16 * i + i16, M - 1)) * lda + 4 * g;
#pragma unroll
  for (int j = 0; j < CT; ++j) w[j] = W + static_cast<size_t>(min(n0 + 16 * j + i16, N - 1)) * ldw + 4 * g;
  const int steps = (K + kStep - 1) / kStep, per = steps_a_segment(K);
  f32x4 sum[RT][CT];
  const int from = 2 * wave * per;
  chain<RT, CT>(a, w, min(from, steps), min(from + per, steps), 4 * g, K, sum);
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int j = 0; j < CT; ++j) parts[wave][i * CT + j][lane] = sum[i][j];
  chain<RT, CT>(a, w, min(from + per, steps), min(from + 2 * per, steps), 4 * g, K, sum);
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int j = 0; j < CT; ++j) sum[i][j] += parts[wave][i * CT + j][lane];
  // the tree: neighbours first
#pragma unroll
  for (int apart = 1; apart < kSegs / 2; apart *= 2) {
    if (wave % (2 * apart) == apart) {
#pragma unroll
      for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < CT; ++j) parts[wave][i * CT + j][lane] = sum[i][j];
    }
    __syncthreads();
    if (wave % (2 * apart) == 0) {
#pragma unroll
      for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < CT; ++j) sum[i][j] += parts[wave + apart][i * CT + j][lane];
    }
  }
  if (wave != 0) return;
  const bool quads = ldc % 4 == 0 && (reinterpret_cast<uintptr_t>(C) & 15) == 0;
#pragma unroll
  for (int i = 0; i < RT; ++i) {
    const int m = m0 + 16 * i + i16;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < CT; ++j) {
      const int n = n0 + 16 * j + 4 * g;
      float* dst = C + static_cast<size_t>(m) * ldc + n;
      if (quads && n + 4 <= N) {
        *reinterpret_cast<f32x4*>(dst) = sum[i][j];
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + e < N) dst[e] = sum[i][j][e];
      }
    }
  }
}

// Very many outputs: a block of eight waves makes 128 x 128 of them, a wave 64 x 32, and the operands
// come through LDS, 32 values of K at a time, so a row is read from the caches once for 128 outputs and
// not once for 64, 128 bytes at a time.  A wave goes through all of K; what the pieces of K leave is
// added up as the tree wants it as soon as two neighbours are there (`fold`), so three sums wait at
// most and two waves fit a SIMD (224 registers).  2,048 rows, 151,936 outputs, K 1,024: 5.58 ms, 114
// TFLOP/s (147 the instruction's own rate); the kernel above 8.58, plain multiply-adds from LDS 7.2.
constexpr int kTile = 128, kStage = 2 * kStep, kRowFloats = kStage + 4;   // (LDS rows: no bank twice)
constexpr int kTileThreads = 512;

__global__ void __launch_bounds__(kTileThreads, 2)
gemm_f32_lds_kernel(const float* __restrict__ A, const float* __restrict__ W, float* __restrict__ C,
                    int M, int N, int K, long long lda, long long ldw, long long ldc, int row_tiles,
                    int col_tiles) {
  constexpr int RT = 4, CT = 2;                          // tiles of 16 x 16 a wave
  constexpr int kLoads = kTile * kStage / 4 / kTileThreads;
  __shared__ __attribute__((aligned(16))) float a_lds[2][kTile * kRowFloats];
  __shared__ __attribute__((aligned(16))) float w_lds[2][kTile * kRowFloats];
  // blocks go to the eight dies in turn: those of a die share a column tile, row tile by row tile
  const int die = blockIdx.x % 8, there = blockIdx.x / 8;
  const int row_tile = there % row_tiles, col_tile = there / row_tiles * 8 + die;
  if (col_tile >= col_tiles) return;
  const int m0 = row_tile * kTile, n0 = col_tile * kTile;
  const int lane = threadIdx.x % EI_WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / EI_WAVE);
  const int i16 = lane % 16, g = lane / 16;
  const int wm = wave / 4 * 64, wn = wave % 4 * 32;      // the wave's part of the block's tile
  const f32x4 zero = f32x4{0.f, 0.f, 0.f, 0.f};
  // thread -> piece f = t + 512 u of a stage: row f / 8, floats 4 (f % 8) .. + 3
  const int piece = threadIdx.x % 8 * 4;
  const float* a_row[kLoads];
  const float* w_row[kLoads];
  int at_lds[kLoads];
#pragma unroll
  for (int u = 0; u < kLoads; ++u) {
    const int row = threadIdx.x / 8 + u * (kTileThreads / 8);
    a_row[u] = A + static_cast<size_t>(min(m0 + row, M - 1)) * lda + piece;
    w_row[u] = W + static_cast<size_t>(min(n0 + row, N - 1)) * ldw + piece;
    at_lds[u] = row * kRowFloats + piece;
  }
  f32x4 a_next[kLoads], w_next[kLoads];
  auto fetch = [&](int k0) __attribute__((always_inline)) {
    const bool live = k0 + piece < K;
#pragma unroll
    for (int u = 0; u < kLoads; ++u) {
      a_next[u] = live ? *reinterpret_cast<const f32x4_any*>(a_row[u] + k0) : zero;
      w_next[u] = live ? *reinterpret_cast<const f32x4_any*>(w_row[u] + k0) : zero;
    }
  };
  f32x4 acc[RT][CT], one[RT][CT], two[RT][CT], four[RT][CT];   // sums of that many pieces of K
  auto each = [&](auto&& f) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int j = 0; j < CT; ++j) f(i, j);
  };
  each([&](int i, int j) { acc[i][j] = one[i][j] = two[i][j] = four[i][j] = zero; });
  // piece `seg` is there: it, and what it completes, joins its neighbour
  auto fold = [&](int seg) __attribute__((always_inline)) {
    if (seg % 2 == 0) {
      each([&](int i, int j) { one[i][j] = acc[i][j]; });
    } else {
      each([&](int i, int j) { acc[i][j] = one[i][j] + acc[i][j]; });
      if (seg % 4 == 1) {
        each([&](int i, int j) { two[i][j] = acc[i][j]; });
      } else {
        each([&](int i, int j) { acc[i][j] = two[i][j] + acc[i][j]; });
        if (seg % 8 == 3) each([&](int i, int j) { four[i][j] = acc[i][j]; });
        else each([&](int i, int j) { four[i][j] = four[i][j] + acc[i][j]; });
      }
    }
    each([&](int i, int j) { acc[i][j] = zero; });
  };
  const int steps = (K + kStep - 1) / kStep, per = steps_a_segment(K), stages = (steps + 1) / 2;
  fetch(0);
  int seg = 0, left = per;                               // the piece of K, and the steps left of it
  for (int stage = 0; stage < stages; ++stage) {
    float* a_now = a_lds[stage % 2];
    float* w_now = w_lds[stage % 2];
#pragma unroll
    for (int u = 0; u < kLoads; ++u) {
      *reinterpret_cast<f32x4*>(a_now + at_lds[u]) = a_next[u];
      *reinterpret_cast<f32x4*>(w_now + at_lds[u]) = w_next[u];
    }
    // (the other half is read no more: every wave has passed the last barrier behind its reads)
    __syncthreads();
    if (stage + 1 < stages) fetch((stage + 1) * kStage);
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      if (2 * stage + half < steps) {
        f32x4 ad[RT], wd[CT];
#pragma unroll
        for (int i = 0; i < RT; ++i)
          ad[i] = *reinterpret_cast<const f32x4*>(a_now + (wm + 16 * i + i16) * kRowFloats + kStep * half + 4 * g);
#pragma unroll
        for (int j = 0; j < CT; ++j)
          wd[j] = *reinterpret_cast<const f32x4*>(w_now + (wn + 16 * j + i16) * kRowFloats + kStep * half + 4 * g);
#pragma unroll
        for (int s = 0; s < 4; ++s)
          each([&](int i, int j) {
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(wd[j][s], ad[i][s], acc[i][j], 0, 0, 0);
          });
        if (--left == 0) {
          fold(seg++);
          left = per;
        }
      }
    }
  }
  for (; seg < kSegs; ++seg) fold(seg);                  // (pieces cut short, and those without a step)
  const bool quads = ldc % 4 == 0 && (reinterpret_cast<uintptr_t>(C) & 15) == 0;
#pragma unroll
  for (int i = 0; i < RT; ++i) {
    const int m = m0 + wm + 16 * i + i16;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < CT; ++j) {
      const int n = n0 + wn + 16 * j + 4 * g;
      float* dst = C + static_cast<size_t>(m) * ldc + n;
      if (quads && n + 4 <= N) {
        *reinterpret_cast<f32x4*>(dst) = four[i][j];
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + e < N) dst[e] = four[i][j][e];
      }
    }
  }
}

// Few rows (decode): bound by how fast the weights arrive.  A block of eight waves owns 16 CT rows
// of W, a wave a piece of K; X of up to 16 RT rows is read from the caches beside it (twice as
// many rows of W for every X where that leaves enough blocks).  Two steps are asked for while
// two are multiplied: more of them cost waves a SIMD and read slower (622 MB, one row: 2 + 2
// steps 119 us, 4 + 4 steps 140, 8 + 8 steps 157).
//
// Where strips of 16 rows leave units without a block, a block owns ROWS = 8 (the instruction's other
// rows repeat them and are not stored) and asks for DEEP = 4 steps at a time: what bounds it there is
// how long a wave's own piece takes to arrive (one row, 2,048 -> 1,024: 9.2 -> 8.0 us, 3,072 -> 1,024:
// 12.6 -> 10.5; 4 rows a block read no faster, 8 steps at a time neither).
template <int RT, int CT, int ROWS = 16, int DEEP = 2>
__global__ void __launch_bounds__(512)
gemm_f32_few_kernel(const float* __restrict__ A, const float* __restrict__ W, float* __restrict__ C,
                    int M, int N, int K, long long lda, long long ldw, long long ldc) {
  constexpr int kDeep = DEEP;
  static_assert(ROWS == 16 || CT == 1, "narrow strips come one a block");
  __shared__ f32x4 parts[kSegs][RT * CT][EI_WAVE];
  const int lane = threadIdx.x % EI_WAVE, wave = threadIdx.x / EI_WAVE;
  const int i16 = lane % 16, g = lane / 16;
  const int n0 = blockIdx.x * ROWS * CT;
  const f32x4 zero = f32x4{0.f, 0.f, 0.f, 0.f};
  const float* w[CT];
#pragma unroll
  for (int j = 0; j < CT; ++j)
    w[j] = W + static_cast<size_t>(min(n0 + 16 * j + i16 % ROWS, N - 1)) * ldw + 4 * g;
  const float* a[RT];
  bool row_live[RT];
#pragma unroll
  for (int i = 0; i < RT; ++i) {
    row_live[i] = 16 * i + i16 < M;
    a[i] = A + static_cast<size_t>(min(16 * i + i16, M - 1)) * lda + 4 * g;
  }
  const int steps = (K + kStep - 1) / kStep, per = steps_a_segment(K);
  const int first = min(wave * per, steps), last = min(first + per, steps);
  f32x4 acc[RT][CT];
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int j = 0; j < CT; ++j) acc[i][j] = zero;
  f32x4 wx[2][kDeep][CT], ax[2][kDeep][RT];
  auto fetch = [&](int step, f32x4 (&wd)[kDeep][CT], f32x4 (&ad)[kDeep][RT]) {
#pragma unroll
    for (int u = 0; u < kDeep; ++u) {
      const int k = (step + u) * kStep;
      const bool live = step + u < last && k + 4 * g < K;
#pragma unroll
      for (int j = 0; j < CT; ++j) wd[u][j] = live ? *reinterpret_cast<const f32x4_any*>(w[j] + k) : zero;
#pragma unroll
      for (int i = 0; i < RT; ++i)
        ad[u][i] = (live && row_live[i]) ? *reinterpret_cast<const f32x4_any*>(a[i] + k) : zero;
    }
  };
  auto multiply = [&](int step, const f32x4 (&wd)[kDeep][CT], const f32x4 (&ad)[kDeep][RT]) {
#pragma unroll
    for (int u = 0; u < kDeep; ++u) {
      if (step + u < last) {
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
          for (int i = 0; i < RT; ++i)
#pragma unroll
            for (int j = 0; j < CT; ++j)
              acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(wd[u][j][s], ad[u][i][s], acc[i][j], 0, 0, 0);
      }
    }
  };
  fetch(first, wx[0], ax[0]);
  for (int step = first; step < last; step += 2 * kDeep) {
    if (step + kDeep < last) fetch(step + kDeep, wx[1], ax[1]);
    multiply(step, wx[0], ax[0]);
    if (step + kDeep < last) {
      if (step + 2 * kDeep < last) fetch(step + 2 * kDeep, wx[0], ax[0]);
      multiply(step + kDeep, wx[1], ax[1]);
    }
  }
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int j = 0; j < CT; ++j) parts[wave][i * CT + j][lane] = acc[i][j];
  __syncthreads();
  const bool quads = ldc % 4 == 0 && (reinterpret_cast<uintptr_t>(C) & 15) == 0;
  for (int at = threadIdx.x; at < RT * CT * EI_WAVE; at += 512) {
    const int tile = at / EI_WAVE, l = at % EI_WAVE;
    f32x4 c[kSegs];
#pragma unroll
    for (int s = 0; s < kSegs; ++s) c[s] = parts[s][tile][l];
    const f32x4 sum = ((c[0] + c[1]) + (c[2] + c[3])) + ((c[4] + c[5]) + (c[6] + c[7]));
    const int m = 16 * (tile / CT) + l % 16, n = n0 + 16 * (tile % CT) + 4 * (l / 16);
    if (m >= M || 4 * (l / 16) >= ROWS) continue;
    float* dst = C + static_cast<size_t>(m) * ldc + n;
    if (quads && n + 4 <= N) {
      *reinterpret_cast<f32x4*>(dst) = sum;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (n + e < N) dst[e] = sum[e];
    }
  }
}

}  // namespace

extern "C" int ei_gemm_f32(const float* A, const float* W, float* C, int M, int N, int K,
                           long long lda, long long ldw, long long ldc, hipStream_t stream) {
  EI_REQUIRE(M > 0 && N > 0 && K > 0, "gemm_f32: sizes must be positive");
  EI_REQUIRE(A && W && C, "gemm_f32: null pointer");
  EI_REQUIRE(lda >= K && ldw >= K && ldc >= N, "gemm_f32: leading dimension too small");
  const bool fours = K % 4 == 0;
  if (fours && M <= 64) {
    // (two strips a block where the chip still gets eight blocks a unit)
    const bool wide = (N + 31LL) / 32 >= 8LL * ei_compute_units();
#define EI_FEW(RT, CT)                                                                   \
  gemm_f32_few_kernel<RT, CT><<<static_cast<unsigned>((N + 16LL * CT - 1) / (16 * CT)), 512, 0, stream>>>( \
      A, W, C, M, N, K, lda, ldw, ldc)
    // Up to 16 rows and at most a strip of 8 a unit: strips of 8 (1,024 outputs, K 3,072: 12.6 -> 10.5
    // us at one row, 15.0 -> 14.3 at 16; K 1,024 and 16 rows: 5.8 against 6.0, left as it was).  Up to
    // 4 rows and at most a strip of 16 a unit: 4 steps at a time (4,096 outputs, K 1,024: 7.0 -> 6.5 us;
    // at 16 rows, K 4,096, 20.0 against 21.1; with more strips than units 9.0 against 9.3).
    const long long units_few = ei_compute_units();
    if ((N + 7LL) / 8 <= units_few && (M <= 8 || (M <= 16 && K >= 2048))) {
      gemm_f32_few_kernel<1, 1, 8, 4><<<static_cast<unsigned>((N + 7LL) / 8), 512, 0, stream>>>(
          A, W, C, M, N, K, lda, ldw, ldc);
    } else if ((N + 15LL) / 16 <= units_few && M <= 4) {
      gemm_f32_few_kernel<1, 1, 16, 4><<<static_cast<unsigned>((N + 15LL) / 16), 512, 0, stream>>>(
          A, W, C, M, N, K, lda, ldw, ldc);
    } else if (M <= 16) {
      if (wide) EI_FEW(1, 2);
      else EI_FEW(1, 1);
    } else if (M <= 32) {
      if (wide) EI_FEW(2, 2);
      else EI_FEW(2, 1);
    } else {
      if (wide) EI_FEW(4, 2);
      else EI_FEW(4, 1);
    }
#undef EI_FEW
    EI_LAUNCH_CHECK();
  }
  if (fours) {
    const long long units = ei_compute_units();
    auto blocks_of = [&](int rt, int ct) {
      return ((M + 16LL * rt - 1) / (16 * rt)) * ((N + 16LL * ct - 1) / (16 * ct));
    };
    auto grid_of = [&](int rt, int ct) {
      const long long rows = (M + 16LL * rt - 1) / (16 * rt), cols = (N + 16LL * ct - 1) / (16 * ct);
      return rows * (rows <= kFewRowTiles ? (cols + 7) / 8 * 8 : cols);
    };
    // Blocks of 128 x 128 where they are done sooner: a unit holds one at a time, and a round of them over
    // the chip lasts as long as three rounds of 64 x 64 tiles (K 1,024: 75 to 78 us against 25 to 29).  Rows x
    // outputs x K, us by 128 x 128 and by 64 x 64: taken 1,024 x 4,096 x 1,024 78 and 100, 513 x 6,144 x 2,048
    // 150 and 179, 100 x 151,936 x 1,024 380 and 525, 2,048 x 24,576 x 4,096 3,520 and 4,650; left, a last round
    // being nearly empty, 261 x 11,264 x 2,048 290 and 181, 800 x 6,144 x 4,096 583 and 421.  Over 220 products of
    // 65 to 3,554 rows the choice is within 3 % of the better of the two.
    const long long big_rows = (M + kTile - 1LL) / kTile, big_cols = (N + kTile - 1LL) / kTile;
    const long long big = big_rows * ((big_cols + 7) / 8 * 8);
    const long long big_rounds = (big_rows * big_cols + units - 1) / units;
    const long long small_rounds = (blocks_of(4, 4) + units - 1) / units;
    if (3 * big_rounds < small_rounds) {
      EI_REQUIRE(big <= 0x7fffffff, "gemm_f32: too many outputs for one launch");
      gemm_f32_lds_kernel<<<static_cast<unsigned>(big), kTileThreads, 0, stream>>>(
          A, W, C, M, N, K, lda, ldw, ldc, static_cast<int>(big_rows), static_cast<int>(big_cols));
      EI_LAUNCH_CHECK();
    }
    EI_REQUIRE(grid_of(2, 2) <= 0x7fffffff || blocks_of(4, 4) <= 0x7ffffff0,
               "gemm_f32: too many outputs for one launch");
    // else the largest tile that leaves no compute unit without a block
#define EI_TILE(RT, CT)                                                                     \
  gemm_f32_tile_kernel<RT, CT><<<static_cast<unsigned>(grid_of(RT, CT)), 256, 0, stream>>>( \
      A, W, C, M, N, K, lda, ldw, ldc, (N + 16 * CT - 1) / (16 * CT))
    if (blocks_of(4, 4) >= units) EI_TILE(4, 4);
    else if (blocks_of(2, 4) >= units) EI_TILE(2, 4);
    else EI_TILE(2, 2);
#undef EI_TILE
    EI_LAUNCH_CHECK();
  }
  const long long gy = (M + BM - 1) / BM;
  EI_REQUIRE(gy <= 65535, "gemm_f32: too many rows for one launch");
  dim3 grid((N + BN - 1) / BN, static_cast<unsigned>(gy));
  gemm_f32_kernel<<<grid, 256, 0, stream>>>(A, W, C, M, N, K, lda, ldw, ldc);
  EI_LAUNCH_CHECK();
}
