// Few-rows products whose sums are whole inside one block, for at most 16 rows of X and W in the
// streaming layout of ei_gemm_bf16_skinny_packed: what needs the whole sum (an addition to the stream
// with the squares of the next norm, a gated product, an activation) is done by the block that made it.
#pragma once

#include "common.h"

namespace ei {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kPackedTile = 16 * 32;      // elements of one packed tile: 16 rows x 32 k, 1 KB
constexpr int kStatsWidth = 4096;         // widest row whose norm a product finishes (RowNorm)
constexpr int kStatsParts = kStatsWidth / 16;
constexpr int kWholeRows = 16;            // most rows of X

// Rows of X that are a norm's rows times its weight, not yet divided by their root mean square: the
// sums of the squares of what the norm is taken of, [rows, parts] with 16 or 8 columns each, and the
// norm's eps.  The sums of a row of the product are multiplied by 1 / sqrt(mean + eps).  Sixteen threads
// a row (thread t: row t / 16, part t % 16) ask for its sums before anything else and add them up when
// the products are done.
struct RowNorm {
  const float* squares;
  int parts;
  float eps;
};

template <int MB> struct RowFactors {
  static constexpr int kGroups = kStatsParts / 64;          // of 4 sums a thread
  f32x4 held[MB][kGroups];
  __device__ __forceinline__ void ask(const float* squares, int M, int count, int t) {
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int j = 0; j < kGroups; ++j)       // (surplus threads and groups repeat others)
        held[mb][j] = *reinterpret_cast<const f32x4*>(squares + min(mb * 16 + (t >> 4 & 15), M - 1) * count +
                                                      min(4 * (t & 15) + 64 * j, count - 4));
  }
  // into factor[MB * 16] in LDS; the caller's barrier follows
  __device__ __forceinline__ void finish(float* factor, int count, int width, float eps, int t) const {
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      float sum = 0.f;
#pragma unroll
      for (int j = 0; j < kGroups; ++j)
        if (4 * (t & 15) + 64 * j < count)
          sum += held[mb][j][0] + held[mb][j][1] + held[mb][j][2] + held[mb][j][3];
      sum = row16_sum(sum);
      if (t < 256 && (t & 15) == 0)
        factor[mb * 16 + (t >> 4)] = rsqrtf(sum / static_cast<float>(width) + eps);
    }
  }
};

// What a block does with its sums.  kAddRows: residual[m][n] (float32) += them, in place; `rows` takes
// the new residual times `vector` [N] (the weight of the norm that reads the stream next), rounded,
// and `squares` [M, parts] the sums of the new residual's squares, a block's columns each: with these the norm has no kernel of
// its own, see RowNorm.  kGatedRows: the strips of W alternate between 16 gate rows and their 16 up
// rows; `rows` [M, N / 2] takes the gated product.  kActivatedRows: `rows` [M, N] takes
// activate(sum).  `vector`, where BIAS, is what the sums of the last two start from ([N]).
constexpr int kAddRows = 0, kGatedRows = 1, kActivatedRows = 2;

// A block takes one strip of 16 rows of W (kGatedRows: a gate strip and its up strip) and all of K: its
// waves take every WAVES-th pair of tiles of 32 k (together a cache line of a row of X), and their sums
// meet in LDS.  No wave shares an operand with another, so W and X go straight into registers, DEPTH pairs
// a wave on their way at once, and no barrier stands in the loop; the sums of a row do not depend on
// the other rows.
// Bound by memory: a 8B layer's matrices of 201 and 101 MB at 8 rows take 31.1 and 17.1 us (6.5 and 5.9
// TB/s), small ones two dependent trips to memory (1024 x 2048: 3.5 us of which 1.6 are the launch).
// Measured against the sliced kernel with one slice, gated, 8 rows: 1024 -> 3072 6.7 -> 4.8 us,
// 2048 -> 5632 11.6 -> 11.1, 4096 -> 12288 32.6 -> 31.1; and against the sliced product and the norm's kernel,
// a layer's two at 1 / 8 rows: width 1024 10.6 -> 7.8 / 11.5 -> 9.3 us, 4096 32.0 -> 23.2 / 32.3 -> 25.0.
// HALF (at most 8 rows of X): a block takes 8 rows of W, and a wave's load of a kilobyte holds them for
// both tiles of a pair, as rows 0 .. 7 and 8 .. 15 of the operand; X comes as columns 0 .. 7 for the
// first tile and 8 .. 15 for the second.  The product's diagonal quarters are the two tiles' sums, the
// others are dropped: half the instructions and twice the blocks for the same bytes.  For narrow
// matrices, whose strips leave half the chip idle: at 1 / 8 rows 2048 -> 1024 3.3 / 3.8 -> 3.0 / 3.3 us,
// 3072 -> 1024 4.0 / 4.8 -> 3.3 / 4.2, 8192 -> 2048 8.9 / 10.3 -> 7.6 / 8.9; with a strip for every unit it
// loses (4096 -> 4096, 8 rows: 7.8 -> 8.7).
// With 32 rows every operand of X is twice as large as that of W and it loses (78.8 -> 87 us for
// the four products of a 8B layer), with 16 it still gains (76.3 -> 72.4).
template <int WAVES, int DEPTH, int END, bool STATS, bool BIAS, bool HALF>
__global__ void __launch_bounds__(WAVES * EI_WAVE)
whole_product_kernel(const bf16_t* __restrict__ W, const bf16_t* __restrict__ X, int M, int N, int K,
                     float* __restrict__ residual, const float* __restrict__ vector,
                     bf16_t* __restrict__ rows, float* __restrict__ squares, int parts, float eps,
                     GateAct act) {
  static_assert(END != kAddRows || (!STATS && !BIAS), "the stream takes plain sums");
  static_assert(!HALF || END == kAddRows, "a gate strip and its up strip are whole");
  constexpr int STRIPS = END == kGatedRows ? 2 : 1;
  constexpr int LOADS = HALF ? 1 : 2;       // wave loads of W a strip (and of X) in a pair of tiles
  __shared__ f32x4 sums[WAVES][STRIPS][EI_WAVE];
  const int t = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(t / EI_WAVE), lane = t % EI_WAVE;
  const int r16 = lane & 15, c = lane >> 4;
  const int strips = (N + 15) / 16;
  const int strip = HALF ? blockIdx.x >> 1 : blockIdx.x * STRIPS;
  const int pairs = (K + 63) / 64;
  const int mine = (pairs - wave + WAVES - 1) / WAVES;      // pairs of this wave (may be none)
  const char* w_base = reinterpret_cast<const char*>(W + static_cast<size_t>(strip) * kPackedTile);
  const size_t tile_bytes = static_cast<size_t>(strips) * kPackedTile * sizeof(bf16_t);
  // (rows past the last repeat it; their sums are dropped)
  const int m = min(HALF ? r16 & 7 : r16, M - 1);
  const int second = HALF ? r16 >> 3 : 0;   // the lane's tile of the pair
  const unsigned w_lane = HALF ? second * static_cast<unsigned>(tile_bytes) +
                                     (c * 16 + (blockIdx.x & 1) * 8 + (r16 & 7)) * 16
                               : lane * 16;
  const bf16_t* x_row = X + static_cast<size_t>(m) * K;
  const int x_lane = 32 * second + 8 * c;

  RowFactors<1> factors;
  if constexpr (STATS) factors.ask(squares, M, parts, t);
  bf16x8 w[DEPTH][LOADS][STRIPS], x[DEPTH][LOADS];
  auto load = [&](int d, int i) {           // pair i of this wave, or the last one of all
    const int pair = min(wave + i * WAVES, pairs - 1);
#pragma unroll
    for (int h = 0; h < LOADS; ++h)
#pragma unroll
      for (int s = 0; s < STRIPS; ++s)
        w[d][h][s] = __builtin_nontemporal_load(reinterpret_cast<const bf16x8*>(
            w_base + (2 * pair + h) * tile_bytes + s * kPackedTile * sizeof(bf16_t) + w_lane));
#pragma unroll
    for (int h = 0; h < LOADS; ++h)         // (past K the weights are zeros, whatever finite X meets them)
      x[d][h] = *reinterpret_cast<const bf16x8*>(x_row + min(64 * pair + 32 * h + x_lane, K - 8));
  };
  f32x4 acc[STRIPS];
#pragma unroll
  for (int s = 0; s < STRIPS; ++s) acc[s] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto multiply = [&](int d) {
#pragma unroll
    for (int h = 0; h < LOADS; ++h)
#pragma unroll
      for (int s = 0; s < STRIPS; ++s)
        acc[s] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[d][h][s], x[d][h], acc[s], 0, 0, 0);
  };
#pragma unroll
  for (int d = 0; d < DEPTH; ++d) load(d, d);
  // what the end needs, on its way while the products run (every wave asks, the first one writes: the
  // values of a branch would be waited for where it ends).  Lane (c, r16): columns n0 .. n0 + 3 (HALF:
  // c < 2 and r16 < 8, the other lanes ask for what these do).
  const int n0 = strip * 16 + (HALF ? (blockIdx.x & 1) * 8 + 4 * (c & 1) : 4 * c);
  f32x4 old, extra[STRIPS];
  if constexpr (END == kAddRows) {
    old = *reinterpret_cast<const f32x4*>(residual + static_cast<size_t>(m) * N + n0);
    extra[0] = *reinterpret_cast<const f32x4*>(vector + n0);
  }
  if constexpr (BIAS) {
#pragma unroll
    for (int s = 0; s < STRIPS; ++s)
#pragma unroll
      for (int r = 0; r < 4; ++r) extra[s][r] = vector[min(n0 + 16 * s + r, N - 1)];
  }
  int i = 0;
  for (; i + DEPTH < mine; i += DEPTH) {
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      multiply(d);
      load(d, i + DEPTH + d);
    }
  }
#pragma unroll
  for (int d = 0; d < DEPTH; ++d)
    if (i + d < mine) multiply(d);

  __shared__ float factor[kWholeRows];
#pragma unroll
  for (int s = 0; s < STRIPS; ++s) sums[wave][s][lane] = acc[s];
  if constexpr (STATS) factors.finish(factor, parts, K, eps, t);
  __syncthreads();
  if (wave > 0) return;
  f32x4 v[STRIPS];
#pragma unroll
  for (int s = 0; s < STRIPS; ++s) {
    v[s] = sums[0][s][lane];
#pragma unroll
    for (int k = 1; k < WAVES; ++k) v[s] += sums[k][s][lane];
    if constexpr (HALF) {                   // the second tiles' sums: row r + 8 of W, column m + 8
#pragma unroll
      for (int k = 0; k < WAVES; ++k) v[s] += sums[k][s][(lane + 40) % EI_WAVE];
    }
    if constexpr (STATS) {
#pragma unroll
      for (int r = 0; r < 4; ++r) v[s][r] *= factor[r16];
    }
    if constexpr (BIAS) v[s] += extra[s];
  }
  if constexpr (END == kAddRows) {
    v[0] += old;
    const float own = v[0][0] * v[0][0] + v[0][1] * v[0][1] + v[0][2] * v[0][2] + v[0][3] * v[0][3];
    const float sum = HALF ? own + __shfl_xor(own, 16, EI_WAVE) : rows_sum(own);
    if (r16 >= M || (HALF && c > 1)) return;
    *reinterpret_cast<f32x4*>(residual + static_cast<size_t>(m) * N + n0) = v[0];
    const float y[4] = {v[0][0] * extra[0][0], v[0][1] * extra[0][1], v[0][2] * extra[0][2], v[0][3] * extra[0][3]};
    Vec4<bf16_t>::store(rows + static_cast<size_t>(m) * N + n0, y);
    if (c == 0) squares[static_cast<size_t>(m) * parts + blockIdx.x] = sum;
  } else if constexpr (END == kGatedRows) {
    if (r16 >= M) return;
    float y[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) y[r] = gated_product<bf16_t>(v[0][r], v[STRIPS - 1][r], act);
    Vec4<bf16_t>::store(rows + static_cast<size_t>(m) * (N / 2) + blockIdx.x * 16 + 4 * c, y);
  } else {
    if (r16 >= M) return;
    float y[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) y[r] = activate(v[0][r], act.kind);
    bf16_t* p = rows + static_cast<size_t>(m) * N + n0;
    if (n0 + 3 < N && (N & 3) == 0) {
      Vec4<bf16_t>::store(p, y);
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (n0 + r < N) p[r] = f32_to_bf16(y[r]);
    }
  }
}

// Pairs a wave has on their way: as many as it takes in all where that is little, else the count
// that leaves the last round the fuller (one strip: 8 or 12; two strips: 4 or 8, for the registers).
// Additions with a strip for every compute unit and a K of at most 4096 take eight waves of two pairs
// (4096 -> 4096, 8 rows: 7.8 -> 7.4 us; 12288 -> 4096 is even), half strips of a longer K eight of four.
template <int END, bool STATS, bool BIAS>
void launch_whole_product(const bf16_t* w, const bf16_t* x, int M, int N, int K, float* residual,
                          const float* vector, bf16_t* rows, float* squares, int parts, float eps,
                          const GateAct& act, hipStream_t stream) {
  const int mine = ((K + 63) / 64 + 3) / 4;     // of four waves
  const int strips = (N + 15) / 16;
#define EI_WHOLE(WAVES, DEPTH, HALF, BLOCKS)                                                   \
  whole_product_kernel<WAVES, DEPTH, END, STATS, BIAS, HALF><<<BLOCKS, WAVES * EI_WAVE, 0, stream>>>( \
      w, x, M, N, K, residual, vector, rows, squares, parts, eps, act)
  if constexpr (END == kAddRows) {
    if (parts == N / 8) {
      if (mine <= 4) EI_WHOLE(4, 4, true, parts);
      else if (mine <= 8) EI_WHOLE(4, 8, true, parts);
      else if (mine <= 12) EI_WHOLE(4, 12, true, parts);
      else EI_WHOLE(8, 4, true, parts);
      return;
    }
    if (strips >= 256 && mine > 4 && mine <= 16) {
      EI_WHOLE(8, 2, false, strips);
      return;
    }
  }
  const int blocks = END == kGatedRows ? strips / 2 : strips;
  if (mine <= 4) EI_WHOLE(4, 4, false, blocks);
  else if (END == kGatedRows || (mine + 7) / 8 * 8 < (mine + 11) / 12 * 12) EI_WHOLE(4, 8, false, blocks);
  else EI_WHOLE(4, (END == kGatedRows ? 8 : 12), false, blocks);
#undef EI_WHOLE
}

}  // namespace ei
