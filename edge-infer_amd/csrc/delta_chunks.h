// The gated delta rule over a prompt's rows in chunks of 64 tokens:
//
//   S <- g_t S;  u_t = beta_t (v_t - S^T k_t);  S <- S + k_t u_t^T;  o_t = S^T q_t
//
// With c_t the product of a chunk's decays up to token t and S_0 the state before the chunk, the
// chunk's u solve a triangular system, (I + A) U = diag(beta) (V - diag(c) K S_0) with
// A[t, s] = beta_t (c_t / c_s) (k_t . k_s), s < t, and
//
//   S_n = c_n S_0 + sum_s (c_n / c_s) k_s u_s^T     o_t = c_t S_0^T q_t + sum_{s <= t} (c_t / c_s) (q_t . k_s) u_s
//
// `solve` does what needs no state, all chunks side by side: the matrices of the system, its solutions
// for the right sides diag(beta) V and diag(beta c) K, and the operands below.  `walk` takes the chunks
// of a sequence in order, 16 columns of S a block: U = U_v - W S, the outputs, and S.  Everything
// is float32 on v_mfma_f32_16x16x4_f32 and 32x32x2 (IEEE float32 operands and sums); decays' ratios
// are exponentials of differences of float64 sums.
//
// An accumulator of the 16x16x4 product holds rows 4 g + r (r = 0 .. 3, g = lane / 16) of column
// lane % 16, which is also how that product wants a B operand whose four k values of step r are
// 4 g + r: a sum can be multiplied on without leaving its registers, the A operand's lane then
// bringing four neighbouring k values.
//
// Causality holds for values that are not finite too: where the system's right sides or U hold such a
// one, the products with matrices that are zero above the diagonal are taken term by term (zero
// times infinity is not zero).
//
// What bounds it: the walk is a chain over chunks of 112 products (of 32 cycles) a wave, two barriers
// and 116 KB of operands a block, 2.9 us a chunk of one sequence.  2,048 tokens of 16 heads of 128 x
// 128: 671 us token by token, 128 by chunks (solve 34, walk 93); 8 x 512: 298 and 151.
#pragma once
#include "recurrence_chunks.h"

namespace ei {
namespace delta_chunks {

using chunks::any_not_finite;
using chunks::chunk_place;
using chunks::rows_of;
using chunks::f32x16;
using chunks::f32x4;
using chunks::Gates;
using chunks::Sequences;
using chunks::State;

constexpr int kTokens = 64;
constexpr int kThreads = 256;

// A chunk's scratch of one head: W [64][DK], the queries times c_t [64][DK], the keys times c_n / c_t
// transposed [DK][64], the weights of the values [64][64], U_v [64][DV], c_n.  All but the last
// lie by tiles of 16 x 16, a tile as its 64 lanes want it (four floats a lane, a kilobyte a load):
// neighbouring lanes of an operand are different rows, and loads of rows far apart take the
// compute unit's address path four times as long (2,048 tokens: the walk 147 -> 92 us).
template <int DK, int DV>
struct Scratch {
  static constexpr int w = 0, q = w + kTokens * DK, k = q + kTokens * DK, p = k + DK * kTokens,
                       u = p + kTokens * kTokens, whole = u + kTokens * DV, floats = whole + 4;
};

// Where element (row, col) of an A operand `cols` wide lies.
__device__ __forceinline__ int operand_at(int row, int col, int cols) {
  return ((row / 16 * (cols / 16) + col / 16) * EI_WAVE + col % 16 / 4 * 16 + row % 16) * 4 + col % 4;
}

struct Rows {               // float32 rows: q, k (one of `share` heads), v
  const float* rows;
  size_t stride;
  int q, k, v, share;
  float q_scale, unit_eps;
};

// A barrier that orders what went through LDS and leaves loads from global memory on their way
// (__syncthreads waits for all of them).
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// A block of eight waves a (head, chunk, sequence).
constexpr int kSolvers = 512;

template <int DK, int DV>
__global__ void __launch_bounds__(kSolvers, 4)
solve_kernel(Rows in, Gates gates, Sequences seqs, float* __restrict__ scratch) {
  typedef Scratch<DK, DV> At;
  constexpr int QS = DK + 4, AS = kTokens + 4, TS = 20, kWaves = kSolvers / EI_WAVE;
  __shared__ __attribute__((aligned(16))) float q_lds[kTokens * QS];
  __shared__ __attribute__((aligned(16))) float k_lds[kTokens * QS];
  // (the queries' place, once they are done with: minus A, and the inverses of its diagonal blocks;
  // two blocks then fit a compute unit)
  static_assert(kTokens * AS + 4 * 16 * TS <= kTokens * QS || DK < 128, "A and the inverses in the queries' place");
  __shared__ __attribute__((aligned(16))) float a_own[DK < 128 ? kTokens * AS + 4 * 16 * TS : 4];
  float* a_lds = DK < 128 ? a_own : q_lds;
  float* t_lds = a_lds + kTokens * AS;
  __shared__ double log_sums[kTokens];
  __shared__ float betas[kTokens], from_start[kTokens], to_end[kTokens];
  const int head = blockIdx.x, chunk = blockIdx.y, seq = blockIdx.z;
  const int nt = min(kTokens, rows_of(seqs, seq) - chunk * kTokens);
  if (nt <= 0) return;
  const int first = seqs.row0[seq] + chunk * kTokens;
  float* mine = scratch + (chunk_place(seqs, seq, chunk) * gridDim.x + head) * At::floats;
  const int lane = threadIdx.x % EI_WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / EI_WAVE);
  const int i16 = lane % 16, g = lane / 16;
  {
    // the unit keys and the scaled unit queries: DK / 4 neighbouring lanes a row
    constexpr int kPieces = DK / 4, kLoads = kTokens * kPieces / kSolvers;
    const float* q_at = in.rows + in.q + (head / in.share) * DK;
    const float* k_at = in.rows + in.k + (head / in.share) * DK;
    f32x4 q4[kLoads], k4[kLoads];
#pragma unroll
    for (int u = 0; u < kLoads; ++u) {
      const int i = threadIdx.x + u * kSolvers;
      const size_t at = static_cast<size_t>(first + min(i / kPieces, nt - 1)) * in.stride + i % kPieces * 4;
      q4[u] = *reinterpret_cast<const f32x4*>(q_at + at);
      k4[u] = *reinterpret_cast<const f32x4*>(k_at + at);
    }
    if (wave == kWaves - 1) {        // lane t: token t's gates (beyond the end: no decay, no write)
      double each = 0.0;
      float beta = 0.f;
      if (lane < nt) {
        const size_t row = static_cast<size_t>(first) + lane;
        beta = 1.0f / (1.0f + expf(-chunks::gate_column(gates, row, gates.at + head)));
        const float z = chunks::gate_column(gates, row, gates.at2 + head) + gates.c1[head];
        const float soft = z > 30.f ? z : log1pf(expf(z));
        each = chunks::bounded_log(-static_cast<double>(expf(gates.c0[head])) * soft);
      }
#pragma unroll
      for (int step = 1; step < kTokens; step *= 2) {
        const double other = __shfl_up(each, step, EI_WAVE);
        if (lane >= step) each += other;
      }
      const double whole = __shfl(each, EI_WAVE - 1, EI_WAVE);
      log_sums[lane] = each;
      betas[lane] = beta;
      from_start[lane] = expf(static_cast<float>(each));
      to_end[lane] = expf(static_cast<float>(whole - each));
      if (lane == 0) mine[At::whole] = expf(static_cast<float>(whole));
    }
#pragma unroll
    for (int u = 0; u < kLoads; ++u) {
      const int i = threadIdx.x + u * kSolvers;
      float qq = (q4[u][0] * q4[u][0] + q4[u][1] * q4[u][1]) + (q4[u][2] * q4[u][2] + q4[u][3] * q4[u][3]);
      float kk = (k4[u][0] * k4[u][0] + k4[u][1] * k4[u][1]) + (k4[u][2] * k4[u][2] + k4[u][3] * k4[u][3]);
#pragma unroll
      for (int apart = 1; apart < kPieces; apart *= 2) {
        qq += __shfl_xor(qq, apart, kPieces);
        kk += __shfl_xor(kk, apart, kPieces);
      }
      const float qf = in.q_scale / sqrtf(qq + in.unit_eps), kf = 1.0f / sqrtf(kk + in.unit_eps);
      *reinterpret_cast<f32x4*>(q_lds + i / kPieces * QS + i % kPieces * 4) = q4[u] * qf;
      *reinterpret_cast<f32x4*>(k_lds + i / kPieces * QS + i % kPieces * 4) = k4[u] * kf;
    }
  }
  __syncthreads();
  // right sides: 16 columns a tile of diag(beta c) K, then of diag(beta) V, asked for early
  constexpr int kTiles = (DK + DV) / 16, kMine = (kTiles + kWaves - 1) / kWaves;
  f32x4 x[4][kMine];
#pragma unroll
  for (int c = 0; c < kMine; ++c) {
    const int col = (wave * kMine + c) * 16 + i16;
    const float* v_at = in.rows + in.v + head * DV + col - DK;
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int t = 16 * b + 4 * g + r;
        x[b][c][r] = col < DK ? k_lds[t * QS + col]
                     : col < DK + DV ? v_at[static_cast<size_t>(first + min(t, nt - 1)) * in.stride] : 0.f;
      }
  }
  // k k^T and q k^T in tiles of 16 x 16 on and below the diagonal, ten of each, in turn
  constexpr int kBlocks = 10, kTurns = (2 * kBlocks + kWaves - 1) / kWaves;
  f32x4 product[kTurns];
  auto block_row = [](int n) { return n < 1 ? 0 : n < 3 ? 1 : n < 6 ? 2 : 3; };
#pragma unroll
  for (int turn = 0; turn < kTurns; ++turn) {
    const int n = turn * kWaves + wave;
    if (n < 2 * kBlocks) {
      const int m = n % kBlocks, rb = block_row(m), cb = m - rb * (rb + 1) / 2;
      const float* left = (n < kBlocks ? k_lds : q_lds) + (16 * rb + i16) * QS + 4 * g;
      const float* right = k_lds + (16 * cb + i16) * QS + 4 * g;
      f32x4 sums[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) sums[u] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < DK / 16; ++j) {
        const f32x4 l4 = *reinterpret_cast<const f32x4*>(left + 16 * j);
        const f32x4 r4 = *reinterpret_cast<const f32x4*>(right + 16 * j);
#pragma unroll
        for (int r = 0; r < 4; ++r)
          sums[r] = __builtin_amdgcn_mfma_f32_16x16x4f32(l4[r], r4[r], sums[r], 0, 0, 0);
      }
      product[turn] = (sums[0] + sums[1]) + (sums[2] + sums[3]);
    }
  }
  // the queries and keys of the walk, and zeros above the diagonal of the weights
#pragma unroll 4
  for (int tile = wave; tile < 4 * (DK / 16); tile += kWaves) {
    const int t = tile / (DK / 16) * 16, k = tile % (DK / 16) * 16;
    *reinterpret_cast<f32x4*>(mine + At::q + (tile * EI_WAVE + lane) * 4) =
        *reinterpret_cast<const f32x4*>(q_lds + (t + i16) * QS + k + 4 * g) * from_start[t + i16];
  }
#pragma unroll 4
  for (int tile = wave; tile < 4 * (DK / 16); tile += kWaves) {
    const int k = tile / 4 * 16 + i16, t = tile % 4 * 16 + 4 * g;
    f32x4 v;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = k_lds[(t + e) * QS + k] * to_end[t + e];
    *reinterpret_cast<f32x4*>(mine + At::k + (tile * EI_WAVE + lane) * 4) = v;
  }
  if (wave < 6) {
    const int rb = wave < 3 ? 0 : wave < 5 ? 1 : 2, cb = wave < 3 ? wave + 1 : wave < 5 ? wave - 1 : 3;
    *reinterpret_cast<f32x4*>(mine + At::p + ((rb * 4 + cb) * EI_WAVE + lane) * 4) = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  __syncthreads();
#pragma unroll
  for (int turn = 0; turn < kTurns; ++turn) {
    const int n = turn * kWaves + wave;
    if (n < 2 * kBlocks) {
      const int m = n % kBlocks, rb = block_row(m), cb = m - rb * (rb + 1) / 2;
      const int s = 16 * cb + i16;
      const double ls = log_sums[s];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int t = 16 * rb + 4 * g + r;
        const float ratio = s <= t ? expf(static_cast<float>(log_sums[t] - ls)) : 0.f;
        if (n < kBlocks) a_lds[t * AS + s] = s < t ? -product[turn][r] * (ratio * betas[t]) : 0.f;
        else mine[At::p + operand_at(t, s, kTokens)] = product[turn][r] * ratio;
      }
    }
  }
#pragma unroll
  for (int c = 0; c < kMine; ++c)
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int t = 16 * b + 4 * g + r;
        x[b][c][r] *= (wave * kMine + c) * 16 < DK ? betas[t] * from_start[t] : betas[t];
      }
  __syncthreads();
  if (wave < 4) {
    // (I + A)^-1 of a diagonal block of 16 a wave, a column a lane (four lanes the same)
    const float* a = a_lds + wave * 16 * AS + wave * 16;
    float y[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      float sums[4] = {i == i16 ? 1.f : 0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int m0 = 0; m0 < i; m0 += 4) {
        const f32x4 row = *reinterpret_cast<const f32x4*>(a + i * AS + m0);
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (m0 + e < i) sums[e] = fmaf(row[e], y[m0 + e], sums[e]);
      }
      y[i] = (sums[0] + sums[1]) + (sums[2] + sums[3]);
    }
    if (g == 0) {
#pragma unroll
      for (int i = 0; i < 16; ++i) t_lds[(wave * 16 + i) * TS + i16] = y[i];
    }
  }
  __syncthreads();
  // the system, block row by block row
#pragma unroll
  for (int b = 0; b < 4; ++b) {
#pragma unroll
    for (int before = 0; before < b; ++before) {
      const f32x4 a = *reinterpret_cast<const f32x4*>(a_lds + (16 * b + i16) * AS + 16 * before + 4 * g);
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int c = 0; c < kMine; ++c)
          x[b][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[r], x[before][c][r], x[b][c], 0, 0, 0);
    }
    const f32x4 inv = *reinterpret_cast<const f32x4*>(t_lds + (16 * b + i16) * TS + 4 * g);
    f32x4 solved[kMine];
#pragma unroll
    for (int c = 0; c < kMine; ++c) solved[c] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int c = 0; c < kMine; ++c)
        solved[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(inv[r], x[b][c][r], solved[c], 0, 0, 0);
    float met = 0.f;
#pragma unroll
    for (int c = 0; c < kMine; ++c) met += solved[c][0] * 0.f;
    if (any_not_finite(met)) {
#pragma unroll
      for (int c = 0; c < kMine; ++c) {
        f32x4 sum = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int m = 0; m < 16; ++m) {
          const float xm = __shfl(x[b][c][m % 4], m / 4 * 16 + i16, EI_WAVE);
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (m <= 4 * g + r) sum[r] += t_lds[(16 * b + 4 * g + r) * TS + m] * xm;
        }
        solved[c] = sum;
      }
    }
#pragma unroll
    for (int c = 0; c < kMine; ++c) {
      x[b][c] = solved[c];
      const int tile = wave * kMine + c;
      if (tile < DK / 16) {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          mine[At::w + operand_at(16 * b + 4 * g + r, tile * 16 + i16, DK)] = solved[c][r];
      } else if (tile < kTiles) {        // (as an accumulator holds it)
        *reinterpret_cast<f32x4*>(mine + At::u + ((b * (DV / 16) + tile - DK / 16) * EI_WAVE + lane) * 4) = solved[c];
      }
    }
  }
}

// A block a (head, sequence, 16 NC columns of S), wave w having rows 16 (DK / 64) w on of S and tokens
// 16 w .. 16 w + 15 of a chunk.  A chunk's operands are asked for a chunk ahead.  (Keys of 64 and 32
// columns: bound to the registers that let a SIMD hold two waves.)
template <int DK, int DV, int NC>
__global__ void __launch_bounds__(kThreads, DK == 64 && NC == 2 ? 2 : 1)
walk_kernel(State state, Sequences seqs, const float* __restrict__ scratch, float* __restrict__ out) {
  typedef Scratch<DK, DV> At;
  constexpr int KT = DK / 64;                    // tiles of 16 rows of S a wave
  constexpr int SS = DK + 4, US = kTokens + 4;
  __shared__ __attribute__((aligned(16))) float s_lds[NC * 16 * SS];      // S by columns
  __shared__ __attribute__((aligned(16))) float u_lds[NC * 16 * US];      // U by columns
  const int head = blockIdx.x, seq = blockIdx.y, col0 = blockIdx.z * 16 * NC;
  const int count = rows_of(seqs, seq);
  if (count <= 0) return;
  const int n_chunks = (count + kTokens - 1) / kTokens;
  const int lane = threadIdx.x % EI_WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / EI_WAVE);
  const int i16 = lane % 16, g = lane / 16;
  const size_t apart = static_cast<size_t>(gridDim.x) * At::floats;
  const float* base = scratch + (chunk_place(seqs, seq, 0) * gridDim.x + head) * At::floats;
  // S of a head lies in the table by columns, [DV][DK]
  const size_t column = head * state.head_floats + static_cast<size_t>(col0 + i16) * DK;
  const float* in = state.rows + static_cast<size_t>(seqs.in[seq]) * state.row_floats + column;
  float* to = state.rows + static_cast<size_t>(seqs.out[seq]) * state.row_floats + column;
  f32x4 S[NC][KT];
#pragma unroll
  for (int n = 0; n < NC; ++n)
#pragma unroll
    for (int i = 0; i < KT; ++i) {
      const int k = (wave * KT + i) * 16 + 4 * g;
      S[n][i] = *reinterpret_cast<const f32x4*>(in + static_cast<size_t>(n) * 16 * DK + k);
      *reinterpret_cast<f32x4*>(s_lds + (16 * n + i16) * SS + k) = S[n][i];
    }
  struct Operands {
    f32x4 w[DK / 16], q[DK / 16], k[KT][4], p[4], u[NC];
    float whole;
  };
  auto ask = [&](Operands& o, int c) __attribute__((always_inline)) {
    const float* at = base + min(c, n_chunks - 1) * apart + lane * 4;
    auto tile = [&](int from, int index) { return *reinterpret_cast<const f32x4*>(at + from + index * EI_WAVE * 4); };
#pragma unroll
    for (int j = 0; j < DK / 16; ++j) o.w[j] = tile(At::w, wave * (DK / 16) + j);
#pragma unroll
    for (int j = 0; j < DK / 16; ++j) o.q[j] = tile(At::q, wave * (DK / 16) + j);
#pragma unroll
    for (int n = 0; n < NC; ++n) o.u[n] = tile(At::u, wave * (DV / 16) + blockIdx.z * NC + n);
#pragma unroll
    for (int i = 0; i < KT; ++i)
#pragma unroll
      for (int b = 0; b < 4; ++b) o.k[i][b] = tile(At::k, (wave * KT + i) * 4 + b);
#pragma unroll
    for (int b = 0; b < 4; ++b) o.p[b] = tile(At::p, wave * 4 + b);
    o.whole = base[min(c, n_chunks - 1) * apart + At::whole];
  };
  const f32x4 zero = f32x4{0.f, 0.f, 0.f, 0.f};
  const size_t width = static_cast<size_t>(gridDim.x) * DV;
  auto step = [&](const Operands& in_chunk, int c) __attribute__((always_inline)) {
    constexpr int kSums = 2;       // chains a sum (whatever NC, which depends on the whole step: a row's
                                   // bits do not)
    f32x4 ws[NC][kSums], qs[NC][kSums];
#pragma unroll
    for (int n = 0; n < NC; ++n)
#pragma unroll
      for (int u = 0; u < kSums; ++u) ws[n][u] = qs[n][u] = zero;
#pragma unroll
    for (int j0 = 0; j0 < DK / 16; j0 += 4) {
      f32x4 sb[4][NC];
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int n = 0; n < NC; ++n)
          sb[j][n] = *reinterpret_cast<const f32x4*>(s_lds + (16 * n + i16) * SS + 16 * (j0 + j) + 4 * g);
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
          for (int n = 0; n < NC; ++n) {
            ws[n][r % kSums] = __builtin_amdgcn_mfma_f32_16x16x4f32(in_chunk.w[j0 + j][r], sb[j][n][r], ws[n][r % kSums], 0, 0, 0);
            qs[n][r % kSums] = __builtin_amdgcn_mfma_f32_16x16x4f32(in_chunk.q[j0 + j][r], sb[j][n][r], qs[n][r % kSums], 0, 0, 0);
          }
    }
#pragma unroll
    for (int n = 0; n < NC; ++n) {
      const f32x4 seen = ws[n][0] + ws[n][1];
      *reinterpret_cast<f32x4*>(u_lds + (16 * n + i16) * US + 16 * wave + 4 * g) = in_chunk.u[n] - seen;
    }
    lds_barrier();                               // U is there, and S has been read
    f32x4 add[NC][KT], o[NC][kSums];
#pragma unroll
    for (int n = 0; n < NC; ++n) {
#pragma unroll
      for (int i = 0; i < KT; ++i) add[n][i] = zero;
#pragma unroll
      for (int u = 0; u < kSums; ++u) o[n][u] = zero;
    }
    f32x4 ub[4][NC];
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int n = 0; n < NC; ++n)
        ub[b][n] = *reinterpret_cast<const f32x4*>(u_lds + (16 * n + i16) * US + 16 * b + 4 * g);
#pragma unroll
    for (int b = 0; b < 4; ++b) {        // (the weights above the diagonal are zeros)
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int n = 0; n < NC; ++n) {
#pragma unroll
          for (int i = 0; i < KT; ++i)
            add[n][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(in_chunk.k[i][b][r], ub[b][n][r], add[n][i], 0, 0, 0);
          o[n][r % kSums] = __builtin_amdgcn_mfma_f32_16x16x4f32(in_chunk.p[b][r], ub[b][n][r], o[n][r % kSums], 0, 0, 0);
        }
    }
    float met = 0.f;
#pragma unroll
    for (int n = 0; n < NC; ++n) met += o[n][0][0] * 0.f + o[n][1][0] * 0.f;
    if (any_not_finite(met)) {
      const float* weights = base + c * apart + At::p;
#pragma unroll
      for (int n = 0; n < NC; ++n) {
        o[n][0] = o[n][1] = zero;
#pragma unroll 1
        for (int s = 0; s < 16 * (wave + 1); ++s) {
          const float u = u_lds[(16 * n + i16) * US + s];
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int t = 16 * wave + 4 * g + r;
            if (s <= t) o[n][0][r] += weights[operand_at(t, s, kTokens)] * u;
          }
        }
      }
    }
#pragma unroll
    for (int n = 0; n < NC; ++n)
#pragma unroll
      for (int i = 0; i < KT; ++i) {
        S[n][i] = in_chunk.whole * S[n][i] + add[n][i];
        *reinterpret_cast<f32x4*>(s_lds + (16 * n + i16) * SS + (wave * KT + i) * 16 + 4 * g) = S[n][i];
      }
    const int t0 = c * kTokens + 16 * wave + 4 * g;
    float* dst = out + (static_cast<size_t>(seqs.row0[seq]) + t0) * width + head * DV + col0 + i16;
#pragma unroll
    for (int n = 0; n < NC; ++n) {
      const f32x4 read = (o[n][0] + o[n][1]) + (qs[n][0] + qs[n][1]);
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (t0 + r < count) dst[r * width + 16 * n] = read[r];
    }
    lds_barrier();                               // S is there, and U has been read
  };
  // two sets of operands: a chunk's are asked for while the one before it is worked on, so that a
  // trip to the scratch, which lies beyond the L2, has a whole chunk's time
  Operands even, odd;
  ask(even, 0);
  lds_barrier();
  for (int c = 0; c < n_chunks; c += 2) {
    ask(odd, c + 1);
    step(even, c);
    if (c + 1 < n_chunks) {
      ask(even, c + 2);
      step(odd, c + 1);
    }
  }
#pragma unroll
  for (int n = 0; n < NC; ++n)
#pragma unroll
    for (int i = 0; i < KT; ++i)
      *reinterpret_cast<f32x4*>(to + static_cast<size_t>(n) * 16 * DK + (wave * KT + i) * 16 + 4 * g) = S[n][i];
}

inline bool sizes_fit(int dk, int dv) { return chunks::sizes_fit(dk, dv); }
inline int chunk_floats(int dk, int dv) { return kTokens * (3 * dk + kTokens + dv) + 4; }

template <int DK, int DV>
inline void launch(const Rows& in, const Gates& gates, const State& state, const Sequences& seqs,
                   float* scratch, float* out, int rows, int n_seqs, int heads, int longest,
                   hipStream_t stream) {
  static_assert(Scratch<DK, DV>::floats == kTokens * (3 * DK + kTokens + DV) + 4, "what the host allots");
  solve_kernel<DK, DV><<<dim3(heads, (longest + kTokens - 1) / kTokens, n_seqs), kSolvers, 0, stream>>>(
      in, gates, seqs, scratch);
  // 16 columns a block, the shortest chain, while that makes at most a block for every compute unit: keys
  // of 128 take the registers of one (16 heads of 128 x 128, 2 sequences of 1,024 tokens, 256 blocks: 85 us
  // against 110 by 32 columns; 3 sequences 150 against 128, 4 sequences 163 against 142), and keys of 64,
  // of which two fit, gain no more by the second (384 blocks: 88 us either way, 512: 96); 32 columns
  // read every operand half as often.  Sequences count by their share of the longest one, whose chain the
  // walk lasts as long as: those of a token are not the chunks' anyway
  const long long chains = min(n_seqs, (rows + longest - 1) / longest);
  if (heads * chains * (DV / 16) <= ei_compute_units())
    walk_kernel<DK, DV, 1><<<dim3(heads, n_seqs, DV / 16), kThreads, 0, stream>>>(state, seqs, scratch, out);
  else
    walk_kernel<DK, DV, 2><<<dim3(heads, n_seqs, DV / 32), kThreads, 0, stream>>>(state, seqs, scratch, out);
}

}  // namespace delta_chunks
}  // namespace ei
