// Linear recurrences with a decay per head and token, a prompt's tokens in chunks of 64:
//
//   S_t = a_t S_{t-1} + b_t k_t v_t^T        o_t = S_t^T q_t          S [DK, DV] a head
//
// Token by token this is a chain whose every link waits for the one before it; by chunks the chain
// is only over chunks.  With A_t the product of a chunk's decays up to token t, S_0 the state
// before the chunk and n its tokens:
//
//   S_n = A_n S_0 + sum_s (A_n / A_s) b_s k_s v_s^T
//   o_t = A_t S_0^T q_t + sum_{s <= t} (A_t / A_s) b_s (q_t . k_s) v_s
//
// so three kernels do it: `add` makes every chunk's own sum (all chunks side by side), `carry` walks
// the chunks of a sequence element by element of S and leaves the state before each of them, and
// `read` makes the outputs (again all chunks side by side).  Everything is float32 as in the walk:
// the products run on the float32 matrix instruction (v_mfma_f32_32x32x2_f32, IEEE float32
// operands and sums), ratios of decays are exponentials of differences of sums of logarithms
// held in float64, so no quotient of small numbers occurs.
//
// What bounds them: 2 DK DV + 48 (DK + DV) multiply-adds a token and head (S_0^T q and k v^T; of q k^T
// and of the weights times v three of a chunk's four tiles) are 20 us for 2,048 tokens of 16 heads of
// 128 x 128 at the instruction's 147 TFLOP/s, and the chunks' states, written once, carried and read,
// are 134 MB, 28 us at the 4.85 TB/s of a large copy.
//
// Rows of a chunk beyond its sequence's end are its last row again, with weight zero.
//
// Causality holds for values that are not finite too: the products with the weights below the
// diagonal multiply zeros above it, and zero times infinity is none, so a tile of values that holds
// such a one takes its sum term by term, without the places above the diagonal.  (Every row of a
// product meets every value of its column, so one row of the result tells.)
#pragma once
#include "common.h"

namespace ei {
namespace chunks {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kTokens = 64;
constexpr int kThreads = 256;
constexpr int kScalars = 4;        // floats behind a chunk's state: what is known of it as a whole

// kFixed: a decay a head.  kSelective: a_t = exp(-exp(a_log) dt_t), b_t = dt_t, a skip term.
// kMatrix: exponential input gates and sigmoid forget gates with a running maximum, a normaliser.
enum Kind { kFixed, kSelective, kMatrix };

// Where a head's q, k and v lie in a row of T, `share` heads having one q and k.
struct Rows {
  size_t stride;
  int q, k, v, share;
};

// The step's sequences, one behind the other in its rows.  Those of fewer than `least` rows (at
// least 1) are not the chunks' to take: what a sequence's rows go through depends on how many they
// are, not on what else the step holds.
struct Sequences {
  const int32_t *in, *out, *count, *row0;
  int least;
};

__device__ __forceinline__ int rows_of(const Sequences& seqs, int seq) {
  const int count = seqs.count[seq];
  return count >= seqs.least ? count : 0;
}

// What the gates are made of: per-head constants, and columns `at + head` and `at2 + head` of the
// rows `raw` (float32 slices or one bfloat16 piece), as the kinds need them.
struct Gates {
  const float *c0, *c1, *c2;
  const void* raw;
  int raw_bf16, nsplit;
  size_t split_stride, stride;
  int at, at2;
  float cap, q_scale, bottom_eps;
};

// A head's place in the state rows: head * head_floats on, [DK][DV] or (turned) [DV][DK].
struct State {
  float* rows;
  size_t row_floats, head_floats;
};

template <int KIND>
__host__ __device__ constexpr bool turned() { return KIND != kFixed; }

// Floats of a chunk's scratch for one head.
__host__ __device__ constexpr size_t chunk_floats(int kind, int dk, int dv) {
  return static_cast<size_t>(dk) * dv + (kind == kMatrix ? dk : 0) + kScalars;
}

// The scratch of chunk c of sequence s: ceil(count / 64) <= floor((row0 + count) / 64) -
// floor(row0 / 64) + 1, and from one sequence that is taken to the next both row0 / least and s grow
// by one or more, so no two sequences' parts meet, and chunk_places hold all of them.
__device__ __forceinline__ size_t chunk_place(const Sequences& seqs, int seq, int chunk) {
  const int row0 = seqs.row0[seq];
  return static_cast<size_t>(row0 / kTokens) + min(row0 / seqs.least, seq) + chunk;
}

inline long long chunk_places(int rows, int n_seqs, int least) {
  return rows / kTokens + (rows / least < n_seqs ? rows / least : n_seqs);
}

__device__ __forceinline__ float gate_column(const Gates& g, size_t row, int column) {
  float v = 0.f;
  for (int s = 0; s < g.nsplit; ++s) {
    const size_t i = s * g.split_stride + row * g.stride + column;
    v += g.raw_bf16 ? bf16_to_f32(static_cast<const bf16_t*>(g.raw)[i]) : static_cast<const float*>(g.raw)[i];
  }
  return v;
}

// The logarithm of a decay, so low a one that one step of it leaves nothing of a float32 (the least
// is e^-103.98) as e^-128: a sum of logarithms then stays below 2^13, where float64 has 13 digits
// behind the point, however low they are and even if they are minus infinity (the difference of two of
// those would be no number).
__device__ __forceinline__ double bounded_log(double each) { return each < -128.0 ? -128.0 : each; }

// A chunk's gates, lane t having token t: `log_sum` the sum of the log decays up to t (float64),
// `take` the input weight b_t (kMatrix: its logarithm).  Tokens beyond the chunk's end do not
// decay and bring nothing.
template <int KIND>
__device__ __forceinline__ void lane_gates(const Gates& g, int head, size_t row, int t, int nt,
                                           double& log_sum, float& take) {
  if constexpr (KIND == kFixed) {
    const float d = g.c0[head];
    const double each = bounded_log(log(static_cast<double>(d)));
    log_sum = each * (min(t, nt - 1) + 1);
    take = t < nt ? 1.f : 0.f;
  } else {
    double each = 0.0;
    if constexpr (KIND == kSelective) {
      take = 0.f;
      if (t < nt) {
        const float z = gate_column(g, row, g.at + head) + g.c1[head];
        const float dt = z > 20.f ? z : log1pf(expf(z));
        each = bounded_log(-static_cast<double>(expf(g.c0[head])) * dt);
        take = dt;
      }
    } else {
      take = -INFINITY;
      if (t < nt) {
        const float xi = gate_column(g, row, g.at + head) + g.c0[head];
        const float xf = gate_column(g, row, g.at2 + head) + g.c1[head];
        take = g.cap * tanhf(xi / g.cap);
        const float z = g.cap * tanhf(xf / g.cap);
        each = fminf(z, 0.f) - log1pf(expf(-fabsf(z)));
      }
    }
#pragma unroll
    for (int step = 1; step < kTokens; step *= 2) {
      const double other = __shfl_up(each, step, EI_WAVE);
      if (t >= step) each += other;
    }
    log_sum = each;
  }
}

// Whether some lane of the wave has a value that is not finite.
__device__ __forceinline__ bool any_not_finite(float value) { return __any(value * 0.f != 0.f); }

__device__ __forceinline__ float at(const float* p) { return *p; }
__device__ __forceinline__ float at(const bf16_t* p) { return bf16_to_f32(*p); }

// A block a (chunk, head, sequence): the chunk's own sum W_n = sum_s w_s k_s v_s^T and what is known
// of the chunk as a whole.  Both operands of k^T v lie as the matrix instruction wants them (32
// neighbouring elements of a row), so they go from global memory into its registers.
template <int KIND, typename T, int DK, int DV>
__global__ void __launch_bounds__(kThreads)
add_kernel(const T* __restrict__ rows, Rows at_row, Gates gates, Sequences seqs,
           float* __restrict__ scratch) {
  constexpr int KT = DK / 32, VT = DV / 32;              // tiles of 32 x 32 of S
  constexpr int WV = VT >= 4 ? 2 : 1;                    // waves side by side along the columns
  constexpr int MK = KT / (4 / WV) > 0 ? KT / (4 / WV) : 1, MV = VT / WV;   // tiles a wave
  __shared__ float weight[kTokens];
  const int chunk = blockIdx.x, head = blockIdx.y, seq = blockIdx.z;
  const int nt = min(kTokens, rows_of(seqs, seq) - chunk * kTokens);
  if (nt <= 0) return;
  const int first = seqs.row0[seq] + chunk * kTokens;
  float* mine = scratch + (chunk_place(seqs, seq, chunk) * gridDim.y + head) *
                              chunk_floats(KIND, DK, DV);
  float* scalars = mine + chunk_floats(KIND, DK, DV) - kScalars;
  const int lane = threadIdx.x % EI_WAVE, wave = threadIdx.x / EI_WAVE;
  if (wave == 0) {
    double log_sum;
    float take;
    lane_gates<KIND>(gates, head, static_cast<size_t>(first) + min(lane, nt - 1), lane, nt, log_sum, take);
    const double whole = __shfl(log_sum, EI_WAVE - 1, EI_WAVE);
    if constexpr (KIND == kMatrix) {
      const float log_w = static_cast<float>(whole - log_sum) + take;
      const float most = wave_max(log_w);
      weight[lane] = lane < nt ? expf(log_w - most) : 0.f;
      if (lane == 0) {
        scalars[0] = static_cast<float>(whole);
        scalars[1] = most;
      }
    } else {
      weight[lane] = expf(static_cast<float>(whole - log_sum)) * take;
      if (lane == 0) scalars[0] = expf(static_cast<float>(whole));
    }
  }
  __syncthreads();
  const int half = lane / 32, l = lane % 32;
  const T* k_at = rows + at_row.k + (head / at_row.share) * DK;
  const T* v_at = rows + at_row.v + head * DV;
  const int kt0 = wave / WV * MK, vt0 = wave % WV * MV;
  if (kt0 < KT) {
    f32x16 acc[MK][MV];
#pragma unroll
    for (int i = 0; i < MK; ++i)
#pragma unroll
      for (int j = 0; j < MV; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
    constexpr int kGroup = 8;                            // products (two tokens each) asked for at once
    float a[kGroup][MK], b[kGroup][MV];
    auto ask = [&](int t0) {
#pragma unroll
      for (int u = 0; u < kGroup; ++u) {
        const size_t row = static_cast<size_t>(first + min(t0 + 2 * u + half, nt - 1)) * at_row.stride;
#pragma unroll
        for (int i = 0; i < MK; ++i) a[u][i] = at(k_at + row + (kt0 + i) * 32 + l);
#pragma unroll
        for (int j = 0; j < MV; ++j) b[u][j] = at(v_at + row + (vt0 + j) * 32 + l);
      }
    };
    for (int t0 = 0; t0 < nt; t0 += 2 * kGroup) {
      ask(t0);
#pragma unroll
      for (int u = 0; u < kGroup; ++u) {
        const float w = weight[t0 + 2 * u + half];
#pragma unroll
        for (int i = 0; i < MK; ++i)
#pragma unroll
          for (int j = 0; j < MV; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[u][i] * w, b[u][j], acc[i][j], 0, 0, 0);
      }
    }
#pragma unroll
    for (int i = 0; i < MK; ++i)
#pragma unroll
      for (int j = 0; j < MV; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int k = (kt0 + i) * 32 + e % 4 + 8 * (e / 4) + 4 * half;
          mine[k * DV + (vt0 + j) * 32 + l] = acc[i][j][e];
        }
  }
  if constexpr (KIND == kMatrix) {                       // the normaliser's part: sum_s w_s k_s
    for (int k = threadIdx.x; k < DK; k += kThreads) {
      float sum = 0.f;
      for (int t = 0; t < nt; ++t)
        sum += weight[t] * at(k_at + static_cast<size_t>(first + t) * at_row.stride + k);
      mine[DK * DV + k] = sum;
    }
  }
}

// A thread four neighbouring elements of a head's S (kMatrix: the last block the normaliser): the
// chunks of a sequence in order, each chunk's own sum replaced by the state before it, the state
// after the last one to the table.
template <int KIND, int DK, int DV>
__global__ void __launch_bounds__(kThreads)
carry_kernel(State state, Sequences seqs, float* __restrict__ scratch) {
  constexpr int kBatch = 8;                              // chunks whose sums are asked for at once
  const int head = blockIdx.y, seq = blockIdx.z;
  const int count = rows_of(seqs, seq);
  if (count <= 0) return;
  const int chunks = (count + kTokens - 1) / kTokens;
  constexpr size_t kFloats = chunk_floats(KIND, DK, DV);
  const size_t apart = gridDim.y * kFloats;              // from one chunk to the next
  float* base = scratch + (chunk_place(seqs, seq, 0) * gridDim.y + head) * kFloats;
  const float* in = state.rows + static_cast<size_t>(seqs.in[seq]) * state.row_floats + head * state.head_floats;
  float* out = state.rows + static_cast<size_t>(seqs.out[seq]) * state.row_floats + head * state.head_floats;
  const int e0 = 4 * (blockIdx.x * kThreads + threadIdx.x);
  constexpr int kElements = DK * DV + (KIND == kMatrix ? DK : 0);
  if (e0 >= kElements) return;
  // where the four elements lie in the table
  size_t place[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int e = e0 + i;
    place[i] = (turned<KIND>() && e < DK * DV) ? static_cast<size_t>(e % DV) * DK + e / DV : e;
  }
  f32x4 S;
#pragma unroll
  for (int i = 0; i < 4; ++i) S[i] = in[place[i]];
  float m = KIND == kMatrix ? in[static_cast<size_t>(DV) * DK + DK] : 0.f;
  for (int c0 = 0; c0 < chunks; c0 += kBatch) {
    f32x4 own[kBatch];
    float whole[kBatch], most[kBatch];
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      const float* at_chunk = base + min(c0 + u, chunks - 1) * apart;
      own[u] = *reinterpret_cast<const f32x4*>(at_chunk + e0);
      whole[u] = at_chunk[kFloats - kScalars];
      if constexpr (KIND == kMatrix) most[u] = at_chunk[kFloats - kScalars + 1];
    }
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      if (c0 + u < chunks) {
        float* at_chunk = base + (c0 + u) * apart;
        *reinterpret_cast<f32x4*>(at_chunk + e0) = S;
        if constexpr (KIND == kMatrix) {
          if (e0 == 0) at_chunk[kFloats - kScalars + 2] = m;
          const float next = fmaxf(whole[u] + m, most[u]);
          const float keep = expf(whole[u] + m - next), take = expf(most[u] - next);
#pragma unroll
          for (int i = 0; i < 4; ++i) S[i] = keep * S[i] + take * own[u][i];
          m = next;
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i) S[i] = whole[u] * S[i] + own[u][i];
        }
      }
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) out[place[i]] = S[i];
  if (KIND == kMatrix && e0 == 0) out[static_cast<size_t>(DV) * DK + DK] = m;
}

// A wave a tile of 32 x 32 outputs.
constexpr int read_threads(int dv) { return EI_WAVE * 2 * (dv / 32); }

// A block a (chunk, head, sequence): the outputs.  q and k lie in LDS for q k^T (one of the three
// tiles of 32 x 32 below the diagonal a wave), whose masked and weighted values take k's place as
// an operand; S_0 and v come from global memory, 32 neighbouring columns a load.  A product of
// four steps takes the k values 8 j + 4 half + s, so a lane's four are one 16-byte read of LDS.
template <int KIND, typename T, int DK, int DV>
__global__ void __launch_bounds__(read_threads(DV))
read_kernel(const T* __restrict__ rows, Rows at_row, Gates gates, Sequences seqs,
            const float* __restrict__ scratch, float* __restrict__ out) {
  constexpr int VT = DV / 32;                            // column tiles
  constexpr int kReaders = read_threads(DV);
  constexpr int QS = DK + 4, PS = kTokens + 4;           // LDS rows: 16-byte reads of 16 lanes, no bank twice
  __shared__ __attribute__((aligned(16))) float q_lds[kTokens * QS];
  __shared__ __attribute__((aligned(16))) float k_lds[kTokens * (QS > PS ? QS : PS)];
  __shared__ double log_sums[kTokens];
  __shared__ float takes[kTokens], from_state[kTokens], over[kTokens], rowmax[kTokens];
  const int chunk = blockIdx.x, head = blockIdx.y, seq = blockIdx.z;
  const int nt = min(kTokens, rows_of(seqs, seq) - chunk * kTokens);
  if (nt <= 0) return;
  const int first = seqs.row0[seq] + chunk * kTokens;
  const float* mine = scratch + (chunk_place(seqs, seq, chunk) * gridDim.y + head) *
                                    chunk_floats(KIND, DK, DV);
  const int lane = threadIdx.x % EI_WAVE, wave = threadIdx.x / EI_WAVE;
  const int half = lane / 32, l = lane % 32;
  {
    const T* q_at = rows + at_row.q + (head / at_row.share) * DK;
    const T* k_at = rows + at_row.k + (head / at_row.share) * DK;
    constexpr int kPieces = DK / 4, kLoads = kTokens * kPieces / kReaders;
    float q4[kLoads][4], k4[kLoads][4];
#pragma unroll
    for (int u = 0; u < kLoads; ++u) {
      const int i = threadIdx.x + u * kReaders;
      const size_t at_piece = static_cast<size_t>(first + min(i / kPieces, nt - 1)) * at_row.stride + i % kPieces * 4;
      Vec4<T>::load(q_at + at_piece, q4[u]);
      Vec4<T>::load(k_at + at_piece, k4[u]);
    }
#pragma unroll
    for (int u = 0; u < kLoads; ++u) {
      const int i = threadIdx.x + u * kReaders;
      if constexpr (KIND == kMatrix) {
#pragma unroll
        for (int e = 0; e < 4; ++e) q4[u][e] *= gates.q_scale;
      }
      Vec4<float>::store(q_lds + i / kPieces * QS + i % kPieces * 4, q4[u]);
      Vec4<float>::store(k_lds + i / kPieces * QS + i % kPieces * 4, k4[u]);
    }
  }
  if (wave == 3) {       // (a wave without a tile of q k^T)
    double log_sum;
    float take;
    lane_gates<KIND>(gates, head, static_cast<size_t>(first) + min(lane, nt - 1), lane, nt, log_sum, take);
    if constexpr (KIND == kMatrix) {
      // relative to the running maximum: m_t = F_t + M_t, M_t = max(m before the chunk, i_s - F_s)
      const double u = static_cast<double>(take) - log_sum;
      float top = lane < nt ? static_cast<float>(u) : -INFINITY;
#pragma unroll
      for (int step = 1; step < kTokens; step *= 2) {
        const float other = __shfl_up(top, step, EI_WAVE);
        if (lane >= step) top = fmaxf(top, other);
      }
      const float before = mine[chunk_floats(KIND, DK, DV) - kScalars + 2];
      top = fmaxf(top, before);
      log_sums[lane] = u;
      rowmax[lane] = top;
      from_state[lane] = expf(before - top);
      takes[lane] = expf(-static_cast<float>(log_sum + top));      // e^(-m_t), the denominator's least
    } else {
      log_sums[lane] = log_sum;
      takes[lane] = take;
      from_state[lane] = expf(static_cast<float>(log_sum));
    }
  }
  __syncthreads();
  const int qt = wave == 0 ? 0 : 1, kt = wave == 2 ? 1 : 0;        // the wave's tile of q k^T
  const bool has_tile = wave < 3 && (qt == 0 || nt > 32);
  // (every sum of products is cut into kSums chains, added at the end: one chain of 128 loses
  // twice the precision that the walk's shorter sums do)
  constexpr int kSums = 4;
  f32x16 scores[kSums];
#pragma unroll
  for (int u = 0; u < kSums; ++u)
#pragma unroll
    for (int e = 0; e < 16; ++e) scores[u][e] = 0.f;
  if (has_tile) {
    const float* qr = q_lds + (qt * 32 + l) * QS + 4 * half;
    const float* kr = k_lds + (kt * 32 + l) * QS + 4 * half;
#pragma unroll 4
    for (int j = 0; j < DK / 8; ++j) {
      const f32x4 a = *reinterpret_cast<const f32x4*>(qr + 8 * j);
      const f32x4 b = *reinterpret_cast<const f32x4*>(kr + 8 * j);
#pragma unroll
      for (int s = 0; s < 4; ++s)
        scores[s] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[s], b[s], scores[s], 0, 0, 0);
    }
  }
  const f32x16 score = (scores[0] + scores[1]) + (scores[2] + scores[3]);
  __syncthreads();                                       // k has been read: the weights take its place
  float* p_lds = k_lds;
  if (has_tile) {
    const int s = kt * 32 + l;
    const double ls = log_sums[s];
    const float take = takes[s];
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int t = qt * 32 + e % 4 + 8 * (e / 4) + 4 * half;
      float p = 0.f;
      if (s <= t && s < nt) {
        if constexpr (KIND == kMatrix) p = score[e] * expf(static_cast<float>(ls - static_cast<double>(rowmax[t])));
        else p = score[e] * (expf(static_cast<float>(log_sums[t] - ls)) * take);
      }
      p_lds[t * PS + s] = p;
    }
  }
  __syncthreads();
  if constexpr (KIND == kMatrix) {
    // the denominators: n_t . q_t = e^(m' - M_t) (n_0 . q_t) + the row's sum of weights
    const int t = threadIdx.x / 4 % kTokens, part = threadIdx.x % 4;     // (256 threads, or twice the same)
    float with_n = 0.f, sum = 0.f;
    for (int k = part * 4; k < DK; k += 16) {
      const f32x4 n4 = *reinterpret_cast<const f32x4*>(mine + DK * DV + k);
      const f32x4 q4 = *reinterpret_cast<const f32x4*>(q_lds + t * QS + k);
#pragma unroll
      for (int e = 0; e < 4; ++e) with_n += n4[e] * q4[e];
    }
    const int seen = t < 32 ? 32 : kTokens;              // (columns that were written)
    if (t < nt)
      for (int s = part; s < seen; s += 4) sum += p_lds[t * PS + s];
    float nq = from_state[t] * with_n + sum;
    nq += __shfl_xor(nq, 1, 4);
    nq += __shfl_xor(nq, 2, 4);
    if (part == 0) over[t] = 1.0f / (fmaxf(fabsf(nq), takes[t]) + gates.bottom_eps);
    __syncthreads();
  }
  const int ct = wave % VT, rt = wave / VT;
  if (rt * 32 < nt) {
    f32x16 sums[kSums];
    auto clear = [&]() {
#pragma unroll
      for (int u = 0; u < kSums; ++u)
#pragma unroll
        for (int e = 0; e < 16; ++e) sums[u][e] = 0.f;
    };
    clear();
    const float* s_at = mine + 4 * half * DV + ct * 32 + l;
    constexpr int kGroup = 4;
#pragma unroll 1
    for (int j0 = 0; j0 < DK / 8; j0 += kGroup) {
      float b[kGroup][4];
#pragma unroll
      for (int u = 0; u < kGroup; ++u)
#pragma unroll
        for (int s = 0; s < 4; ++s) b[u][s] = s_at[static_cast<size_t>(8 * (j0 + u) + s) * DV];
#pragma unroll
      for (int u = 0; u < kGroup; ++u) {
        const f32x4 a = *reinterpret_cast<const f32x4*>(q_lds + (rt * 32 + l) * QS + 8 * (j0 + u) + 4 * half);
#pragma unroll
        for (int s = 0; s < 4; ++s)
          sums[s] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[s], b[u][s], sums[s], 0, 0, 0);
      }
    }
    f32x16 acc = (sums[0] + sums[1]) + (sums[2] + sums[3]);
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[e] *= from_state[rt * 32 + e % 4 + 8 * (e / 4) + 4 * half];
    clear();
    const T* v_at = rows + at_row.v + head * DV + ct * 32 + l;
#pragma unroll
    for (int j0 = 0; j0 < kTokens / 8; j0 += kGroup) {   // tokens 0 .. 31, then 32 .. 63
      if (8 * j0 < nt && 8 * j0 < 32 * (rt + 1)) {           // (above the diagonal: nothing)
        float b[kGroup][4];
#pragma unroll
        for (int u = 0; u < kGroup; ++u)
#pragma unroll
          for (int s = 0; s < 4; ++s)
            b[u][s] = at(v_at + static_cast<size_t>(first + min(8 * (j0 + u) + 4 * half + s, nt - 1)) * at_row.stride);
#pragma unroll
        for (int u = 0; u < kGroup; ++u) {
          const f32x4 a = *reinterpret_cast<const f32x4*>(p_lds + (rt * 32 + l) * PS + 8 * (j0 + u) + 4 * half);
#pragma unroll
          for (int s = 0; s < 4; ++s)
            sums[s] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[s], b[u][s], sums[s], 0, 0, 0);
        }
      }
    }
    f32x16 own = (sums[0] + sums[1]) + (sums[2] + sums[3]);
    if (any_not_finite(own[0])) {
#pragma unroll
      for (int e = 0; e < 16; ++e) own[e] = 0.f;
#pragma unroll 1
      for (int s = 0; s < min(nt, 32 * (rt + 1)); ++s) {
        const float v = at(v_at + static_cast<size_t>(first + s) * at_row.stride);
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int t = rt * 32 + e % 4 + 8 * (e / 4) + 4 * half;
          if (s <= t) own[e] += p_lds[t * PS + s] * v;
        }
      }
    }
    acc += own;
    const size_t width = static_cast<size_t>(gridDim.y) * DV;
    const float skip = KIND == kSelective ? gates.c2[head] : 0.f;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int t = rt * 32 + e % 4 + 8 * (e / 4) + 4 * half;
      if (t < nt) {
        float o = acc[e];
        if constexpr (KIND == kSelective) o += skip * at(v_at + static_cast<size_t>(first + t) * at_row.stride);
        if constexpr (KIND == kMatrix) o *= over[t];
        out[static_cast<size_t>(first + t) * width + head * DV + ct * 32 + l] = o;
      }
    }
  }
}

// The sizes that the kernels take: heads of 64 or 128 key and value elements.
inline bool sizes_fit(int dk, int dv) { return (dk == 64 || dk == 128) && (dv == 64 || dv == 128); }

template <int KIND, typename T, int DK, int DV>
inline void launch(const T* rows, const Rows& at_row, const Gates& gates, const State& state,
                   const Sequences& seqs, float* scratch, float* out, int n_seqs, int heads,
                   int longest, hipStream_t stream) {
  const dim3 grid((longest + kTokens - 1) / kTokens, heads, n_seqs);
  add_kernel<KIND, T, DK, DV><<<grid, kThreads, 0, stream>>>(rows, at_row, gates, seqs, scratch);
  constexpr int kElements = DK * DV + (KIND == kMatrix ? DK : 0);
  const dim3 elements((kElements / 4 + kThreads - 1) / kThreads, heads, n_seqs);
  carry_kernel<KIND, DK, DV><<<elements, kThreads, 0, stream>>>(state, seqs, scratch);
  read_kernel<KIND, T, DK, DV><<<grid, read_threads(DV), 0, stream>>>(rows, at_row, gates, seqs, scratch, out);
}

template <int KIND, typename T>
inline void launch_sized(int dk, int dv, const T* rows, const Rows& at_row, const Gates& gates,
                         const State& state, const Sequences& seqs, float* scratch, float* out,
                         int n_seqs, int heads, int longest, hipStream_t stream) {
  if (dk == 128 && dv == 128) launch<KIND, T, 128, 128>(rows, at_row, gates, state, seqs, scratch, out, n_seqs, heads, longest, stream);
  else if (dk == 128) launch<KIND, T, 128, 64>(rows, at_row, gates, state, seqs, scratch, out, n_seqs, heads, longest, stream);
  else if (dv == 128) launch<KIND, T, 64, 128>(rows, at_row, gates, state, seqs, scratch, out, n_seqs, heads, longest, stream);
  else launch<KIND, T, 64, 64>(rows, at_row, gates, state, seqs, scratch, out, n_seqs, heads, longest, stream);
}

}  // namespace chunks
}  // namespace ei
