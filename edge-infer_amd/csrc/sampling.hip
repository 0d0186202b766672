// Sampling from float32 logits, one block per row of the batch.
//
// Greedy: argmax, ties to the lowest index.  Stochastic, in the reference's order
// (operators/src/cuda/execution.cu:193-234, 455-498): z = logit / temperature
// (NaN -> -inf); the k = min(top_k, V) largest, sorted descending with ties to the
// lower index; e_i = exp(z_i - z_0); the shortest prefix whose mass reaches
// top_p * total, at least one element and including the one that crosses; a uniform
// u in (0, 1]; the first kept element whose cumulative mass reaches u * retained.
// Instead of sorting the whole vocabulary the k-th largest value is found by a radix
// select and only the k candidates are sorted.  The uniform number comes from a
// counter-based generator keyed by (seed, request stream, step counter), so a
// request draws the same numbers alone or in any batch.
#include "common.h"
#include "sampling_static.h"

#include <atomic>

namespace {

constexpr int kThreads = 1024;
constexpr int kMaxTopK = 1024;

__device__ __forceinline__ uint32_t sortable_key(float z) {
  const uint32_t u = __float_as_uint(z);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);  // ascending in z
}

__device__ __forceinline__ float key_value(uint32_t key) {
  const uint32_t u = (key & 0x80000000u) ? (key & 0x7fffffffu) : ~key;
  return __uint_as_float(u);
}

__device__ __forceinline__ float scaled_logit(float logit, float temperature, bool scale) {
  if (isnan(logit)) return -INFINITY;
  return scale ? logit / temperature : logit;
}

// splitmix64 finalizer of seed + golden * (stream * 2^32 + counter + 1); (0, 1].
__device__ __forceinline__ float uniform_draw(uint64_t seed, uint32_t stream, uint32_t counter) {
  uint64_t z = seed + 0x9E3779B97F4A7C15ull *
                          ((static_cast<uint64_t>(stream) << 32) + counter + 1ull);
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  z ^= z >> 31;
  return (static_cast<float>(z >> 40) + 1.0f) * (1.0f / 16777216.0f);
}

__global__ void __launch_bounds__(kThreads)
argmax_kernel(const float* __restrict__ logits, int V, int32_t* __restrict__ tokens,
              float* __restrict__ probabilities) {
  __shared__ float best_value[kThreads / EI_WAVE];
  __shared__ int best_index[kThreads / EI_WAVE];
  const float* row = logits + static_cast<size_t>(blockIdx.x) * V;
  float value = -INFINITY;
  int index = 0x7fffffff;
  for (int i = threadIdx.x; i < V; i += kThreads) {
    const float z = scaled_logit(row[i], 1.f, false);
    if (z > value || (z == value && i < index)) {
      value = z;
      index = i;
    }
  }
#pragma unroll
  for (int offset = EI_WAVE / 2; offset > 0; offset >>= 1) {
    const float other_value = __shfl_xor(value, offset, EI_WAVE);
    const int other_index = __shfl_xor(index, offset, EI_WAVE);
    if (other_value > value || (other_value == value && other_index < index)) {
      value = other_value;
      index = other_index;
    }
  }
  const int wave = threadIdx.x / EI_WAVE, lane = threadIdx.x % EI_WAVE;
  if (lane == 0) {
    best_value[wave] = value;
    best_index[wave] = index;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < kThreads / EI_WAVE; ++w) {
      if (best_value[w] > value || (best_value[w] == value && best_index[w] < index)) {
        value = best_value[w];
        index = best_index[w];
      }
    }
    tokens[blockIdx.x] = index == 0x7fffffff ? 0 : index;
    if (probabilities) probabilities[blockIdx.x] = 1.f;
  }
}

// Wide vocabularies, two steps: every block finds the best of one chunk of a row, then one
// wave a row picks the best chunk.  The same order (larger value, then lower index) as above.
constexpr int kArgmaxThreads = 256;
constexpr int kArgmaxChunk = 4096;

__device__ __forceinline__ void keep_better(float& value, int& index, float other_value,
                                            int other_index) {
  if (other_value > value || (other_value == value && other_index < index)) {
    value = other_value;
    index = other_index;
  }
}

__global__ void __launch_bounds__(kArgmaxThreads)
argmax_chunks_kernel(const float* __restrict__ logits, int V, float2* __restrict__ partial) {
  __shared__ float best_value[kArgmaxThreads / EI_WAVE];
  __shared__ int best_index[kArgmaxThreads / EI_WAVE];
  const float* row = logits + static_cast<size_t>(blockIdx.y) * V;
  const int begin = blockIdx.x * kArgmaxChunk;
  const int end = min(V, begin + kArgmaxChunk);
  float value = -INFINITY;
  int index = 0x7fffffff;
  constexpr int kPerThread = kArgmaxChunk / kArgmaxThreads;
  float z[kPerThread];
#pragma unroll
  for (int j = 0; j < kPerThread; ++j) {          // all loads first
    const int i = begin + threadIdx.x + j * kArgmaxThreads;
    z[j] = i < end ? row[i] : -INFINITY;
  }
#pragma unroll
  for (int j = 0; j < kPerThread; ++j) {
    const int i = begin + threadIdx.x + j * kArgmaxThreads;
    if (i < end) keep_better(value, index, scaled_logit(z[j], 1.f, false), i);
  }
#pragma unroll
  for (int offset = EI_WAVE / 2; offset > 0; offset >>= 1)
    keep_better(value, index, __shfl_xor(value, offset, EI_WAVE), __shfl_xor(index, offset, EI_WAVE));
  const int wave = threadIdx.x / EI_WAVE, lane = threadIdx.x % EI_WAVE;
  if (lane == 0) {
    best_value[wave] = value;
    best_index[wave] = index;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < kArgmaxThreads / EI_WAVE; ++w)
      keep_better(value, index, best_value[w], best_index[w]);
    partial[static_cast<size_t>(blockIdx.y) * gridDim.x + blockIdx.x] =
        make_float2(value, __int_as_float(index));
  }
}

__global__ void __launch_bounds__(EI_WAVE)
argmax_merge_kernel(const float2* __restrict__ partial, int chunks, int32_t* __restrict__ tokens,
                    float* __restrict__ probabilities) {
  const float2* mine = partial + static_cast<size_t>(blockIdx.x) * chunks;
  float value = -INFINITY;
  int index = 0x7fffffff;
  for (int c = threadIdx.x; c < chunks; c += EI_WAVE)
    keep_better(value, index, mine[c].x, __float_as_int(mine[c].y));
#pragma unroll
  for (int offset = EI_WAVE / 2; offset > 0; offset >>= 1)
    keep_better(value, index, __shfl_xor(value, offset, EI_WAVE), __shfl_xor(index, offset, EI_WAVE));
  if (threadIdx.x == 0) {
    tokens[blockIdx.x] = index == 0x7fffffff ? 0 : index;
    if (probabilities) probabilities[blockIdx.x] = 1.f;
  }
}

// For the first 256 threads of a block, each holding the count of its bin (thread t: bin t):
// the counts of all higher bins added up (an exclusive suffix sum).  `wave_totals`: four
// words of shared memory; every thread of the block calls this (it synchronizes).
__device__ __forceinline__ unsigned count_above(unsigned own, unsigned* wave_totals) {
  const int t = threadIdx.x, lane = t % EI_WAVE, wave = t / EI_WAVE;
  unsigned inclusive = own;
#pragma unroll
  for (int offset = 1; offset < EI_WAVE; offset <<= 1) {
    const unsigned other = __shfl_down(inclusive, offset, EI_WAVE);
    if (lane + offset < EI_WAVE) inclusive += other;
  }
  if (lane == 0 && wave < 256 / EI_WAVE) wave_totals[wave] = inclusive;
  __syncthreads();
  unsigned above = inclusive - own;
  for (int w = wave + 1; w < 256 / EI_WAVE; ++w) above += wave_totals[w];
  return above;
}

constexpr int kBins = 4096, kBinShift = 20;

struct SampleShared {
  __attribute__((aligned(16))) unsigned histogram[kBins];
  __attribute__((aligned(16))) unsigned long long candidates[kMaxTopK];  // (key << 32) | ~index
  int equal_index[kMaxTopK];
  unsigned select_prefix, select_remaining, n_taken, n_equal_taken, n_equal_seen;
  unsigned wave_totals[kThreads / EI_WAVE];
};

// Sorts the first k candidates, descending; the caller's barrier came before.
__device__ void sort_candidates(SampleShared& sh, int k) {
  unsigned long long (&candidates)[kMaxTopK] = sh.candidates;
  const int t = threadIdx.x;
  // pad to a power of two and sort descending (bitonic)
  int padded = 1;
  while (padded < k) padded <<= 1;
  for (int i = k + t; i < padded; i += kThreads) candidates[i] = 0ull;
  __syncthreads();
  for (int size = 2; size <= padded; size <<= 1) {
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      for (int i = t; i < padded; i += kThreads) {
        const int partner = i ^ stride;
        if (partner > i) {
          const bool descending = (i & size) == 0;
          const unsigned long long a = candidates[i], b = candidates[partner];
          if ((a < b) == descending) {
            candidates[i] = b;
            candidates[partner] = a;
          }
        }
      }
      __syncthreads();
    }
  }
}

// The draw among the k candidates of a row, sorted.  Masses in parallel, their running sums by one
// wave in index order (the order of the sums is part of the result: the draw compares against
// them): 64 masses at a time lie in the lanes and are added lane by lane, so a sum costs an
// addition and no read of LDS that depends on the one before (for 20 candidates the three walks
// by one thread were a fifth of the kernel).
__device__ void draw_row(SampleShared& sh, int k, float top_p, uint64_t seed, uint32_t stream,
                         uint32_t counter, int32_t* token, float* probability) {
  const int t = threadIdx.x;
  const unsigned long long* candidates = sh.candidates;
  const float z0 = key_value(static_cast<uint32_t>(candidates[0] >> 32));
  float* sums = reinterpret_cast<float*>(sh.equal_index);   // the tie table is done with
  __syncthreads();
  if (t >= EI_WAVE) return;
  if (!isfinite(z0)) {
    if (t == 0) {
      *token = static_cast<int>(~static_cast<uint32_t>(candidates[0] & 0xffffffffull));
      if (probability) *probability = 1.f;
    }
    return;
  }
  float total = 0.f;
  for (int begin = 0; begin < k; begin += EI_WAVE) {
    const int i = begin + t;
    const float mass = i < k ? expf(key_value(static_cast<uint32_t>(candidates[i] >> 32)) - z0) : 0.f;
    float mine = 0.f;
    const int here = min(EI_WAVE, k - begin);
    for (int l = 0; l < here; ++l) {
      total += __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, mass), l));
      if (l == t) mine = total;
    }
    if (i < k) sums[i] = mine;              // read below by the lane that wrote it, or after them all
  }
  __builtin_amdgcn_wave_barrier();
  // the first element whose sum reaches a value; `none` if no element of the first n does
  auto first_reaching = [&](float value, int n, int none) {
    for (int begin = 0; begin < n; begin += EI_WAVE) {
      const int i = begin + t;
      const unsigned long long reached = __ballot(i < n && !(sums[min(i, n - 1)] < value));
      if (reached) return begin + static_cast<int>(__builtin_ctzll(reached));
    }
    return none;
  };
  const int kept = first_reaching(top_p * total, k, k - 1) + 1;
  const float retained = sums[kept - 1];
  const int selected = first_reaching(uniform_draw(seed, stream, counter) * retained, kept, kept - 1);
  if (t == 0) {
    *token = static_cast<int>(~static_cast<uint32_t>(candidates[selected] & 0xffffffffull));
    if (probability)
      *probability = expf(key_value(static_cast<uint32_t>(candidates[selected] >> 32)) - z0) / retained;
  }
}

// One block samples one row of V >= k logits.
__device__ void sample_row(const float* __restrict__ row, int V, float temperature, int k,
                           float top_p, uint64_t seed, uint32_t stream, uint32_t counter,
                           int32_t* token, float* probability, SampleShared& sh) {
  unsigned (&histogram)[kBins] = sh.histogram;
  unsigned long long (&candidates)[kMaxTopK] = sh.candidates;
  int (&equal_index)[kMaxTopK] = sh.equal_index;
  unsigned& select_prefix = sh.select_prefix;
  unsigned& select_remaining = sh.select_remaining;
  unsigned& n_taken = sh.n_taken;
  unsigned& n_equal_taken = sh.n_equal_taken;
  unsigned& n_equal_seen = sh.n_equal_seen;
  const int t = threadIdx.x;
  auto key_of = [&](int i) { return sortable_key(scaled_logit(row[i], temperature, true)); };

  // radix select of the k-th largest key, eight bits at a time from the top
  if (t == 0) {
    select_prefix = 0u;
    select_remaining = static_cast<unsigned>(k);
  }
  unsigned mask = 0u;
  for (int shift = 24; shift >= 0; shift -= 8) {
    if (t < 256) histogram[t] = 0u;
    __syncthreads();
    const unsigned prefix = select_prefix;
    for (int i = t; i < V; i += kThreads) {
      const uint32_t key = key_of(i);
      if ((key & mask) == prefix) atomicAdd(&histogram[(key >> shift) & 0xffu], 1u);
    }
    __syncthreads();
    {
      // the highest bin that, together with the bins above it, holds the keys still wanted
      const unsigned remaining = select_remaining;
      const unsigned own = t < 256 ? histogram[t] : 0u;
      const unsigned above = count_above(own, sh.wave_totals);
      __syncthreads();                      // everybody has read select_remaining
      if (t < 256 && above < remaining && above + own >= remaining) {
        select_remaining = remaining - above;
        select_prefix = prefix | (static_cast<unsigned>(t) << shift);
      }
    }
    mask |= 0xffu << shift;
    __syncthreads();
  }
  const uint32_t kth = select_prefix;
  const unsigned need_equal = select_remaining;  // how many keys equal to kth belong to the top k
  if (t == 0) {
    n_taken = 0u;
    n_equal_taken = 0u;
    n_equal_seen = 0u;
  }
  __syncthreads();
  // keys above the k-th: all of them, in any order (the sort below orders them);
  // keys equal to it are listed aside
  for (int i = t; i < V; i += kThreads) {
    const uint32_t key = key_of(i);
    if (key > kth) {
      const unsigned at = atomicAdd(&n_taken, 1u);
      candidates[at] = (static_cast<unsigned long long>(key) << 32) |
                       (~static_cast<uint32_t>(i));
    } else if (key == kth) {
      const unsigned at = atomicAdd(&n_equal_seen, 1u);
      if (at < kMaxTopK) equal_index[at] = i;
    }
  }
  __syncthreads();
  const unsigned base = n_taken;  // == k - need_equal
  if (n_equal_seen <= kMaxTopK) {
    // few ties: the `need_equal` lowest indices by counting smaller ones
    const unsigned count = n_equal_seen;
    if (static_cast<unsigned>(t) < count) {
      const int mine = equal_index[t];
      unsigned rank = 0u;
      for (unsigned j = 0; j < count; ++j) rank += equal_index[j] < mine;
      if (rank < need_equal)
        candidates[base + rank] =
            (static_cast<unsigned long long>(kth) << 32) | (~static_cast<uint32_t>(mine));
    }
  } else {
    // many ties: walk the vocabulary in index order until enough are found
    for (int start = 0; start < V; start += kThreads) {
      if (n_equal_taken >= need_equal) break;
      const int i = start + t;
      const bool equal = i < V && key_of(i) == kth;
      const unsigned long long ballot = __ballot(equal);
      const int lane = t % EI_WAVE, wave = t / EI_WAVE;
      const unsigned in_wave = __popcll(ballot & ((1ull << lane) - 1ull));
      __syncthreads();
      if (lane == 0) histogram[wave] = __popcll(ballot);
      __syncthreads();
      unsigned before = 0u;
      for (int w = 0; w < wave; ++w) before += histogram[w];
      unsigned total = 0u;
      for (int w = 0; w < kThreads / EI_WAVE; ++w) total += histogram[w];
      const unsigned already = n_equal_taken;
      if (equal) {
        const unsigned rank = already + before + in_wave;
        if (rank < need_equal)
          candidates[base + rank] =
              (static_cast<unsigned long long>(kth) << 32) | (~static_cast<uint32_t>(i));
      }
      __syncthreads();
      if (t == 0) n_equal_taken = already + total;
      __syncthreads();
    }
  }
  __syncthreads();
  sort_candidates(sh, k);
  draw_row(sh, k, top_p, seed, stream, counter, token, probability);
}

// Stream numbers and counters of the rows: in arrays on the GPU, or, for up to kKeyRows rows, in the
// kernel's arguments, which saves a copy to the GPU (a device operation of 3 us and its gap).
constexpr int kKeyRows = 64;
struct RowKeys {
  const int32_t* streams;                   // null: `given`
  const int32_t* counters;
  int32_t given[2 * kKeyRows];              // streams, then counters
  __device__ __forceinline__ uint32_t stream(int r) const {
    return static_cast<uint32_t>(streams ? streams[r] : given[r]);
  }
  __device__ __forceinline__ uint32_t counter(int r) const {
    return static_cast<uint32_t>(streams ? counters[r] : given[kKeyRows + r]);
  }
};

__global__ void __launch_bounds__(kThreads)
sample_kernel(const float* __restrict__ logits, int V, float temperature, float top_p, int top_k,
              uint64_t seed, RowKeys keys, int32_t* __restrict__ tokens,
              float* __restrict__ probabilities) {
  __shared__ SampleShared sh;
  const int r = blockIdx.x;
  sample_row(logits + static_cast<size_t>(r) * V, V, temperature, top_k < V ? top_k : V, top_p, seed,
             keys.stream(r), keys.counter(r), tokens + r, probabilities ? probabilities + r : nullptr, sh);
}

// Wide vocabularies, with many blocks a row before one block finishes it.  A small k takes two
// steps, (A) and (3), any other three:
// (A) every block writes to its part of the row's list what of its 4,096 keys can belong to the top k;
// (1) counts of the rows' keys by their upper 12 bits (sign, exponent, three bits of the
//     fraction), summed over the blocks of a row in `bins` [rows, 4096];
// (2) every block finds the bin T that holds the k-th largest key and appends its keys from
//     bins >= T to the row's list (fewer than k pairs above T, plus whatever shares T);
// (3) one block a row samples from the list exactly as sample_kernel does from the row, or
//     from the row itself if the list overflowed or is tied beyond reach; it then clears the
//     row's count and, after (1), its bins, which therefore start at zero in every call once
//     they did in the first.
// 8 rows of 151,936, k 20: (1) 7.2, (2) 7.4 and (3) 11.9 us before, (A) 6.5 and (3) 8.5 now.
constexpr int kChunk = 4096, kChunkThreads = 256;
// a row's scratch, in 4-byte units: its bins, its count (4 units, which keeps the list
// 8-byte aligned) and its list of up to kListCapacity pairs; a row's place does not depend
// on how many rows a call has
constexpr int kListCapacity = 8192;
constexpr long long kScratchPerRow = kBins + 4 + 2ll * kListCapacity;
__device__ __forceinline__ unsigned* row_bins(unsigned* scratch, int r) {
  return scratch + static_cast<size_t>(r) * kScratchPerRow;
}
__device__ __forceinline__ unsigned* row_count(unsigned* scratch, int r) {
  return row_bins(scratch, r) + kBins;
}
__device__ __forceinline__ unsigned long long* row_list(unsigned* scratch, int r) {
  return reinterpret_cast<unsigned long long*>(row_bins(scratch, r) + kBins + 4);
}

__global__ void __launch_bounds__(kChunkThreads)
sample_count_kernel(const float* __restrict__ logits, int V, float temperature,
                    unsigned* __restrict__ scratch) {
  __shared__ unsigned local[kBins];
  const int t = threadIdx.x, r = blockIdx.y;
  for (int b = t; b < kBins; b += kChunkThreads) local[b] = 0u;
  __syncthreads();
  const float* row = logits + static_cast<size_t>(r) * V;
  const int begin = blockIdx.x * kChunk, end = min(V, begin + kChunk);
  for (int i = begin + t; i < end; i += kChunkThreads)
    atomicAdd(&local[sortable_key(scaled_logit(row[i], temperature, true)) >> kBinShift], 1u);
  __syncthreads();
  for (int b = t; b < kBins; b += kChunkThreads)
    if (local[b]) atomicAdd(&row_bins(scratch, r)[b], local[b]);
}

__global__ void __launch_bounds__(kChunkThreads)
sample_gather_kernel(const float* __restrict__ logits, int V, float temperature, int k,
                     unsigned* __restrict__ scratch) {
  static_assert(kChunkThreads == 256, "count_above works on 256 counts");
  __shared__ unsigned partial[4];
  __shared__ unsigned long long mine[kChunk];
  __shared__ unsigned threshold_bin, n_mine, base;
  const int t = threadIdx.x, r = blockIdx.y;
  constexpr int per = kBins / kChunkThreads;
  const unsigned* bins = row_bins(scratch, r);
  unsigned own[per], sum = 0u;
#pragma unroll
  for (int j = 0; j < per; ++j) {
    own[j] = bins[t * per + j];
    sum += own[j];
  }
  if (t == 0) n_mine = 0u;
  unsigned above = count_above(sum, partial);   // keys in the bins of the threads after this one
  if (above < static_cast<unsigned>(k) && above + sum >= static_cast<unsigned>(k)) {
    int bin = per - 1;                      // exactly one thread gets here (k <= V = all keys)
#pragma unroll
    for (; bin > 0; --bin) {
      if (above + own[bin] >= static_cast<unsigned>(k)) break;
      above += own[bin];
    }
    threshold_bin = static_cast<unsigned>(t * per + bin);
  }
  __syncthreads();
  const unsigned first_bin = threshold_bin;
  const float* row = logits + static_cast<size_t>(r) * V;
  const int begin = blockIdx.x * kChunk, end = min(V, begin + kChunk);
  for (int i = begin + t; i < end; i += kChunkThreads) {
    const uint32_t key = sortable_key(scaled_logit(row[i], temperature, true));
    if ((key >> kBinShift) >= first_bin)
      mine[atomicAdd(&n_mine, 1u)] =
          (static_cast<unsigned long long>(key) << 32) | (~static_cast<uint32_t>(i));
  }
  __syncthreads();
  const unsigned count = n_mine;
  if (t == 0) base = count ? atomicAdd(row_count(scratch, r), count) : 0u;
  __syncthreads();
  unsigned long long* list = row_list(scratch, r);
  for (unsigned j = t; j < count; j += kChunkThreads)
    if (base + j < static_cast<unsigned>(kListCapacity)) list[base + j] = mine[j];
}

// Step (A), k <= kLocalTopK.  L, the k-th largest of the largest keys of 256 groups of 8, is no larger
// than the k-th largest key of the chunk, and few keys lie above it (k 20: 21 of 2,048 evenly spread
// ones).  The block writes every key above L and of those equal to L the first in index order as far as
// k is not reached, so a chunk of equal keys (a masked part of the vocabulary) gives k pairs and not
// 2,048.  Every chunk has the same number of places in the list and fills the rest with zeros (no
// logit has this key); one that needs more leaves kOverflow.
// A chain of short steps, bound by their latency: 6.5 us for 8 rows of 151,936; with 16 keys a thread, unrolled, 17.2 (14 KB of code that runs
// once), in loops 11.5; with the search for L by every wave instead of one 12.3 (its scalar
// instructions fill a compute unit's issue slots).
constexpr int kLocalTopK = 128, kLocalThreads = 512, kLocalChunk = 2048;
constexpr unsigned long long kOverflow = ~0ull;        // (no logit has this key either)
__global__ void __launch_bounds__(kLocalThreads)
sample_local_kernel(const float* __restrict__ logits, int V, float temperature, int k,
                    unsigned* __restrict__ scratch, unsigned places) {
  constexpr int per = kLocalChunk / kLocalThreads, waves = kLocalThreads / EI_WAVE;
  static_assert(kLocalThreads == 2 * 256 && per * waves <= EI_WAVE, "two threads a group; one lane a (round, wave) in the scan");
  __shared__ __attribute__((aligned(16))) uint32_t largest[kLocalThreads];
  __shared__ unsigned counts[2][per * waves], totals[2];
  __shared__ uint32_t threshold;
  const int t = threadIdx.x, r = blockIdx.y, lane = t % EI_WAVE, wave = t / EI_WAVE;
  const float* row = logits + static_cast<size_t>(r) * V;
  const int begin = blockIdx.x * kLocalChunk + t;
  float z[per];
#pragma unroll
  for (int j = 0; j < per; ++j) z[j] = row[min(begin + j * kLocalThreads, V - 1)];
  uint32_t key[per], best = 0u;
#pragma unroll
  for (int j = 0; j < per; ++j) {           // (0: past the row's end)
    key[j] = begin + j * kLocalThreads < V ? sortable_key(scaled_logit(z[j], temperature, true)) : 0u;
    best = max(best, key[j]);
  }
  largest[t] = best;
  __syncthreads();
  if (wave == 0) {                          // bit by bit from the top
    uint32_t m[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {           // (any two threads' keys make a group)
      const uint2 two = reinterpret_cast<const uint2*>(largest)[j * EI_WAVE + lane];
      m[j] = max(two.x, two.y);
    }
    uint32_t limit = 0u;
#pragma unroll 1
    for (int bit = 31; bit >= 0; --bit) {
      const uint32_t at_least = limit | (1u << bit);
      const int count = __popcll(__ballot(m[0] >= at_least)) + __popcll(__ballot(m[1] >= at_least)) +
                        __popcll(__ballot(m[2] >= at_least)) + __popcll(__ballot(m[3] >= at_least));
      if (count >= k) limit = at_least;
      if (count == k) {                     // exactly the k groups wanted: what is above at_least - 1
        limit = at_least - 1u;
        break;
      }
    }
    if (lane == 0) threshold = limit;
  }
  __syncthreads();
  const uint32_t limit = threshold;
  unsigned long long above[per], equal[per];
#pragma unroll
  for (int j = 0; j < per; ++j) {           // (round j, wave): index order
    above[j] = __ballot(key[j] > limit);
    equal[j] = __ballot(key[j] == limit && limit != 0u);
    if (lane == 0) {
      counts[0][j * waves + wave] = static_cast<unsigned>(__popcll(above[j]));
      counts[1][j * waves + wave] = static_cast<unsigned>(__popcll(equal[j]));
    }
  }
  __syncthreads();
  if (wave < 2) {                           // exclusive sums: keys above by wave 0, equal by wave 1
    const unsigned own = lane < per * waves ? counts[wave][lane] : 0u;
    unsigned inclusive = own;
#pragma unroll
    for (int offset = 1; offset < per * waves; offset <<= 1) {
      const unsigned other = __shfl_up(inclusive, offset, EI_WAVE);
      if (lane >= offset) inclusive += other;
    }
    if (lane < per * waves) counts[wave][lane] = inclusive - own;
    if (lane == per * waves - 1) totals[wave] = inclusive;
  }
  __syncthreads();
  const unsigned n_above = totals[0];
  const unsigned n_equal = n_above < static_cast<unsigned>(k)
                               ? min(totals[1], static_cast<unsigned>(k) - n_above) : 0u;
  const unsigned taken = n_above + n_equal;
  unsigned long long* list = row_list(scratch, r) + blockIdx.x * places;
  if (taken > places) {                     // the same for the whole block
    if (t == 0) list[0] = kOverflow;
    return;
  }
  const unsigned long long below = (1ull << lane) - 1ull;
#pragma unroll
  for (int j = 0; j < per; ++j) {
    if ((above[j] | equal[j]) == 0ull) continue;        // (most: 64 keys of which none is taken)
    const bool is_above = key[j] > limit, is_equal = key[j] == limit && limit != 0u;
    const unsigned among_above = counts[0][j * waves + wave] + __popcll(above[j] & below);
    const unsigned among_equal = counts[1][j * waves + wave] + __popcll(equal[j] & below);
    if (is_above || (is_equal && among_equal < n_equal))
      list[is_above ? among_above : n_above + among_equal] =
          (static_cast<unsigned long long>(key[j]) << 32) | (~static_cast<uint32_t>(begin + j * kLocalThreads));
  }
  for (unsigned j = taken + t; j < places; j += kLocalThreads) list[j] = 0ull;
}

// One block samples one row from a list of at least k pairs, held in registers (zeros are no pairs).
// Bins of the upper 12 bits leave the pairs that can belong to the top k; while more than kRanked
// are left, the next 12 bits and the last 8 narrow them down.  Up to kRanked pairs are put in order
// by counting the larger ones (no two are equal, and ties of a key are in index order by
// themselves); more are sorted.  False (nothing written): more than kMaxTopK pairs are left at the
// end, i.e. ties that need the row in index order.
constexpr int kRanked = 256;
__device__ bool sample_list(const unsigned long long (&pair)[kListCapacity / kThreads], int k,
                            float top_p, uint64_t seed, uint32_t stream, uint32_t counter,
                            int32_t* token, float* probability, SampleShared& sh) {
  constexpr int per = kListCapacity / kThreads, bins_each = kBins / kThreads;
  static_assert(bins_each == 4, "a thread's bins are one 16-byte access");
  const int t = threadIdx.x, lane = t % EI_WAVE, wave = t / EI_WAVE;
  uint4* bins = reinterpret_cast<uint4*>(sh.histogram);
  unsigned prefix = 0u, wanted = static_cast<unsigned>(k), sure = 0u, left = 0u;
  int shift = 32;
  for (int bits = 12; shift > 0; bits = shift < 12 ? shift : 12) {
    const int next = shift - bits;
    bins[t] = uint4{0u, 0u, 0u, 0u};
    if (t == 0) sh.n_taken = 0u;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < per; ++j) {
      const uint32_t key = static_cast<uint32_t>(pair[j] >> 32);
      if (key != 0u && (shift == 32 || key >> shift == prefix))
        atomicAdd(&sh.histogram[(key >> next) & ((1u << bits) - 1u)], 1u);
    }
    __syncthreads();
    const uint4 own = bins[t];              // the counts of all higher bins, see count_above
    const unsigned sum = own.x + own.y + own.z + own.w;
    unsigned inclusive = sum;
#pragma unroll
    for (int offset = 1; offset < EI_WAVE; offset <<= 1) {
      const unsigned other = __shfl_down(inclusive, offset, EI_WAVE);
      if (lane + offset < EI_WAVE) inclusive += other;
    }
    if (lane == 0) sh.wave_totals[wave] = inclusive;
    __syncthreads();
    unsigned above = inclusive - sum;
    for (int w = wave + 1; w < kThreads / EI_WAVE; ++w) above += sh.wave_totals[w];
    if (above < wanted && above + sum >= wanted) {      // exactly one thread
      int bin = 3;
      const unsigned each[4] = {own.x, own.y, own.z, own.w};
      unsigned count = each[3];
#pragma unroll
      for (int j = 2; j >= 0; --j)
        if (bin == j + 1 && above + count < wanted) {
          above += count;
          bin = j;
          count = each[j];
        }
      sh.select_prefix = prefix << bits | static_cast<unsigned>(4 * t + bin);
      sh.select_remaining = wanted - above;
      sh.n_equal_seen = count;
    }
    __syncthreads();
    prefix = sh.select_prefix;
    sure += wanted - sh.select_remaining;
    wanted = sh.select_remaining;
    left = sure + sh.n_equal_seen;
    shift = next;
    if (left <= static_cast<unsigned>(kRanked)) break;
  }
  if (left > static_cast<unsigned>(kMaxTopK)) return false;             // the same for every thread
#pragma unroll
  for (int j = 0; j < per; ++j)
    if (pair[j] != 0ull && static_cast<uint32_t>(pair[j] >> 32) >> shift >= prefix)
      sh.candidates[atomicAdd(&sh.n_taken, 1u)] = pair[j];
  __syncthreads();
  if (left <= static_cast<unsigned>(kRanked)) {
    unsigned long long mine = 0ull;
    int rank = k;
    if (t < static_cast<int>(left)) {
      mine = sh.candidates[t];
      rank = 0;
      for (unsigned j = 0; j < left; j += 16) {         // (16 reads on their way at once)
        unsigned long long other[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) other[u] = sh.candidates[j + u];
#pragma unroll
        for (int u = 0; u < 16; ++u) rank += j + u < left && other[u] > mine;
      }
    }
    __syncthreads();
    if (rank < k) sh.candidates[rank] = mine;
    __syncthreads();
  } else {
    sort_candidates(sh, static_cast<int>(left));
  }
  draw_row(sh, k, top_p, seed, stream, counter, token, probability);
  return true;
}

__global__ void __launch_bounds__(kThreads)
sample_list_kernel(const float* __restrict__ logits, int V, float temperature, float top_p,
                   int top_k, uint64_t seed, RowKeys keys, int32_t* __restrict__ tokens,
                   float* __restrict__ probabilities, unsigned* __restrict__ scratch, int local_pairs) {
  __shared__ SampleShared sh;
  const int r = blockIdx.x, t = threadIdx.x;
  const int k = top_k < V ? top_k : V;
  // after step (A) `local_pairs` places, else what the row's count says
  const unsigned listed = local_pairs > 0 ? static_cast<unsigned>(local_pairs) : *row_count(scratch, r);
  unsigned long long pair[kListCapacity / kThreads];    // asked for with the count, not after it
#pragma unroll
  for (int j = 0; j < kListCapacity / kThreads; ++j)
    if (local_pairs == 0 || j * kThreads < local_pairs) pair[j] = row_list(scratch, r)[t + j * kThreads];
  bool overflow = listed > static_cast<unsigned>(kListCapacity);
#pragma unroll
  for (int j = 0; j < kListCapacity / kThreads; ++j) {
    if (static_cast<unsigned>(t + j * kThreads) >= listed) pair[j] = 0ull;
    overflow = overflow || pair[j] == kOverflow;
  }
  const uint32_t stream = keys.stream(r), counter = keys.counter(r);
  float* probability = probabilities ? probabilities + r : nullptr;
  bool done = false;
  if (!__syncthreads_or(overflow))
    done = sample_list(pair, k, top_p, seed, stream, counter, tokens + r, probability, sh);
  if (!done) {
    __syncthreads();
    sample_row(logits + static_cast<size_t>(r) * V, V, temperature, k, top_p, seed, stream, counter,
               tokens + r, probability, sh);
  }
  if (local_pairs > 0) return;
  for (int b = t; b < kBins; b += kThreads) row_bins(scratch, r)[b] = 0u;
  if (t == 0) *row_count(scratch, r) = 0u;  // (every thread has read it: there were barriers since)
}


}  // namespace

// Elements of `partial` (float2) that ei_argmax wants for these sizes; 0: it needs none.
extern "C" int ei_argmax_partial_size(int rows, int V) {
  if (rows < 1 || V <= 2 * kArgmaxChunk) return 0;
  const long long size = static_cast<long long>(rows) * ((V + kArgmaxChunk - 1) / kArgmaxChunk);
  return size < (1ll << 30) ? static_cast<int>(size) : 0;
}

// `partial` (float2 [rows, chunks], or null) lets a wide vocabulary be searched by many
// blocks a row; without it one block takes a row.  The result is the same either way.
extern "C" int ei_argmax(const float* logits, int rows, int V, int32_t* tokens,
                         float* probabilities, void* partial, long long partial_size,
                         hipStream_t stream) {
  EI_REQUIRE(rows > 0 && V > 0, "argmax: sizes must be positive");
  EI_REQUIRE(logits && tokens, "argmax: null pointer");
  const int want = ei_argmax_partial_size(rows, V);
  if (partial && want > 0) {
    EI_REQUIRE(partial_size >= want, "argmax: the partial buffer is too small");
    const int chunks = (V + kArgmaxChunk - 1) / kArgmaxChunk;
    argmax_chunks_kernel<<<dim3(chunks, rows), kArgmaxThreads, 0, stream>>>(
        logits, V, static_cast<float2*>(partial));
    argmax_merge_kernel<<<rows, EI_WAVE, 0, stream>>>(static_cast<const float2*>(partial), chunks,
                                                      tokens, probabilities);
    EI_LAUNCH_CHECK();
  }
  argmax_kernel<<<rows, kThreads, 0, stream>>>(logits, V, tokens, probabilities);
  EI_LAUNCH_CHECK();
}

// The partial results of ei_argmax_static: one copy on every GPU, at an address of its own
// there.  Host code never passes this name to a kernel (on the host it is a stand-in, not a
// device address); it asks the runtime for the address once per device and uses that.
static __device__ __align__(256) float2 argmax_static_scratch[EI_ARGMAX_STATIC_MAX_PARTIALS];

constexpr int kStaticDevices = 64;
static std::atomic<float2*> argmax_static_address[kStaticDevices];

// The array's address on the current device: looked up once per device (with that device
// current) and kept.  The lookup may load the library's code on the device, which a stream
// that is being captured does not allow, so it is never started from a call under capture.
static int argmax_static_resolve(float2** out, bool capturing) {
  int device = -1;
  hipError_t status = hipGetDevice(&device);
  if (status != hipSuccess) {
    ei_set_error(hipGetErrorString(status));
    return static_cast<int>(status);
  }
  EI_REQUIRE(device >= 0 && device < kStaticDevices, "argmax_static: device index out of range");
  float2* partial = argmax_static_address[device].load(std::memory_order_acquire);
  if (partial == nullptr) {
    EI_REQUIRE(!capturing, "argmax_static: the first call on a device cannot run under stream "
                           "capture; call ei_argmax_static_prepare() on that device before");
    void* address = nullptr;
    status = hipGetSymbolAddress(&address, HIP_SYMBOL(argmax_static_scratch));
    if (status != hipSuccess) {
      ei_set_error(hipGetErrorString(status));
      return static_cast<int>(status);
    }
    EI_REQUIRE(address != nullptr, "argmax_static: the static buffer has no device address");
    partial = static_cast<float2*>(address);
    argmax_static_address[device].store(partial, std::memory_order_release);
  }
  *out = partial;
  return 0;
}

// See sampling_static.h.
extern "C" int ei_argmax_static_prepare() {
  float2* partial = nullptr;
  return argmax_static_resolve(&partial, false);
}

// See sampling_static.h.  Nothing is allocated, by this call or by the lookup.
extern "C" int ei_argmax_static(const float* logits, int rows, int V, int32_t* tokens,
                                float* probabilities, hipStream_t stream) {
  EI_REQUIRE(rows > 0 && V > 0, "argmax_static: sizes must be positive");
  EI_REQUIRE(logits && tokens, "argmax_static: null pointer");
  const long long chunks = (static_cast<long long>(V) + kArgmaxChunk - 1) / kArgmaxChunk;
  if (V <= 2 * kArgmaxChunk) {          // one block a row: no partial results
    argmax_kernel<<<rows, kThreads, 0, stream>>>(logits, V, tokens, probabilities);
    EI_LAUNCH_CHECK();
  }
  EI_REQUIRE(static_cast<long long>(rows) * chunks <= EI_ARGMAX_STATIC_MAX_PARTIALS,
             "argmax_static: rows * ceil(V / 4096) exceeds the 65536 partial results that the "
             "library's static buffer holds");
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(stream, &capture) != hipSuccess) capture = hipStreamCaptureStatusNone;
  float2* partial = nullptr;
  const int resolved = argmax_static_resolve(&partial, capture != hipStreamCaptureStatusNone);
  if (resolved != 0) return resolved;
  argmax_chunks_kernel<<<dim3(static_cast<unsigned>(chunks), rows), kArgmaxThreads, 0, stream>>>(
      logits, V, partial);
  argmax_merge_kernel<<<rows, EI_WAVE, 0, stream>>>(partial, static_cast<int>(chunks), tokens,
                                                    probabilities);
  EI_LAUNCH_CHECK();
}

// Scratch that ei_sample wants for a wide vocabulary, in 4-byte units (0: it needs none).
// It must be zero before its first use; every call leaves the bins and counts of its rows
// zero again, and a row's part lies at the same place whatever the number of rows.
constexpr int kWideVocabulary = 4 * kChunk;

extern "C" int ei_sample_scratch_size(int rows, int V) {
  if (rows < 1 || V <= kWideVocabulary) return 0;
  const long long size = rows * kScratchPerRow;
  return size < (1ll << 30) ? static_cast<int>(size) : 0;
}

// Places of a chunk's pairs in the list: evenly spread logits give 1.0 k pairs a chunk for a small k
// and 1.33 k at kLocalTopK.  Step (A) instead of (1) and (2) where there are half as many again as k;
// of a vocabulary of 151,936 a chunk can have 109, so for k <= 70 there.
static int local_places(int V, int k) {
  const int most = kListCapacity / ((V + kLocalChunk - 1) / kLocalChunk);
  return most < 2 * k + 16 ? most : 2 * k + 16;
}

static int sample_rows(const float* logits, int rows, int V, float temperature, float top_p, int top_k,
                       unsigned long long seed, const RowKeys& keys, int32_t* tokens,
                       float* probabilities, void* scratch, long long scratch_size, hipStream_t stream) {
  EI_REQUIRE(rows > 0 && V > 0, "sample: sizes must be positive");
  EI_REQUIRE(logits && tokens, "sample: null pointer");
  EI_REQUIRE(temperature > 0.f && temperature < 3.0e38f, "sample: temperature must be positive");
  EI_REQUIRE(top_p > 0.f && top_p <= 1.f, "sample: top_p must lie in (0, 1]");
  EI_REQUIRE(top_k >= 1 && (top_k < V ? top_k : V) <= kMaxTopK,
             "sample: min(top_k, vocabulary) must lie in 1..1024");
  const int want = ei_sample_scratch_size(rows, V);
  if (scratch && want > 0) {
    EI_REQUIRE(scratch_size >= want, "sample: the scratch buffer is too small");
    EI_REQUIRE((reinterpret_cast<uintptr_t>(scratch) & 7) == 0, "sample: scratch must be 8-byte aligned");
    unsigned* words = static_cast<unsigned*>(scratch);
    const int k = top_k < V ? top_k : V;
    int local_pairs = 0;
    if (k <= kLocalTopK && local_places(V, k) >= k + k / 2 + 4) {
      const int chunks = (V + kLocalChunk - 1) / kLocalChunk;
      const int places = local_places(V, k);
      local_pairs = places * chunks;
      sample_local_kernel<<<dim3(chunks, rows), kLocalThreads, 0, stream>>>(logits, V, temperature, k, words,
                                                                            static_cast<unsigned>(places));
    } else {
      const dim3 grid((V + kChunk - 1) / kChunk, rows);
      sample_count_kernel<<<grid, kChunkThreads, 0, stream>>>(logits, V, temperature, words);
      sample_gather_kernel<<<grid, kChunkThreads, 0, stream>>>(logits, V, temperature, k, words);
    }
    sample_list_kernel<<<rows, kThreads, 0, stream>>>(logits, V, temperature, top_p, top_k, seed, keys,
                                                      tokens, probabilities, words, local_pairs);
    EI_LAUNCH_CHECK();
  }
  sample_kernel<<<rows, kThreads, 0, stream>>>(logits, V, temperature, top_p, top_k, seed, keys,
                                               tokens, probabilities);
  EI_LAUNCH_CHECK();
}

// temperature > 0, 0 < top_p <= 1, 1 <= min(top_k, V) <= 1024.  `scratch` (uint32
// [scratch_size], or null): see ei_sample_scratch_size; the tokens are the same with or
// without it.
extern "C" int ei_sample(const float* logits, int rows, int V, float temperature, float top_p,
                         int top_k, unsigned long long seed, const int32_t* streams,
                         const int32_t* counters, int32_t* tokens, float* probabilities,
                         void* scratch, long long scratch_size, hipStream_t stream) {
  EI_REQUIRE(streams && counters, "sample: null pointer");
  RowKeys keys{};
  keys.streams = streams;
  keys.counters = counters;
  return sample_rows(logits, rows, V, temperature, top_p, top_k, seed, keys, tokens, probabilities,
                     scratch, scratch_size, stream);
}

// The same for at most 64 rows whose stream numbers and counters are in host memory, which this
// call has read when it returns.
extern "C" int ei_sample_given(const float* logits, int rows, int V, float temperature, float top_p,
                               int top_k, unsigned long long seed, const int32_t* streams,
                               const int32_t* counters, int32_t* tokens, float* probabilities,
                               void* scratch, long long scratch_size, hipStream_t stream) {
  EI_REQUIRE(streams && counters, "sample: null pointer");
  EI_REQUIRE(rows >= 1 && rows <= kKeyRows, "sample: host stream numbers are for 1..64 rows");
  RowKeys keys{};
  for (int r = 0; r < rows; ++r) {
    keys.given[r] = streams[r];
    keys.given[kKeyRows + r] = counters[r];
  }
  return sample_rows(logits, rows, V, temperature, top_p, top_k, seed, keys, tokens, probabilities,
                     scratch, scratch_size, stream);
}
