// Candidate selection for sampled decoding (sample_token_from_logits,
// src/runtime/layers.inl:491-600): per row, the repetition penalty
// (apply_repetition_penalty_inplace, layers.inl:471-489: a counted token's
// logit v becomes v / p when v > 0, else v * p), the temperature scaling
// v *= 1 / temperature (layers.inl:546-549), and the top_k largest values in
// descending order (layers.inl:552-568). Only these k candidates reach the
// host, which finishes the softmax, the nucleus cut and the draw in the
// reference's order. Greedy rows use k = 1 and scale 1: the argmax with the
// lowest index among equal values (argmax_index, layers.inl:459-469).
//
// Each value becomes a 64-bit key: the float's bits mapped to an unsigned
// order (sign flipped for positives, all bits flipped for negatives) in the
// high word and the inverted token id in the low word, so descending keys
// order by value and then by lower token id, and no two keys are equal.
//   stage 1: grid (kSampleSlices, rows): slice s of a row (at most kSliceKeys
//            tokens, 16 keys per thread in registers) keeps its top_k keys,
//            unordered;
//   stage 2: grid (rows): the top_k of the slices' survivors, ordered by
//            counting each key's larger ones, written as the row's candidates.
// The top_k of a workgroup's keys are those at or above the k-th largest,
// found by halving the key range and counting the keys above the midpoint
// (ballots and one barrier a round, about 20 rounds). What bounds it is that
// chain of rounds, not the logits. Sorting every slice of 4096 keys in LDS
// instead (78 barriers of 1024 threads) took 115 us for 16 rows of 248,320
// logits and the second sort 37 us; this form 20 us and 11 us.
#include "q35_device.h"
#include "q35_internal.h"

namespace q35 {
namespace {

constexpr int kSampleSlices = 64;
constexpr int kSliceThreads = 256, kSlicePer = 16, kSliceKeys = kSliceThreads * kSlicePer;
constexpr int kMergeThreads = 1024, kMergePer = kSampleSlices * kMaxCandidates / kMergeThreads;

__device__ __forceinline__ unsigned long long candidate_key(float v, int token) {
  const uint32_t u = __float_as_uint(v);
  const uint32_t ordered = (u & 0x80000000u) != 0u ? ~u : (u | 0x80000000u);
  return (static_cast<unsigned long long>(ordered) << 32) | static_cast<uint32_t>(~static_cast<uint32_t>(token));
}

__device__ __forceinline__ float key_value(unsigned long long key) {
  const uint32_t ordered = static_cast<uint32_t>(key >> 32);
  return __uint_as_float((ordered & 0x80000000u) != 0u ? (ordered & 0x7fffffffu) : ~ordered);
}

// Keys counted over a workgroup of WAVES wavefronts, PER of them in each
// thread's registers. Two count rows take turns, so a round needs one
// barrier: a row is written again only after the next round's barrier, which
// every reader of it has passed.
template <int WAVES, int PER>
struct KeyCounter {
  int (*rows)[WAVES];  // [2][WAVES] in LDS
  int turn = 0;
  template <typename Pred>
  __device__ __forceinline__ int count(const unsigned long long key[PER], Pred pred) {
    int n = 0;
#pragma unroll
    for (int i = 0; i < PER; ++i) n += __builtin_popcountll(q35_ballot(pred(key[i])));
    if ((threadIdx.x & 63) == 0) rows[turn][threadIdx.x >> 6] = n;
    lds_barrier();
    int total = 0;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) total += rows[turn][w];
    turn ^= 1;
    return q35_uniform(total);
  }
};

// The k-th largest of the workgroup's keys (1 <= k <= the number of nonzero
// keys; zeros are empty slots): first the largest high word with at least k
// keys at or above it, then, where several keys share that word, the same
// over their low words. A count of exactly k ends the search early: the
// returned bound then separates the k largest keys from the rest.
template <int WAVES, int PER>
__device__ __forceinline__ unsigned long long kth_key(const unsigned long long key[PER], int k,
                                                      KeyCounter<WAVES, PER> &c) {
  uint32_t lo = 0, hi = 0xffffffffu;
  while (lo < hi) {
    const uint32_t mid = lo + (hi - lo) / 2 + 1;
    const int n = c.count(key, [&](unsigned long long x) { return static_cast<uint32_t>(x >> 32) >= mid; });
    if (n == k) return static_cast<unsigned long long>(mid) << 32;
    if (n > k) lo = mid;
    else hi = mid - 1;
  }
  const uint32_t word = lo;
  k -= c.count(key, [&](unsigned long long x) { return static_cast<uint32_t>(x >> 32) > word; });
  lo = 0;
  hi = 0xffffffffu;
  while (lo < hi) {
    const uint32_t mid = lo + (hi - lo) / 2 + 1;
    const int n = c.count(key, [&](unsigned long long x) {
      return static_cast<uint32_t>(x >> 32) == word && static_cast<uint32_t>(x) >= mid;
    });
    if (n >= k) lo = mid;
    else hi = mid - 1;
  }
  return (static_cast<unsigned long long>(word) << 32) | lo;
}

__device__ __forceinline__ int row_candidates(const SampleArgs &a, int r) {
  return a.top_k != nullptr ? min(max(a.top_k[r], 0), kMaxCandidates) : 1;
}

__global__ __launch_bounds__(kSliceThreads) void sample_slices_kernel(SampleArgs a, unsigned long long *survivors) {
  constexpr int kWaves = kSliceThreads / 64;
  __shared__ int counts_lds[2][kWaves];
  __shared__ unsigned found;
  const int s = blockIdx.x, r = blockIdx.y, tid = threadIdx.x;
  const int per = (a.vocab + kSampleSlices - 1) / kSampleSlices;
  const int t0 = min(s * per, a.vocab), t1 = min(a.vocab, t0 + per);
  const float *logits = a.logits + static_cast<size_t>(r) * a.logits_stride;
  const float pen = a.penalties != nullptr ? a.penalties[r] : 1.0F;
  const int32_t *counts =
      a.counts != nullptr ? a.counts + static_cast<long long>(a.count_rows != nullptr ? a.count_rows[r] : r) * a.vocab
                          : nullptr;
  const float scale = a.inv_temperature != nullptr ? a.inv_temperature[r] : 1.0F;
  const int want = row_candidates(a, r);
  unsigned long long *out = survivors + (static_cast<size_t>(r) * kSampleSlices + s) * kMaxCandidates;
  const int k = min(want, t1 - t0);
  if (tid >= k && tid < want) out[tid] = 0ull;  // fewer tokens than candidates
  if (k <= 0) return;  // whole workgroup
  if (tid == 0) found = 0;
  const bool penalize = pen > 1.0F && counts != nullptr;
  float v[kSlicePer];
  int seen[kSlicePer];
#pragma unroll
  for (int i = 0; i < kSlicePer; ++i) {
    const int t = min(t0 + tid + i * kSliceThreads, t1 - 1);
    v[i] = logits[t];
    seen[i] = penalize ? counts[t] : 0;
  }
  unsigned long long key[kSlicePer];
#pragma unroll
  for (int i = 0; i < kSlicePer; ++i) {
    const int t = t0 + tid + i * kSliceThreads;
    float x = v[i];
    if (seen[i] > 0) x = x > 0.0F ? x / pen : x * pen;
    x *= scale;
    key[i] = t < t1 ? candidate_key(x, t) : 0ull;
  }
  KeyCounter<kWaves, kSlicePer> c{counts_lds};
  const unsigned long long bound = kth_key<kWaves, kSlicePer>(key, k, c);
#pragma unroll
  for (int i = 0; i < kSlicePer; ++i)
    if (key[i] >= bound) {
      const unsigned at = atomicAdd(&found, 1u);
      if (at < static_cast<unsigned>(k)) out[at] = key[i];
    }
}

__global__ __launch_bounds__(kMergeThreads) void sample_merge_kernel(SampleArgs a, const unsigned long long *survivors) {
  constexpr int kWaves = kMergeThreads / 64;
  __shared__ int counts_lds[2][kWaves];
  __shared__ unsigned found;
  __shared__ unsigned long long top[kMaxCandidates];
  const int r = blockIdx.x, tid = threadIdx.x;
  const int want = row_candidates(a, r);
  const unsigned long long *in = survivors + static_cast<size_t>(r) * kSampleSlices * kMaxCandidates;
  unsigned long long key[kMergePer];
#pragma unroll
  for (int i = 0; i < kMergePer; ++i) {
    const int e = tid + i * kMergeThreads;
    key[i] = e % kMaxCandidates < want ? in[e] : 0ull;
  }
  if (tid == 0) found = 0;
  if (tid < kMaxCandidates) top[tid] = 0ull;
  KeyCounter<kWaves, kMergePer> c{counts_lds};
  const int k = min(want, c.count(key, [](unsigned long long x) { return x != 0ull; }));
  if (k > 0) {
    const unsigned long long bound = kth_key<kWaves, kMergePer>(key, k, c);
#pragma unroll
    for (int i = 0; i < kMergePer; ++i)
      if (key[i] >= bound) {
        const unsigned at = atomicAdd(&found, 1u);
        if (at < static_cast<unsigned>(k)) top[at] = key[i];
      }
  }
  __syncthreads();
  if (tid >= kMaxCandidates) return;
  const unsigned long long mine = top[tid];
  int rank = 0;  // of a found key: how many are larger (the empty slots are 0)
#pragma unroll 8
  for (int i = 0; i < kMaxCandidates; ++i) rank += top[i] > mine;
  q35_candidate *out = a.out + static_cast<size_t>(r) * kMaxCandidates;
  if (tid < k) out[rank] = q35_candidate{key_value(mine), static_cast<int32_t>(~static_cast<uint32_t>(mine))};
  else out[tid] = q35_candidate{-INFINITY, -1};
}

}  // namespace

size_t sample_scratch_bytes(int rows) { return static_cast<size_t>(rows) * kSampleSlices * kMaxCandidates * sizeof(unsigned long long); }

hipError_t launch_sample_candidates(const SampleArgs &a, unsigned long long *scratch, hipStream_t stream) {
  if (a.rows <= 0) return hipSuccess;
  if (a.vocab <= 0 || a.vocab > kSampleSlices * kSliceKeys || a.logits == nullptr || a.out == nullptr ||
      scratch == nullptr)
    return hipErrorInvalidValue;
  Q35_LAUNCH((sample_slices_kernel), dim3(kSampleSlices, a.rows), dim3(kSliceThreads), 0, stream, a, scratch);
  Q35_LAUNCH((sample_merge_kernel), dim3(a.rows), dim3(kMergeThreads), 0, stream, a, scratch);
  return hipGetLastError();
}

}  // namespace q35
