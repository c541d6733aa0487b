// Stable sort of (key, index) pairs by counting passes of 8 or 9 bits, for
// the list builds of treebuild_dev.hip.  A pass is three launches: digit
// counts per block, their scan (a block per digit), and the scatter, whose
// ranks inside a block come from ballots (a wavefront takes consecutive pairs,
// so rank order is index order).  Bound: latency and the scattered writes; a
// block of 4096 pairs is 16 wavefronts of 4 pairs a lane, since 2^20 pairs are
// only a block per CU (4 wavefronts of 16 pairs a lane: 30 us a pass of 64-bit
// keys, so: 25; 2^21 pairs 34).  40 of 63 bits and the finish take 135 us for
// 2^20 pairs and 190 for 2^21; the library's merge of up to 2^20 pairs takes
// 205 us for any number of bits, its 63 bits of 2^21 pairs 260 with 70 us of
// memsets between the passes.
#pragma once
#include <hip/hip_runtime.h>

namespace pgsort {

using u64 = unsigned long long;
constexpr int kThreads = 1024;
constexpr int kWaves = kThreads / 64;
constexpr int kPer = 4;                    // pairs per thread
constexpr int kBlock = kThreads * kPer;    // pairs per block
constexpr int kScanThreads = 256;

template <int kDigits, class K>
__device__ inline int digit_of(K key, int shift) {
  return (int)((key >> shift) & (K)(kDigits - 1));
}

// count[digit * gridDim.x + block].
template <int kDigits, class K>
__global__ __launch_bounds__(kThreads) void radix_count(int n, int shift, const K* __restrict__ key,
                                                        int* __restrict__ count) {
  __shared__ int s[kWaves * kDigits];
  const int tid = threadIdx.x, wave = tid >> 6;
  for (int e = tid; e < kWaves * kDigits; e += kThreads) s[e] = 0;
  __syncthreads();
  const long long i0 = (long long)blockIdx.x * kBlock + tid;
#pragma unroll
  for (int r = 0; r < kPer; ++r) {
    const long long i = i0 + r * kThreads;
    if (i < n) atomicAdd(&s[wave * kDigits + digit_of<kDigits>(key[i], shift)], 1);
  }
  __syncthreads();
  if (tid >= kDigits) return;
  int c = 0;
  for (int w = 0; w < kWaves; ++w) c += s[w * kDigits + tid];
  count[(size_t)tid * gridDim.x + blockIdx.x] = c;
}

// Inclusive scan over the block's values; s: an int per wavefront.
__device__ inline int block_scan(int v, int* s) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int o = 1; o < 64; o <<= 1) {
    const int x = __shfl_up(v, o);
    if (lane >= o) v += x;
  }
  __syncthreads();
  if (lane == 63) s[wave] = v;
  __syncthreads();
  for (int w = 0; w < wave; ++w) v += s[w];
  return v;
}

// Block d: exclusive scan of the row of digit d (nb blocks) in place, and its
// total.
__global__ __launch_bounds__(kScanThreads) void radix_scan(int nb, int* __restrict__ count,
                                                       int* __restrict__ total) {
  __shared__ int s[kScanThreads / 64];
  __shared__ int s_all;
  int* row = count + (size_t)blockIdx.x * nb;
  int run = 0;
  for (int b0 = 0; b0 < nb; b0 += kScanThreads) {
    const int b = b0 + threadIdx.x;
    const int c = b < nb ? row[b] : 0;
    const int v = block_scan(c, s);
    if (b < nb) row[b] = run + v - c;
    if (threadIdx.x == kScanThreads - 1) s_all = v;
    __syncthreads();
    run += s_all;
    __syncthreads();
  }
  if (threadIdx.x == 0) total[blockIdx.x] = run;
}

// vin null: the values are the pairs' places.
template <int kDigits, class K>
__global__ __launch_bounds__(kThreads) void radix_scatter(
    int n, int shift, const K* __restrict__ kin, const int* __restrict__ vin,
    K* __restrict__ kout, int* __restrict__ vout, const int* __restrict__ count,
    const int* __restrict__ total) {
  __shared__ int s_at[kWaves * kDigits];
  __shared__ int s_scan[kWaves];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (int e = tid; e < kWaves * kDigits; e += kThreads) s_at[e] = 0;
  __syncthreads();
  const long long i0 = (long long)blockIdx.x * kBlock + wave * (64 * kPer) + lane;
  K key[kPer];
  int val[kPer], rank[kPer];
#pragma unroll
  for (int r = 0; r < kPer; ++r) {
    const long long i = i0 + r * 64;
    key[r] = i < n ? kin[i] : (K)0;
    val[r] = i < n ? (vin ? vin[i] : (int)i) : 0;
  }
  int* cnt = s_at + wave * kDigits;
#pragma unroll
  for (int r = 0; r < kPer; ++r) {
    const bool valid = i0 + r * 64 < n;
    const int d = digit_of<kDigits>(key[r], shift);
    u64 same = __ballot(valid);
#pragma unroll
    for (int b = 0; 1 << b < kDigits; ++b) {
      const bool bit = (d >> b) & 1;
      const u64 m = __ballot(bit);
      same &= bit ? m : ~m;
    }
    const int below = __popcll(same & ((1ULL << lane) - 1ULL));
    const int before = cnt[d];  // of this wavefront's earlier rounds
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    if (valid && below == 0) cnt[d] = before + __popcll(same);
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    rank[r] = before + below;
  }
  __syncthreads();
  {
    // digit tid: first place of each wavefront's pairs
    const int t = tid < kDigits ? total[tid] : 0;
    int at = block_scan(t, s_scan) - t;
    if (tid < kDigits) {
      at += count[(size_t)tid * gridDim.x + blockIdx.x];
      for (int w = 0; w < kWaves; ++w) {
        const int c = s_at[w * kDigits + tid];
        s_at[w * kDigits + tid] = at;
        at += c;
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kPer; ++r) {
    if (i0 + r * 64 >= n) continue;
    const int p = cnt[digit_of<kDigits>(key[r], shift)] + rank[r];
    kout[p] = key[r];
    vout[p] = val[r];
  }
}

// Pairs sorted by the bits from `shift` up, into the order of all bits: every
// pair of a run of equal upper bits counts the ones before it.  A run of more
// than kMaxRun pairs sets *long_run and is left unsorted; its pairs see that from
// the pair kMaxRun places away, without counting (counting up to 2048 others first
// made lists of 2^20 particles in runs of 2048 1.2 ms slower).
// Runs of 512 cost about as much to count as to sort again with all bits.
constexpr int kMaxRun = 512;
template <class K>
__global__ __launch_bounds__(256) void radix_finish(int n, int shift, const K* __restrict__ kin,
                                                    const int* __restrict__ vin,
                                                    K* __restrict__ kout, int* __restrict__ vout,
                                                    int* __restrict__ long_run) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const K own = kin[i], up = own >> shift;
  int at = i;
  auto same = [&](int j) { return j >= 0 && j < n && kin[j] >> shift == up; };
  if (same(i - 1) || same(i + 1)) {
    if ((n - i > kMaxRun && same(i + kMaxRun)) || same(i - kMaxRun)) {
      *long_run = 1;
    } else {  // fewer than 2 kMaxRun pairs to look at
      int lo = i - 1, hi = i + 1;
      for (; same(lo); --lo) at -= kin[lo] > own;  // comes after this one
      for (; same(hi); ++hi) at += kin[hi] < own;
      // the middle of a long run, whose pairs all keep their places
      if (hi - lo - 1 > kMaxRun) at = i;
    }
  }
  kout[at] = own;
  vout[at] = vin[i];
}

inline int blocks_of(int n) { return (int)(((long long)n + kBlock - 1) / kBlock); }

// Ints of scratch for n pairs.
inline size_t scratch_ints(int n) { return (size_t)512 * (blocks_of(n) + 1); }

template <int kDigits, class K>
int radix_passes(int n, K* const key[2], int* const val[2], int begin, int end, int* scratch,
                 hipStream_t st) {
  const int nb = blocks_of(n);
  int* total = scratch + (size_t)kDigits * nb;
  int bits = 0;
  while (1 << bits < kDigits) ++bits;
  int cur = 0;
  for (int shift = begin; shift < end; shift += bits) {
    hipLaunchKernelGGL((radix_count<kDigits, K>), dim3(nb), dim3(kThreads), 0, st, n, shift,
                       key[cur], scratch);
    hipLaunchKernelGGL(radix_scan, dim3(kDigits), dim3(kScanThreads), 0, st, nb, scratch, total);
    hipLaunchKernelGGL((radix_scatter<kDigits, K>), dim3(nb), dim3(kThreads), 0, st, n, shift,
                       key[cur], shift == begin ? nullptr : val[cur], key[1 - cur], val[1 - cur],
                       scratch, total);
    cur = 1 - cur;
  }
  return cur;
}

// Sorts by bits [begin, end) with the values 0, 1, ..., n - 1, through the
// two buffers of each kind; returns which of them (0 or 1) holds the result.
// Input: key[0].  The keys' bits from `end` up are 0.  Passes of 9 bits where
// that makes them fewer.
template <class K>
int radix_sort(int n, K* const key[2], int* const val[2], int begin, int end, int* scratch,
               hipStream_t st) {
  const int bits = end - begin;
  return (bits + 8) / 9 < (bits + 7) / 8
             ? radix_passes<512>(n, key, val, begin, end, scratch, st)
             : radix_passes<256>(n, key, val, begin, end, scratch, st);
}

}  // namespace pgsort
