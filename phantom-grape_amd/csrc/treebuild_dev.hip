// libpgtree_dev.so: the interaction lists of the batched TreePM and
// Barnes-Hut calls, built on the GPU from positions already in HBM.
//
// Same algorithm and same output as the host builder libpgtree.so
// (treebuild.cpp), array for array: Morton keys (21 bits per axis), a stable
// radix sort, the octree (its nodes level by level), bottom-up moments, i-groups of
// <= ncrit particles in Morton order, TreePM ghosts and grid-based j-lists
// in grid-cell order, the Barnes-Hut walk with the opening test of
// PG5/newton_quad/source.cpp:660-707, and groups ordered by decreasing cost.
// Every FP64 operation that decides or produces a value is evaluated in the
// host builder's order with contraction off, so the two agree bit for bit;
// only the numbering of the Barnes-Hut cells differs (here: the order of the
// octree levels), so cell lists match as lists of cell contents.
//
// The build is synchronous on the caller's stream: list lengths are read back
// between phases to size the next allocation.
#include "pgamd_common.h"
#include "pgamd_api.h"

#include "radix_sort.h"

#include <hipcub/device/device_radix_sort.hpp>
#include <hipcub/device/device_scan.hpp>

#include <algorithm>
#include <climits>
#include <cmath>
#include <map>
#include <unordered_map>
#include <vector>

using namespace pgamd;

namespace {

using u64 = unsigned long long;
constexpr int kLevels = 21;  // bits per axis of the Morton key

// ------------------------------------------------------------ allocations
// Device memory of the builds comes from a cache: blocks rounded up to powers
// of two and kept for reuse once released, so that repeated builds make no
// hipMalloc / hipFree calls (hipFree also waits for the whole device).  A
// build releases its temporaries after its stream has drained, lists release
// theirs in pgt_dev_free after a device synchronisation; both run under the
// library's mutex.  The cache holds its peak size until the process ends, or
// until the device has no memory left for another block.
struct Cache {
  std::map<size_t, std::vector<void*>> free;
  std::unordered_map<void*, size_t> size;
  // null if the device has no memory left, also after the unused blocks are
  // given back
  void* try_get(size_t bytes) {
    if (bytes > (size_t)1 << 48) return nullptr;  // a length beyond the range of int
    size_t b = 256;
    while (b < bytes) b <<= 1;
    std::vector<void*>& v = free[b];
    if (!v.empty()) {
      void* p = v.back();
      v.pop_back();
      return p;
    }
    void* p = try_malloc(b);
    if (!p) {
      for (auto& f : free) {
        for (void* q : f.second) {
          PGAMD_HIP_CHECK(hipFree(q));
          size.erase(q);
        }
        f.second.clear();
      }
      p = try_malloc(b);
    }
    if (p) size[p] = b;
    return p;
  }
  void* get(size_t bytes) {
    void* p = try_get(bytes);
    if (!p) PGAMD_HIP_CHECK(hipErrorOutOfMemory);
    return p;
  }
  static void* try_malloc(size_t bytes) {
    void* p = nullptr;
    if (hipMalloc(&p, bytes) == hipSuccess) return p;
    (void)hipGetLastError();
    return nullptr;
  }
  void put(void* p) { free[size.at(p)].push_back(p); }
};
Cache g_cache;

struct Mem {
  std::vector<void*> ptrs;
  template <class T>
  T* get(size_t n) {
    void* p = g_cache.get(std::max<size_t>(n, 1) * sizeof(T));
    ptrs.push_back(p);
    return static_cast<T*>(p);
  }
  template <class T>
  T* try_get(size_t n) {
    void* p = g_cache.try_get(std::max<size_t>(n, 1) * sizeof(T));
    if (p) ptrs.push_back(p);
    return static_cast<T*>(p);
  }
  void free_all() {
    for (void* p : ptrs) g_cache.put(p);
    ptrs.clear();
  }
};

// out[n] = out[n - 1] + in[n - 1] (0 for n = 0): the total of an exclusive
// scan, also written to *host (mapped pinned memory) unless it is null.
__global__ void k_scan_total(const int* __restrict__ in, int* __restrict__ out, int n,
                             int* __restrict__ host) {
  if (threadIdx.x == 0 && blockIdx.x == 0) {
    const int t = n > 0 ? out[n - 1] + in[n - 1] : 0;
    out[n] = t;
    if (host) *host = t;
  }
}

// Exclusive scan of n <= kSmallScan ints in one block: all of a thread's
// loads (four consecutive ints of every tile; in and out are aligned to 16
// bytes, as all allocations are) go out together, wavefronts scan
// their part of each tile, the block scans the wavefronts' sums.  out[n] =
// total, also written to *host (unless null).  14029 ints: 4 us; the library's
// scan and a launch for the total take 9, in three launches.
constexpr int kSmallScanThreads = 1024;
constexpr int kScanTiles = 8;
constexpr int kSmallScan = 4 * kSmallScanThreads * kScanTiles;
__global__ __launch_bounds__(kSmallScanThreads) void k_scan_small(const int* __restrict__ in,
                                                                  int* __restrict__ out, int n,
                                                                  int* __restrict__ host) {
  constexpr int kWaves = kSmallScanThreads / 64, kSums = kWaves * kScanTiles;
  __shared__ int s[kSums];  // tile by tile
  const int lane = threadIdx.x & 63, wave = threadIdx.x / 64;
  int v[kScanTiles][4], end[kScanTiles];
#pragma unroll
  for (int t = 0; t < kScanTiles; ++t) {
    const int i = 4 * (t * kSmallScanThreads + (int)threadIdx.x);
    int4 x = make_int4(0, 0, 0, 0);
    if (i + 3 < n)
      x = *reinterpret_cast<const int4*>(in + i);
    else if (i < n)
      x = make_int4(in[i], i + 1 < n ? in[i + 1] : 0, i + 2 < n ? in[i + 2] : 0, 0);
    v[t][0] = x.x;
    v[t][1] = x.y;
    v[t][2] = x.z;
    v[t][3] = x.w;
  }
#pragma unroll
  for (int t = 0; t < kScanTiles; ++t) {
    if (4 * t * kSmallScanThreads < n) {  // uniform
      int e = v[t][0] + v[t][1] + v[t][2] + v[t][3];
      for (int o = 1; o < 64; o <<= 1) {
        const int x = __shfl_up(e, o);
        if (lane >= o) e += x;
      }
      end[t] = e;
      if (lane == 63) s[t * kWaves + wave] = e;
    } else if (lane == 63) {
      s[t * kWaves + wave] = 0;
    }
  }
  __syncthreads();
  if (wave == 0) {  // inclusive scan of the sums
    int run = 0;
    for (int k = 0; k < kSums; k += 64) {
      int e = s[k + lane];
      for (int o = 1; o < 64; o <<= 1) {
        const int x = __shfl_up(e, o);
        if (lane >= o) e += x;
      }
      s[k + lane] = run + e;
      run += __builtin_amdgcn_readlane(e, 63);
    }
    if (lane == 0) {
      out[n] = run;
      if (host) *host = run;
    }
  }
  __syncthreads();
#pragma unroll
  for (int t = 0; t < kScanTiles; ++t) {
    if (4 * t * kSmallScanThreads >= n) break;
    const int k = t * kWaves + wave;
    const int at = (k > 0 ? s[k - 1] : 0) + end[t] - (v[t][0] + v[t][1] + v[t][2] + v[t][3]);
    const int i = 4 * (t * kSmallScanThreads + (int)threadIdx.x);
    const int4 x = make_int4(at, at + v[t][0], at + v[t][0] + v[t][1],
                             at + v[t][0] + v[t][1] + v[t][2]);
    if (i + 3 < n) {
      *reinterpret_cast<int4*>(out + i) = x;
    } else if (i < n) {
      out[i] = x.x;
      if (i + 1 < n) out[i + 1] = x.y;
      if (i + 2 < n) out[i + 2] = x.z;
    }
  }
}

// Result of one build: device arrays in the host builder's layout.
struct Lists {
  Mem mem;
  long long np = 0, ng = 0, ni = 0, nj = 0, nc = 0, ncells = 0, work_pp = 0, work_pc = 0;
  double* pos = nullptr;  // [np][3]
  int* src = nullptr;
  int *ioff = nullptr, *icnt = nullptr, *ilist = nullptr;
  int *joff = nullptr, *jcnt = nullptr, *jlist = nullptr;
  int *coff = nullptr, *ccnt = nullptr, *clist = nullptr;
  int* order = nullptr;
  double* cells = nullptr;  // [ncells][10]
};

// Pinned ints in which kernels report counts to the host; builds run one at a
// time under the library's mutex.
constexpr int kHostInts = 64;
enum HostSlot {
  kSlotLevels = 0,  // k_tree_levels
  kSlotTotal = 32,  // scan totals
  kSlotTotal2 = 33,
  kSlotPool = 34,  // OpenPool::used
  kSlotWork = 40,  // two 64-bit sums
  kSlotBox = 48,   // six doubles
};
int* host_ints() {
  static int* p = nullptr;
  if (!p) PGAMD_HIP_CHECK(hipHostMalloc((void**)&p, kHostInts * sizeof(int), hipHostMallocMapped));
  return p;
}
int* host_dev(int* host) {
  int* dev = nullptr;
  PGAMD_HIP_CHECK(hipHostGetDevicePointer((void**)&dev, host, 0));
  return dev;
}

// Sorts of fewer pairs go to the library (its one-block and merge sorts), of
// more to radix_sort.h: whole builds of 2^17 particles take 378 us (TreePM)
// and 400 (Barnes-Hut) with the library's sorts, 348 and 418 with those; of
// 2^18 particles 505 and 497 against 380 and 488, of 2^19 610 and 636 against
// 429 and 584.
constexpr int kCountingFrom = 1 << 18;
// The upper bits of a 63-bit Morton key that are sorted first: they tell
// apart cells of 2^-13 of the box, so few particles are left equal.
constexpr int kFirstBits = 40;

__global__ void k_iota(int n, int* __restrict__ v) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) v[i] = i;
}

__global__ void k_fill_int(int n, int v, int* __restrict__ out) {
  for (int i = threadIdx.x; i < n; i += blockDim.x) out[i] = v;
}

inline dim3 grid_for(long long n, int threads = 256) {
  return dim3((unsigned)std::max<long long>(1, (n + threads - 1) / threads));
}

// Temporary storage for one build, released at its end.
struct Build {
  hipStream_t st;
  Mem tmp;
  Mem pool;  // of OpenPool: given up first where the device has no memory left
  void* cub = nullptr;
  size_t cub_bytes = 0;
  explicit Build(hipStream_t s) : st(s) {}
  ~Build() {
    PGAMD_HIP_CHECK(hipStreamSynchronize(st));
    if (cub) g_cache.put(cub);
    tmp.free_all();
    pool.free_all();
  }
  void* cub_tmp(size_t bytes) {
    if (bytes > cub_bytes) {
      PGAMD_HIP_CHECK(hipStreamSynchronize(st));  // the old block may still be in use
      if (cub) g_cache.put(cub);
      cub = g_cache.get(bytes);
      cub_bytes = bytes;
    }
    return cub;
  }
  // out[k] = sum in[0..k), out[n] = total (out has n + 1 entries), not waited
  // for; the total goes to the host's slot (-1: none) through mapped memory.
  void scan(const int* in, int* out, int n, int slot) {
    int* dev = slot < 0 ? nullptr : host_dev(host_ints()) + slot;
    if (n <= kSmallScan) {
      hipLaunchKernelGGL(k_scan_small, dim3(1), dim3(kSmallScanThreads), 0, st, in, out, n, dev);
    } else {
      size_t b = 0;
      PGAMD_HIP_CHECK(hipcub::DeviceScan::ExclusiveSum(nullptr, b, in, out, n, st));
      PGAMD_HIP_CHECK(hipcub::DeviceScan::ExclusiveSum(cub_tmp(b), b, in, out, n, st));
      hipLaunchKernelGGL(k_scan_total, dim3(1), dim3(64), 0, st, in, out, n, dev);
    }
    PGAMD_HIP_CHECK(hipGetLastError());
  }
  // What the kernels queued so far have reported.
  const volatile int* wait() {
    PGAMD_HIP_CHECK(hipStreamSynchronize(st));
    return host_ints();
  }
  // Stable library sort of (key, value) pairs.
  template <class K>
  void sort_pairs(const K* kin, K* kout, const int* vin, int* vout, int n, int end_bit) {
    if (n <= 0) return;
    size_t b = 0;
    PGAMD_HIP_CHECK(
        hipcub::DeviceRadixSort::SortPairs(nullptr, b, kin, kout, vin, vout, n, 0, end_bit, st));
    PGAMD_HIP_CHECK(hipcub::DeviceRadixSort::SortPairs(cub_tmp(b), b, kin, kout, vin, vout, n, 0,
                                                       end_bit, st));
  }
  // Stable sort of n keys (overwritten) by bits [0, bits) with the values 0
  // .. n - 1: *skey and *perm are set to the sorted arrays.  Only the upper
  // `first` bits take counting passes; pairs they leave equal are put in
  // order by one more launch.  *long_run (0 before) is set if a run of them is
  // too long for that: the caller, with its next read-back, then sorts again
  // with first = bits.
  template <class K>
  void sort_keys(K* key, int n, int bits, int first, K** skey, int** perm, int* long_run) {
    K* k[2] = {key, tmp.get<K>(n)};
    int* v[2] = {tmp.get<int>(n), tmp.get<int>(n)};
    int cur = 1;
    if (n < kCountingFrom) {
      hipLaunchKernelGGL(k_iota, grid_for(n), dim3(256), 0, st, n, v[0]);
      sort_pairs(k[0], k[1], v[0], v[1], n, bits);
    } else {
      const int shift = std::max(0, bits - first);
      cur = pgsort::radix_sort(n, k, v, shift, bits, tmp.get<int>(pgsort::scratch_ints(n)), st);
      if (shift > 0) {
        hipLaunchKernelGGL(pgsort::radix_finish<K>, grid_for(n), dim3(256), 0, st, n, shift,
                           k[cur], v[cur], k[1 - cur], v[1 - cur], long_run);
        cur = 1 - cur;
      }
    }
    PGAMD_HIP_CHECK(hipGetLastError());
    *skey = k[cur];
    *perm = v[cur];
  }
};

// Bits needed to hold every value in [0, v].
inline int bits_for(long long v) {
  int b = 1;
  while ((1LL << b) <= v) ++b;
  return b;
}

// ------------------------------------------------------------ Morton keys
__device__ inline u64 spread3(u64 v) {
  v &= 0x1fffffULL;
  v = (v | v << 32) & 0x1f00000000ffffULL;
  v = (v | v << 16) & 0x1f0000ff0000ffULL;
  v = (v | v << 8) & 0x100f00f00f00f00fULL;
  v = (v | v << 4) & 0x10c30c30c30c30c3ULL;
  v = (v | v << 2) & 0x1249249249249249ULL;
  return v;
}

__global__ void k_keys(int n, const double* __restrict__ x, double lo0, double lo1, double lo2,
                       double s, u64* __restrict__ key, int* __restrict__ long_run) {
#pragma clang fp contract(off)
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i == 0) *long_run = 0;  // for sort_keys
  if (i >= n) return;
  const double lo[3] = {lo0, lo1, lo2};
  u64 k = 0;
  for (int d = 0; d < 3; ++d) {
    const double u = (x[3 * i + d] - lo[d]) * s;
    long long q = (long long)floor(u);
    q = q < 0 ? 0 : (q > (1 << kLevels) - 1 ? (1 << kLevels) - 1 : q);
    k |= spread3((u64)q) << (2 - d);
  }
  key[i] = k;
}

// Bounding box: per-block min/max of each axis, then one block over those.
__global__ void k_bbox_part(int n, const double* __restrict__ x, double* __restrict__ part) {
  __shared__ double s[6][256];
  double v[6] = {1e300, 1e300, 1e300, -1e300, -1e300, -1e300};
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
    for (int d = 0; d < 3; ++d) {
      v[d] = fmin(v[d], x[3 * i + d]);
      v[3 + d] = fmax(v[3 + d], x[3 * i + d]);
    }
  for (int k = 0; k < 6; ++k) s[k][threadIdx.x] = v[k];
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h)
      for (int k = 0; k < 6; ++k)
        s[k][threadIdx.x] = k < 3 ? fmin(s[k][threadIdx.x], s[k][threadIdx.x + h])
                                  : fmax(s[k][threadIdx.x], s[k][threadIdx.x + h]);
    __syncthreads();
  }
  if (threadIdx.x == 0)
    for (int k = 0; k < 6; ++k) part[6 * blockIdx.x + k] = s[k][0];
}

// One wavefront over the per-block results (minima and maxima do not depend
// on the order).
__global__ void k_bbox_final(int nb, const double* __restrict__ part, double* __restrict__ out) {
  const int lane = threadIdx.x;
  if (blockIdx.x != 0 || lane >= 64) return;
  double v[6] = {1e300, 1e300, 1e300, -1e300, -1e300, -1e300};
  for (int b = lane; b < nb; b += 64)
    for (int k = 0; k < 6; ++k)
      v[k] = k < 3 ? fmin(v[k], part[6 * b + k]) : fmax(v[k], part[6 * b + k]);
  for (int off = 32; off > 0; off >>= 1)
    for (int k = 0; k < 6; ++k) {
      const double o = __shfl_xor(v[k], off);
      v[k] = k < 3 ? fmin(v[k], o) : fmax(v[k], o);
    }
  if (lane == 0)
    for (int k = 0; k < 6; ++k) out[k] = v[k];
}

// Particles in Morton order: pos[p] = x[perm[p]], mass likewise (optional).
__global__ void k_gather(int n, const int* __restrict__ perm, const double* __restrict__ x,
                         const double* __restrict__ m, double* __restrict__ pos,
                         double* __restrict__ mm, int* __restrict__ src) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  const int i = perm[p];
  for (int d = 0; d < 3; ++d) pos[3 * p + d] = x[3 * i + d];
  if (m) mm[p] = m[i];
  src[p] = i;
}

// ------------------------------------------------------------ octree
// Nodes in level order.  Geometry: centre c (FP64) and side L / 2^level.
struct Nodes {
  int *lo, *hi, *par, *lev, *child;  // child[8 * k + octant], -1 if empty
  double* c;                         // [k][3]
  double *com, *m, *q;               // [k][3], [k], [k][6]
  int* cell;                         // cell index, -1 if none
};

__device__ inline int digit(u64 key, int shift) { return (int)((key >> shift) & 7ULL); }

// The whole octree from the sorted keys, without walking it level by level
// (15 levels of split, scan and read-back took 0.45 ms of a 2^21-particle
// build).  A cell of level l is a run of keys with the same first l digits,
// and it is a node if its parent holds more than `split` particles:
//   * particle i starts a cell at every level from a_i = 1 + the digits it
//     shares with particle i - 1 (0 for i = 0);
//   * its leaf is at level D_i, the first whose cell holds at most `split`
//     particles (or kLevels): a cell holds more if two of its particles are
//     `split` places apart, so D_i = 1 + the most digits shared by any pair
//     (j, j + split) with i - split <= j <= i, a sliding maximum.
// So the nodes that start at i are its cells of levels a_i .. D_i.  Counting
// them per level and block of particles, one scan numbers the nodes level by
// level, in particle order inside a level.
__device__ inline int shared_digits(u64 x, u64 y) {
  const u64 d = x ^ y;
  return d == 0 ? kLevels : (__clzll((long long)d) - 1) / 3;
}

// out[i] = max of v[max(0, i - w + 1) .. i], w <= kMaxWindow + 1, v[j] = 1 + the
// digits shared by keys j and j + split (0 if there is no such key).  By doubling
// in LDS.
constexpr int kWindowOut = 2048;
constexpr int kMaxWindow = 1024;
__global__ __launch_bounds__(256) void k_window_max(int n, int split, int w,
                                                    const u64* __restrict__ key,
                                                    unsigned char* __restrict__ out) {
  __shared__ unsigned char buf[2][kWindowOut + kMaxWindow];
  const int h = w - 1, m = kWindowOut + h;
  const int j0 = blockIdx.x * kWindowOut - h;
  for (int p = threadIdx.x; p < m; p += 256) {
    const int j = j0 + p;
    buf[0][p] = (unsigned char)(j >= 0 && j < n - split ? 1 + shared_digits(key[j], key[j + split]) : 0);
  }
  __syncthreads();
  int cur = 0, len = 1;  // buf[cur][p] = max over [p - len + 1, p]
  for (; 2 * len <= w; len *= 2) {
    for (int p = threadIdx.x; p < m; p += 256)
      buf[1 - cur][p] = max(buf[cur][p], p >= len ? buf[cur][p - len] : (unsigned char)0);
    cur = 1 - cur;
    __syncthreads();
  }
  for (int q = threadIdx.x; q < kWindowOut; q += 256) {
    const int i = blockIdx.x * kWindowOut + q, p = q + h;
    if (i < n) out[i] = max(buf[cur][p], buf[cur][p - (w - len)]);
  }
}

// A window of in (maxima over `len` places) made longer by h <= len places.  Large
// windows double from kMaxWindow + 1 on, so their launches grow with log2(split):
// TreePM lists of 2^18 particles with ncrit = 2^17 took 2753 us with one launch
// per 1024 places of the window, and take 860.
__global__ __launch_bounds__(256) void k_window_grow(int n, int h,
                                                     const unsigned char* __restrict__ in,
                                                     unsigned char* __restrict__ out) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) out[i] = max(in[i], i >= h ? in[i - h] : (unsigned char)0);
}

constexpr int kTreeLevels = kLevels + 1;
constexpr int kTreeRounds = 4;               // particles per thread of the two passes
constexpr int kTreeBlock = 256 * kTreeRounds;  // particles per block

// Levels a .. d of the nodes that start at particle i (a > d: none).
__device__ inline void start_levels(int i, int n, const u64* __restrict__ key,
                                    const unsigned char* __restrict__ leaf, int* a, int* d) {
  *a = 1;
  *d = 0;
  if (i >= n) return;
  *a = i == 0 ? 0 : 1 + shared_digits(key[i - 1], key[i]);
  *d = min((int)leaf[i], kLevels);
}

// count[l * gridDim.x + block] = nodes of level l that start in the block.
__global__ __launch_bounds__(256) void k_tree_count(int n, const u64* __restrict__ key,
                                                    const unsigned char* __restrict__ leaf,
                                                    int* __restrict__ count) {
  __shared__ int s_cnt[4][kTreeLevels];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int mine = 0;  // lane l: nodes of level l seen by this wavefront
  for (int r = 0; r < kTreeRounds; ++r) {
    int a, d;
    start_levels(blockIdx.x * kTreeBlock + r * 256 + threadIdx.x, n, key, leaf, &a, &d);
    for (int l = 0; l < kTreeLevels; ++l) {
      const int c = __popcll(__ballot(a <= l && l <= d));
      mine += lane == l ? c : 0;
    }
  }
  if (lane < kTreeLevels) s_cnt[wave][lane] = mine;
  __syncthreads();
  if (threadIdx.x < kTreeLevels)
    count[threadIdx.x * gridDim.x + blockIdx.x] =
        s_cnt[0][threadIdx.x] + s_cnt[1][threadIdx.x] + s_cnt[2][threadIdx.x] + s_cnt[3][threadIdx.x];
}

// host[l] = first node of level l, host[kTreeLevels] = number of nodes, from
// the scan of k_tree_count's counts (nb blocks), and host[kTreeLevels + 1] =
// *flag.
__global__ void k_tree_levels(int nb, const int* __restrict__ first, const int* __restrict__ flag,
                              int* __restrict__ host) {
  const int l = threadIdx.x;
  if (l == kTreeLevels + 1) host[l] = *flag;
  if (l <= kTreeLevels) host[l] = first[(size_t)l * nb];
}

// Nodes' first particle, level and parent, and the parents' child links
// (child[] is -1 before).  first[l * gridDim.x + block] = number of the
// block's first node of level l.
__global__ __launch_bounds__(256) void k_tree_fill(int n, const u64* __restrict__ key,
                                                   const unsigned char* __restrict__ leaf,
                                                   const int* __restrict__ first, Nodes nd) {
  // number of the first node of each level in wavefront 4 r + wave's particles
  __shared__ int s_at[4 * kTreeRounds][kTreeLevels];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int a[kTreeRounds], d[kTreeRounds];
#pragma unroll
  for (int r = 0; r < kTreeRounds; ++r) {
    start_levels(blockIdx.x * kTreeBlock + r * 256 + threadIdx.x, n, key, leaf, &a[r], &d[r]);
    for (int l = 0; l < kTreeLevels; ++l) {
      const int c = __popcll(__ballot(a[r] <= l && l <= d[r]));
      if (lane == l) s_at[4 * r + wave][l] = c;
    }
  }
  __syncthreads();
  if (threadIdx.x < kTreeLevels) {
    int run = first[threadIdx.x * gridDim.x + blockIdx.x];
    for (int q = 0; q < 4 * kTreeRounds; ++q) {
      const int c = s_at[q][threadIdx.x];
      s_at[q][threadIdx.x] = run;
      run += c;
    }
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kTreeRounds; ++r) {
    const int i = blockIdx.x * kTreeBlock + r * 256 + threadIdx.x;
    const u64 own = i < n ? key[i] : 0;
    int up = 0;  // the last node of the level above that starts at or before i
    for (int l = 0; l < kTreeLevels; ++l) {
      const int base = s_at[4 * r + wave][l];
      const bool starts = a[r] <= l && l <= d[r];
      const u64 m = __ballot(starts);
      const int below = __popcll(m & ((1ULL << lane) - 1ULL));
      if (starts) {
        const int id = base + below;
        nd.lo[id] = i;
        nd.lev[id] = l;
        nd.par[id] = l == 0 ? -1 : up;
        if (l > 0) nd.child[8 * (size_t)up + digit(own, 3 * (kLevels - l))] = id;
      }
      up = base + below + (starts ? 1 : 0) - 1;
    }
  }
}

// Each node's end and centre.  The end is the first key beyond lo with other
// leading digits (doubling steps, then bisection); the centre is the root's
// moved by a quarter of the side per level, in the order a walk from the
// root adds them.
__global__ __launch_bounds__(256) void k_tree_nodes(int nn, int n, const u64* __restrict__ key,
                                                    double L, double c0, double c1, double c2,
                                                    Nodes nd) {
#pragma clang fp contract(off)
  const int k = blockIdx.x * 256 + threadIdx.x;
  if (k >= nn) return;
  const int lo = nd.lo[k], lev = nd.lev[k];
  const u64 own = key[lo];
  const int shift = 3 * (kLevels - lev);
  int a = lo, step = 1;  // key[a] lies in the node
  int b = n;             // key[b] does not (or b = n)
  if (lev > 0) {
    while (lo + step < n) {
      if ((key[lo + step] >> shift) != (own >> shift)) {
        b = lo + step;
        break;
      }
      a = lo + step;
      step *= 2;
    }
    while (b - a > 1) {
      const int mid = a + (b - a) / 2;
      if ((key[mid] >> shift) == (own >> shift))
        a = mid;
      else
        b = mid;
    }
  }
  nd.hi[k] = b;
  double c[3] = {c0, c1, c2};
  double l = L;
  for (int q = 0; q < lev; ++q) {
    const int o = digit(own, 3 * (kLevels - 1 - q));  // octant: x is bit 2, y bit 1, z bit 0
    c[0] = c[0] + ((o & 4) ? 0.25 : -0.25) * l;
    c[1] = c[1] + ((o & 2) ? 0.25 : -0.25) * l;
    c[2] = c[2] + ((o & 1) ? 0.25 : -0.25) * l;
    l *= 0.5;
  }
  for (int q = 0; q < 3; ++q) nd.c[3 * (size_t)k + q] = c[q];
}

__global__ void k_copy_ints(int n, const int* __restrict__ in, int* __restrict__ out) {
  for (int i = threadIdx.x; i < n; i += blockDim.x) out[i] = in[i];
}

__global__ __launch_bounds__(256) void k_fill_int4(size_t n4, int v, int4* __restrict__ out) {
  const size_t i = blockIdx.x * (size_t)256 + threadIdx.x;
  if (i < n4) out[i] = make_int4(v, v, v, v);
}

// Moments of one node; q[5] follows from the trace.
__device__ inline void store_moments(const Nodes& nd, int k, double M, const double com[3],
                                     double q[6]) {
#pragma clang fp contract(off)
  nd.m[k] = M;
  for (int d = 0; d < 3; ++d) nd.com[3 * (size_t)k + d] = com[d];
  q[5] = -(q[0] + q[3]);
  for (int t = 0; t < 6; ++t) nd.q[6 * (size_t)k + t] = q[t];
}

__device__ inline bool is_leaf(const Nodes& nd, int k) {
  const int4* c = reinterpret_cast<const int4*>(nd.child + 8 * (size_t)k);
  const int4 a = c[0], b = c[1];
  return (a.x & a.y & a.z & a.w & b.x & b.y & b.z & b.w) < 0;  // no child: all are -1
}

// Moments of every leaf: sums over its particles in order, the loads of four in
// flight.  A leaf of particles that the key cannot split is one thread's chain:
// 64 of 16384 particles each took 8.8 ms with a load at a time, so 4.1.
__global__ __launch_bounds__(256) void k_leaf_moments(int nn, Nodes nd,
                                                      const double* __restrict__ pos,
                                                      const double* __restrict__ mm) {
#pragma clang fp contract(off)
  const int k = blockIdx.x * 256 + threadIdx.x;
  if (k >= nn || !is_leaf(nd, k)) return;
  const int lo = nd.lo[k], hi = nd.hi[k];
  double M = 0, c[3] = {0, 0, 0}, q[6] = {0, 0, 0, 0, 0, 0}, com[3];
#pragma unroll 4
  for (int p = lo; p < hi; ++p) {
    const double mi = mm[p];
    M += mi;
    for (int d = 0; d < 3; ++d) c[d] += mi * pos[3 * (size_t)p + d];
  }
  for (int d = 0; d < 3; ++d) com[d] = M > 0 ? c[d] / M : nd.c[3 * (size_t)k + d];
#pragma unroll 4
  for (int p = lo; p < hi; ++p) {
    const double mi = mm[p];
    double dd[3];
    for (int d = 0; d < 3; ++d) dd[d] = pos[3 * (size_t)p + d] - com[d];
    const double r2 = dd[0] * dd[0] + dd[1] * dd[1] + dd[2] * dd[2];
    int kk = 0;
    for (int x = 0; x < 2; ++x)
      for (int y = x; y < 3; ++y) {
        double v = 3.0 * dd[x] * dd[y];
        if (x == y) v -= r2;
        q[kk++] += mi * v;
      }
  }
  store_moments(nd, k, M, com, q);
}

// Moments of node k from its children's, in octant order.
__device__ inline void combine_moments(const Nodes& nd, int k) {
#pragma clang fp contract(off)
  if (is_leaf(nd, k)) return;
  double M = 0, c[3] = {0, 0, 0}, q[6] = {0, 0, 0, 0, 0, 0}, com[3];
  for (int o = 0; o < 8; ++o) {
    const int ch = nd.child[8 * (size_t)k + o];
    if (ch < 0) continue;
    M += nd.m[ch];
    for (int d = 0; d < 3; ++d) c[d] += nd.m[ch] * nd.com[3 * (size_t)ch + d];
  }
  for (int d = 0; d < 3; ++d) com[d] = M > 0 ? c[d] / M : nd.c[3 * (size_t)k + d];
  for (int o = 0; o < 8; ++o) {
    const int ch = nd.child[8 * (size_t)k + o];
    if (ch < 0) continue;
    double dd[3];
    for (int d = 0; d < 3; ++d) dd[d] = nd.com[3 * (size_t)ch + d] - com[d];
    const double r2 = dd[0] * dd[0] + dd[1] * dd[1] + dd[2] * dd[2];
    int kk = 0;
    for (int x = 0; x < 2; ++x)
      for (int y = x; y < 3; ++y) {
        double v = 3.0 * dd[x] * dd[y];
        if (x == y) v -= r2;
        q[kk] += nd.q[6 * (size_t)ch + kk] + nd.m[ch] * v;
        ++kk;
      }
  }
  store_moments(nd, k, M, com, q);
}

// The inner nodes [a, b) of one level, children already done.
__global__ __launch_bounds__(64) void k_inner_moments(int a, int b, Nodes nd) {
  const int k = a + blockIdx.x * 64 + threadIdx.x;
  if (k < b) combine_moments(nd, k);
}

// The first levels' inner nodes in one block, level `top` - 1 first.
struct LevelStarts {
  int v[kLevels + 2];
};
constexpr int kTopNodes = 512;  // a level this small is left to the one block
__global__ __launch_bounds__(kTopNodes) void k_top_moments(int top, LevelStarts ls, Nodes nd) {
  for (int l = top - 1; l >= 0; --l) {
    const int k = ls.v[l] + threadIdx.x;
    if (k < ls.v[l + 1]) combine_moments(nd, k);
    __threadfence_block();
    __syncthreads();
  }
}

// i-groups: nodes of <= ncrit particles whose parent holds more, and nodes
// the key cannot split (level kLevels: more than ncrit particles inside one
// cell of side L / 2^21), which form one group of all their particles.
__global__ void k_group_flag(int nn, Nodes nd, int ncrit, int* __restrict__ flag) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nn) return;
  const int cnt = nd.hi[k] - nd.lo[k];
  const int par = nd.par[k];
  flag[k] = (cnt <= ncrit || nd.lev[k] >= kLevels) &&
            (par < 0 || nd.hi[par] - nd.lo[par] > ncrit);
}

__global__ void k_compact(int n, const int* __restrict__ flag, const int* __restrict__ off,
                          int* __restrict__ out) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k < n && flag[k]) out[off[k]] = k;
}

// Groups by first particle: inside a level the nodes are in that order
// already, so a group's rank is the sum over the levels of the groups that
// start before it, by bisection, a lane per level (32 lanes per group).  gn:
// groups in node order, those of level l at [off[level.v[l]],
// off[level.v[l + 1]]).
__global__ __launch_bounds__(256) void k_group_order(int ng, const int* __restrict__ gn,
                                                     const int* __restrict__ off, LevelStarts ls,
                                                     Nodes nd, int* __restrict__ out) {
  __shared__ int s_first[kLevels + 2];
  if (threadIdx.x < kLevels + 2) s_first[threadIdx.x] = off[ls.v[threadIdx.x]];
  __syncthreads();
  const int g = blockIdx.x * 8 + threadIdx.x / 32, l = threadIdx.x % 32;
  if (g >= ng) return;  // uniform per 32 lanes
  const int k = gn[g], lo = nd.lo[k];
  int rank = 0;
  if (l <= kLevels) {
    const int first = s_first[l];
    int a = first, b = s_first[l + 1];
    while (a < b) {
      const int mid = a + (b - a) / 2;
      if (nd.lo[gn[mid]] < lo)
        a = mid + 1;
      else
        b = mid;
    }
    rank = a - first;
  }
  for (int o = 16; o > 0; o >>= 1) rank += __shfl_xor(rank, o, 32);
  if (l == 0) out[rank] = k;
}

__global__ void k_group_icnt(int ng, const int* __restrict__ gnode, Nodes nd,
                             int* __restrict__ icnt) {
  const int g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g < ng) icnt[g] = nd.hi[gnode[g]] - nd.lo[gnode[g]];
}

__global__ void k_group_ilist(int ng, const int* __restrict__ gnode, Nodes nd,
                              const int* __restrict__ ioff, int* __restrict__ ilist) {
  const int g = blockIdx.x;
  const int lo = nd.lo[gnode[g]], hi = nd.hi[gnode[g]];
  for (int p = lo + threadIdx.x; p < hi; p += blockDim.x) ilist[ioff[g] + p - lo] = p;
}

// ------------------------------------------------------------ TreePM
// Periodic images of particle p within rcut of the box.
__device__ inline int ghosts_of(const double* __restrict__ pos, int p, double rcut) {
  int c = 1;
  for (int d = 0; d < 3; ++d) {
    const double v = pos[3 * (size_t)p + d];
    c *= 1 + (v >= 1.0 - rcut ? 1 : 0) + (v < rcut ? 1 : 0);
  }
  return c - 1;
}

// Inclusive scan of v over a block of 256 threads.
__device__ inline int scan256(int v) {
  __shared__ int s[4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x / 64;
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

// Ghosts per block of kGhostBlock particles, four consecutive ones a thread.
constexpr int kGhostBlock = 1024;
__global__ __launch_bounds__(256) void k_ghost_count(int n, const double* __restrict__ pos,
                                                     double rcut, int* __restrict__ cnt) {
  const int p0 = blockIdx.x * kGhostBlock + 4 * threadIdx.x;
  int c = 0;
  for (int q = 0; q < 4; ++q)
    if (p0 + q < n) c += ghosts_of(pos, p0 + q, rcut);
  c = scan256(c);
  if (threadIdx.x == 255) cnt[blockIdx.x] = c;
}

// Ghosts in particle order after the n particles; goff: of each block.
__global__ __launch_bounds__(256) void k_ghost_fill(int n, const int* __restrict__ goff,
                                                    double rcut, double* __restrict__ pos,
                                                    int* __restrict__ src) {
#pragma clang fp contract(off)
  const int p0 = blockIdx.x * kGhostBlock + 4 * threadIdx.x;
  int c[4], sum = 0;
  for (int q = 0; q < 4; ++q) {
    c[q] = p0 + q < n ? ghosts_of(pos, p0 + q, rcut) : 0;
    sum += c[q];
  }
  size_t o = (size_t)n + goff[blockIdx.x] + scan256(sum) - sum;
  for (int q = 0; q < 4; ++q) {
    if (c[q] == 0) continue;
    const size_t p = p0 + q;
    const double x0 = pos[3 * p], x1 = pos[3 * p + 1], x2 = pos[3 * p + 2];
    int lo_s[3], hi_s[3];
    const double xp[3] = {x0, x1, x2};
    for (int d = 0; d < 3; ++d) {
      lo_s[d] = xp[d] >= 1.0 - rcut ? -1 : 0;
      hi_s[d] = xp[d] < rcut ? 1 : 0;
    }
    for (int sx = lo_s[0]; sx <= hi_s[0]; ++sx)
      for (int sy = lo_s[1]; sy <= hi_s[1]; ++sy)
        for (int sz = lo_s[2]; sz <= hi_s[2]; ++sz) {
          if (!sx && !sy && !sz) continue;
          pos[3 * o + 0] = x0 + sx;
          pos[3 * o + 1] = x1 + sy;
          pos[3 * o + 2] = x2 + sz;
          src[o] = src[p];
          ++o;
        }
  }
}

struct Grid {
  double glo, h;
  int nc;
};

__device__ inline int cidx(const Grid& g, double v) {
#pragma clang fp contract(off)
  int c = (int)floor((v - g.glo) / g.h);
  return c < 0 ? 0 : (c > g.nc - 1 ? g.nc - 1 : c);
}

__global__ void k_cell_of(int np, const double* __restrict__ pos, Grid g,
                          unsigned* __restrict__ cell) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= np) return;
  cell[p] = (cidx(g, pos[3 * p]) * g.nc + cidx(g, pos[3 * p + 1])) * g.nc +
            cidx(g, pos[3 * p + 2]);
}

// Candidates in cell order: cpos[k] = position of particle cpart[k] rounded to
// FP32 and its index, so the list walk reads each row of cells as one
// contiguous range.  *wide is set if a coordinate lies outside [-2, 2], where
// kFineReach does not hold.
__global__ void k_cell_pos(int np, const int* __restrict__ cpart, const double* __restrict__ pos,
                           float4* __restrict__ cpos, int* __restrict__ wide) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= np) return;
  const int p = cpart[k];
  const double x = pos[3 * (size_t)p], y = pos[3 * (size_t)p + 1], z = pos[3 * (size_t)p + 2];
  cpos[k] = make_float4((float)x, (float)y, (float)z, __int_as_float(p));
  if (!(fmax(fmax(fabs(x), fabs(y)), fabs(z)) <= 2.0)) *wide = 1;
}

// cstart[c] = first position of cell c in the sorted cell array (c <= ncell).
__global__ void k_cell_start(int ncell, int np, const unsigned* __restrict__ scell,
                             int* __restrict__ cstart) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c > ncell) return;
  int a = 0, b = np;
  while (a < b) {
    const int mid = a + (b - a) / 2;
    if (scell[mid] < (unsigned)c)
      a = mid + 1;
    else
      b = mid;
  }
  cstart[c] = a;
}

// Group bounding boxes: [g][6] = min xyz, max xyz of the group's particles;
// one wavefront per group (minima and maxima do not depend on the order).
__global__ __launch_bounds__(256) void k_group_box(int ng, const int* __restrict__ gnode, Nodes nd,
                                                   const double* __restrict__ pos,
                                                   double* __restrict__ box) {
  const int lane = threadIdx.x & 63;
  const int g = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (g >= ng) return;  // uniform per wavefront
  const int k = gnode[g], lo = nd.lo[k], hi = nd.hi[k];
  double bmin[3] = {1e30, 1e30, 1e30}, bmax[3] = {-1e30, -1e30, -1e30};
  for (int p = lo + lane; p < hi; p += 64)
    for (int d = 0; d < 3; ++d) {
      bmin[d] = fmin(bmin[d], pos[3 * p + d]);
      bmax[d] = fmax(bmax[d], pos[3 * p + d]);
    }
  for (int off = 32; off > 0; off >>= 1)
    for (int d = 0; d < 3; ++d) {
      bmin[d] = fmin(bmin[d], __shfl_xor(bmin[d], off));
      bmax[d] = fmax(bmax[d], __shfl_xor(bmax[d], off));
    }
  if (lane < 3) {
    box[6 * g + lane] = lane == 0 ? bmin[0] : (lane == 1 ? bmin[1] : bmin[2]);
    box[6 * g + 3 + lane] = lane == 0 ? bmax[0] : (lane == 1 ? bmax[1] : bmax[2]);
  }
}

// Whether the box (bx[0..2] .. bx[3..5]) comes within the cut-off of v: the
// larger of the two one-sided distances per axis, or 0 inside.
__device__ inline bool in_reach(const double bx[6], const double v[3], double rc2) {
#pragma clang fp contract(off)
  double d2 = 0;
  for (int d = 0; d < 3; ++d) {
    const double e = fmax(fmax(bx[d] - v[d], v[d] - bx[3 + d]), 0.0);
    d2 += e * e;
  }
  return d2 < rc2;
}

// The squared distance of in_reach in FP32, from positions and box sides of at
// most 2 in size rounded to FP32: the sides' distances e are off by at most 3
// roundings of 2^-23, so near the cut-off the sum of e^2 is off by less than
// 2 sqrt(3) rcut 2^-21 + rcut^2 2^-20.  Farther from rcut^2 than `fine`, more
// than twice that, the FP32 comparison is the FP64 one.
__device__ inline float reach2(const float bx[6], float4 v) {
  const float x = fmaxf(fmaxf(bx[0] - v.x, v.x - bx[3]), 0.f);
  const float y = fmaxf(fmaxf(bx[1] - v.y, v.y - bx[4]), 0.f);
  const float z = fmaxf(fmaxf(bx[2] - v.z, v.z - bx[5]), 0.f);
  return x * x + y * y + z * z;
}
inline float fine_reach(double rcut) { return (float)(4e-6 * rcut + 4e-6 * rcut * rcut + 1e-11); }

// One wavefront per group walks the grid cells around the group box and
// writes the particles in reach to jlist[joff[g]...] and their number to
// jcnt[g], in cell order (cells by x, y, z index; a cell's particles by
// index).  The cells of one (x, y) row are consecutive, so a row is one range
// of the cell-sorted particles.  The rows'
// ranges are read by the lanes side by side, then kJlistDepth pieces of 64
// candidates at a time, whatever rows they belong to, so that their loads
// overlap.  The few candidates that FP32 cannot tell in or out (reach2; all of
// them where *wide) are decided by the FP64 positions.
//
// Bound: what the L2 delivers.  2^20-particle box, 7e7 candidates: 346 us with
// FP64 positions and one piece at a time, each waited for; 177 with four in
// flight (28 bytes a candidate); 145 with 16 bytes a candidate.
constexpr int kJlistDepth = 4;
__global__ __launch_bounds__(256) void k_treepm_jlist(int ng, const double* __restrict__ box,
                                                      const float4* __restrict__ cpos, Grid gr,
                                                      const int* __restrict__ cstart,
                                                      const double* __restrict__ pos,
                                                      const int* __restrict__ wide, float fine,
                                                      double rcut,
                                                      int* __restrict__ jcnt,
                                                      const int* __restrict__ joff,
                                                      int* __restrict__ jlist) {
#pragma clang fp contract(off)
  const int lane = threadIdx.x & 63;
  const int g = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (g >= ng) return;  // uniform per wavefront
  double bx[6];
  for (int d = 0; d < 6; ++d) bx[d] = box[6 * (size_t)g + d];
  const double rc2 = rcut * rcut;
  int c0[3], c1[3];
  for (int d = 0; d < 3; ++d) {
    c0[d] = cidx(gr, bx[d] - rcut);
    c1[d] = cidx(gr, bx[3 + d] + rcut);
  }
  float bf[6];
  for (int d = 0; d < 6; ++d) bf[d] = (float)bx[d];
  const float rc2f = (float)rc2, tol = *wide ? INFINITY : fine;
  int count = 0;
  int* out = jlist + joff[g];
  const int ny = c1[1] - c0[1] + 1, nrows = (c1[0] - c0[0] + 1) * ny;
  const u64 below = (1ULL << lane) - 1ULL;
  for (int r0 = 0; r0 < nrows; r0 += 64) {
    const int r = r0 + lane;
    int k0 = 0, k1 = 0;
    if (r < nrows) {
      const int row = ((c0[0] + r / ny) * gr.nc + c0[1] + r % ny) * gr.nc;
      k0 = cstart[row + c0[2]];
      k1 = cstart[row + c1[2] + 1];
    }
    const int pieces = (k1 - k0 + 63) / 64;
    int end = pieces;  // inclusive scan
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_up(end, o);
      if (lane >= o) end += v;
    }
    const int begin = end - pieces;
    const int total = __builtin_amdgcn_readlane(end, 63);
    for (int p0 = 0; p0 < total; p0 += kJlistDepth) {
      bool in[kJlistDepth];
      float4 v[kJlistDepth];
#pragma unroll
      for (int u = 0; u < kJlistDepth; ++u) {
        // the row of piece p0 + u: the last that begins at or before it
        const int p = min(p0 + u, total - 1);
        const int row = __popcll(__ballot(begin <= p)) - 1;
        const int a = __builtin_amdgcn_readlane(k0, row) +
                      64 * (p - __builtin_amdgcn_readlane(begin, row));
        const int k = a + lane, e = __builtin_amdgcn_readlane(k1, row);
        in[u] = p0 + u < total && k < e;
        v[u] = cpos[k < e ? k : a];
      }
#pragma unroll
      for (int u = 0; u < kJlistDepth; ++u) {
        const float d2 = reach2(bf, v[u]);
        const int part = __float_as_int(v[u].w);
        bool ok = in[u] && d2 < rc2f;
        if (in[u] && !(fabsf(d2 - rc2f) > tol)) {
          const double q[3] = {pos[3 * (size_t)part], pos[3 * (size_t)part + 1],
                               pos[3 * (size_t)part + 2]};
          ok = in_reach(bx, q, rc2);
        }
        const u64 mask = __ballot(ok);
        if (ok) out[count + __popcll(mask & below)] = part;
        count += __popcll(mask);
      }
    }
  }
  if (lane == 0) jcnt[g] = count;
}

// Candidates of each group: the particles in the rows of grid cells its walk
// visits (an upper bound of its list length).  One wavefront per group.
__global__ __launch_bounds__(256) void k_treepm_cand(int ng, const double* __restrict__ box,
                                                     Grid gr, const int* __restrict__ cstart,
                                                     double rcut, int* __restrict__ ccnt) {
#pragma clang fp contract(off)
  const int lane = threadIdx.x & 63;
  const int g = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (g >= ng) return;  // uniform per wavefront
  const double* bx = box + 6 * g;
  int c0[3], c1[3];
  for (int d = 0; d < 3; ++d) {
    c0[d] = cidx(gr, bx[d] - rcut);
    c1[d] = cidx(gr, bx[3 + d] + rcut);
  }
  const int ny = c1[1] - c0[1] + 1, nrows = (c1[0] - c0[0] + 1) * ny;
  int sum = 0;
  for (int r = lane; r < nrows; r += 64) {
    const int row = ((c0[0] + r / ny) * gr.nc + c0[1] + r % ny) * gr.nc;
    sum += cstart[row + c1[2] + 1] - cstart[row + c0[2]];
  }
  for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o);
  if (lane == 0) ccnt[g] = sum;
}

// jlist[joff[g] + k] = scratch[soff[g] + k] for k < jcnt[g]: the lists
// written at their candidate offsets, packed.  One wavefront per group, eight
// loads in flight (one at a time 140 us for 46 million entries).
__global__ __launch_bounds__(256) void k_pack_lists(int ng, const int* __restrict__ soff,
                                                    const int* __restrict__ jcnt,
                                                    const int* __restrict__ joff,
                                                    const int* __restrict__ scratch,
                                                    int* __restrict__ jlist) {
  const int lane = threadIdx.x & 63;
  const int g = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (g >= ng) return;
  const int* __restrict__ src = scratch + soff[g];
  int* __restrict__ dst = jlist + joff[g];
  const int n = jcnt[g];
  int k = lane;
  for (; k + 7 * 64 < n; k += 8 * 64) {
    int v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = src[k + 64 * u];
#pragma unroll
    for (int u = 0; u < 8; ++u) dst[k + 64 * u] = v[u];
  }
  for (; k < n; k += 64) dst[k] = src[k];
}

// ------------------------------------------------------------ Barnes-Hut
__global__ void k_cell_flag(int nn, Nodes nd, int* __restrict__ flag) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k < nn) flag[k] = nd.hi[k] - nd.lo[k] > 1;
}

__global__ void k_cell_fill(int nn, Nodes nd, const int* __restrict__ flag,
                            const int* __restrict__ off, double* __restrict__ cells) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nn) return;
  if (!flag[k]) {
    nd.cell[k] = -1;
    return;
  }
  const int c = off[k];
  nd.cell[k] = c;
  double* o = cells + 10 * (size_t)c;
  o[0] = nd.com[3 * k];
  o[1] = nd.com[3 * k + 1];
  o[2] = nd.com[3 * k + 2];
  o[3] = nd.m[k];
  for (int t = 0; t < 6; ++t) o[4 + t] = nd.q[6 * k + t];
}

__device__ inline double bh_box_d2(const double* __restrict__ gc, double li,
                                   const double* __restrict__ c) {
#pragma clang fp contract(off)
  double d2 = 0;
  for (int d = 0; d < 3; ++d) {
    const double e = fmax(fabs(c[d] - gc[d]) - li, 0.0);
    d2 += e * e;
  }
  return d2;
}

// Node data the Barnes-Hut walk reads for one child: what it becomes if it is
// opened, and its centre of mass (32 bytes), and for the lists its item.
// Arrays of 16 bytes a node: the eight lanes that examine a node's children (numbered
// consecutively in octant order) read 128 consecutive bytes of each, where
// 64-byte records made every lane of every load a cache line of its own; the
// walk is bound by the lookups and misses of the vector cache.
struct WalkNodes {
  // what a list holds of the node: its cell, or its only particle (from a
  // 16-byte record of range and cell k_bh_list took 313 us, so 288)
  int* item;
  // {x, y} of the queue entry (below) and com x as two words
  int4* ex;
  double2* yz;  // com y, z
};

// A node to be expanded: {first child, octant mask}, or a leaf (a node of up
// to nleaf particles or one that the key cannot split), whose particles are
// listed one by one: {lo, kLeafEntry | count}.
constexpr unsigned kLeafEntry = 0x80000000u;

struct WalkNode {
  int x;
  unsigned y;
  double com[3];
  __device__ inline bool leaf() const { return y & kLeafEntry; }
  __device__ inline int count() const { return (int)(y & ~kLeafEntry); }  // of a leaf
};

__device__ inline WalkNode load_walk(const WalkNodes& w, int k) {
  const int4 e = w.ex[k];
  const double2 yz = w.yz[k];
  return WalkNode{e.x, (unsigned)e.y,
                  {__longlong_as_double((long long)((u64)(unsigned)e.w << 32 | (unsigned)e.z)), yz.x, yz.y}};
}

__global__ void k_walk_nodes(int nn, int nleaf, Nodes nd, WalkNodes out) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nn) return;
  const int lo = nd.lo[k], hi = nd.hi[k];
  int first = -1, mask = 0;
  for (int o = 7; o >= 0; --o) {
    const int ch = nd.child[8 * k + o];
    if (ch >= 0) {
      first = ch;
      mask |= 1 << o;
    }
  }
  const bool leaf = hi - lo <= nleaf || mask == 0;
  const u64 cx = (u64)__double_as_longlong(nd.com[3 * k]);
  out.item[k] = hi - lo > 1 ? nd.cell[k] : lo;
  out.ex[k] = make_int4(leaf ? lo : first, leaf ? (int)(kLeafEntry | (unsigned)(hi - lo)) : mask,
                        (int)(unsigned)cx, (int)(unsigned)(cx >> 32));
  out.yz[k] = make_double2(nd.com[3 * k + 1], nd.com[3 * k + 2]);
}

// Depth of the walk stack: the depth-first walk keeps at most 7 pending
// siblings per level below the root, plus the 8 children of the node being
// expanded (internal nodes sit above level kLevels).
constexpr int kWalkDepth = 7 * (kLevels - 1) + 8;
constexpr int kWalkWaves = 4;  // groups (one wavefront each) per block

// Block b of a launch of nb blocks runs on XCD b % 8; renumber the blocks so
// that each XCD takes one contiguous range of groups, whose walks visit
// nearby nodes through that XCD's L2.
__device__ inline int xcd_block(int b, int nb) {
  const int x = b % 8, i = b / 8, q = nb / 8, r = nb % 8;
  return x < r ? x * (q + 1) + i : r * (q + 1) + (x - r) * q + i;
}

// The host builder's walk (source.cpp:832-867) lists, for an opened node, its
// children in octant order 7..0 (singletons and accepted cells), then what
// its opened children list, octant 0 first.  The order of the lists is that
// of a depth-first walk, but which nodes are opened does not depend on it:
// k_bh_open (a wavefront per group) opens nodes breadth first, 8 queue entries
// (64 children) a step and every one of them kept, and k_bh_list (a block per
// group) sums what each entry's subtree lists and from it where its own
// particles and cells go.  A depth-first walk can keep only the work of the
// stack entries before the first one that opens children, and runs twice, the
// first time for the list lengths: 0.67 + 0.81 ms for 2^21 particles at
// theta = 0.5 (14029 groups that open 793 nodes on average), against 0.22 +
// 0.29 ms.  Bound: the vector cache, whose lookups and misses of the
// children's loads (64 lanes of 32 bytes a step) a step waits for.
//
// Leaves need no examining and go to the pool as they are found; the other
// entries wait for their turn in a ring in LDS (those beyond its kOpenRing
// places in their pool entry), so that a step's chain is one LDS read and the
// children's loads.
//
// Entries live in chunks of a pool, handed to the groups as they need them:
// {first child, masks, entry of the first opened child, 0}, masks: bits 0-7
// children, 8-15 those that are single particles, 16-23 accepted cells (the
// rest are opened); or a leaf.
constexpr int kOpenChunk = 256;        // entries per chunk
constexpr int kOpenGroupChunks = 256;  // per group at most: 16 bits of entry index
constexpr int kOpenRing = 512;         // queued entries in LDS per wavefront
constexpr int kOpenLevels = kLevels + 3;
constexpr int kRanOut = -1;  // for the number of levels: the pool or the table was too small

struct OpenPool {
  int4* rec;    // [chunks][kOpenChunk]
  int4* sum;    // the same: k_bh_list's working entries of groups too large for LDS
  int* wait;    // the same: the entry at a ring position beyond the ring
  // [0] != 0: some group ran out of pool or table (and is left to the depth-first
  // walk), [1] != 0: some group is too large for k_bh_list's LDS, then, a
  // cache line each, the chunks handed out of every part of the pool
  int* used;
  int* chunk;   // [group][width]
  int* level;   // [group][kOpenLevels]: first entry of each level, then the number of
                // entries; the last int is the number of levels (0: no entries, or kRanOut)
  int chunks;   // of each part
  int width;    // chunks of a group at most
};
// Parts of the pool with a counter of their own: a group begins with the part
// of its number and goes on to the next ones where that is used up.  The 57000
// chunks of a 2^21-particle build, taken from one counter, kept the walk
// waiting for that address: 627 us, with 64 counters 219.
constexpr int kPoolParts = 64;
constexpr int kPoolTries = 8;  // parts that a group asks
constexpr int kPoolLine = 32;  // ints
constexpr int kPoolUsed = (1 + kPoolParts) * kPoolLine;
// Chunks at most: 4 GiB of records, 1 GiB of queue and, where groups are too
// large for LDS, 4 GiB of working entries, which the cache keeps (to give such
// blocks back to the device and take them again costs 50 ms a GiB).
constexpr double kPoolMost = 1 << 20;

// Opened children, own particles and own cells of an entry.
__device__ inline int open_count(unsigned b) {
  return b & kLeafEntry ? 0 : __popc(b & 0xffu & ~(b >> 8) & ~(b >> 16));
}
__device__ inline int own_particles(unsigned b) {
  return b & kLeafEntry ? (int)(b & ~kLeafEntry) : __popc(b & 0xff00u);
}
__device__ inline int own_cells(unsigned b) {
  return b & kLeafEntry ? 0 : __popc(b & 0xff0000u);
}

constexpr int kListThreads = 256;
constexpr int kListEntries = 1536;  // entries of a group that k_bh_list holds in LDS

__global__ __launch_bounds__(64 * kWalkWaves) void k_bh_open(
    int ng, const int* __restrict__ gnode, Nodes nd, WalkNodes wn, double L,
    double th2, OpenPool pool, int* __restrict__ pcnt, int* __restrict__ ccnt) {
#pragma clang fp contract(off)
  __shared__ int s_chunk[kWalkWaves][kOpenGroupChunks];
  // {first child, mask | level << 8 | entry << 13}
  __shared__ int2 s_ring[kWalkWaves][kOpenRing];
  const int lane = threadIdx.x & 63;
  const int g = xcd_block(blockIdx.x, gridDim.x) * kWalkWaves + (threadIdx.x >> 6);
  if (g >= ng) return;  // uniform per wavefront
  int* chunk = s_chunk[threadIdx.x >> 6];
  int2* ring = s_ring[threadIdx.x >> 6];
  int* level = pool.level + (size_t)g * kOpenLevels;
  const int gk = gnode[g];
  const double gc[3] = {nd.c[3 * gk], nd.c[3 * gk + 1], nd.c[3 * gk + 2]};
  const double li = 0.5 * ldexp(L, -nd.lev[gk]);
  const WalkNode root = load_walk(wn, 0);
  // the whole tree as one cell (source.cpp:832-840): no entries
  if (bh_box_d2(gc, li, root.com) * th2 >= L * L) {
    if (lane == 0) {
      pcnt[g] = 0;
      ccnt[g] = 1;
      level[kOpenLevels - 1] = 0;
    }
    return;
  }
  int nch = 0;
  // one more chunk for this group; false: none left, or no room in its table
  auto grow = [&]() {
    int c = -1;
#pragma unroll 1  // unrolled, its registers cost the launch 257 us for 226
    for (int t = 0; t < kPoolTries && nch < pool.width && c < 0; ++t) {
      const int part = (g + t) % kPoolParts;
      int k = 0;
      if (lane == 0) k = atomicAdd(&pool.used[(1 + part) * kPoolLine], 1);
      k = __builtin_amdgcn_readfirstlane(k);
      if (k < pool.chunks) c = part * pool.chunks + k;
    }
    if (c < 0) return false;
    if (lane == 0) {
      chunk[nch] = c;
      pool.chunk[(size_t)g * pool.width + nch] = c;
    }
    ++nch;
    return true;
  };
  auto ran_out = [&]() {
    if (lane == 0) {
      pool.used[0] = 1;
      pcnt[g] = 0;
      ccnt[g] = 0;
      level[kOpenLevels - 1] = kRanOut;
    }
  };
  auto at = [&](int k) { return (size_t)chunk[k / kOpenChunk] * kOpenChunk + k % kOpenChunk; };
  // order LDS, or LDS and pool, writes before the reads of the wavefront's
  // other lanes
  auto lds_sync = [] {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  auto sync = [] {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  };
  if (!grow()) return ran_out();
  lds_sync();
  int np = 0, nc = 0;         // listed particles (leaves: this lane's) and cells
  int tail = 1;               // entries
  int head = 0, waiting = 1;  // ring positions: next to examine, end
  if (root.leaf()) {
    if (lane == 0) {
      np = root.count();
      pool.rec[at(0)] = make_int4(root.x, (int)root.y, 0, 0);
    }
    waiting = 0;
  } else if (lane == 0) {
    ring[0] = make_int2(root.x, (int)root.y);
  }
  // next = ring position of the first entry of the newest level
  int nlev = 1, next = 0;
  if (lane == 0) level[0] = 0;
  const int e = lane >> 3, o = lane & 7;
  while (head < waiting) {
    lds_sync();
    const int npop = min(8, waiting - head);
    const bool valid = e < npop;
    const int2 r = valid ? ring[(head + e) % kOpenRing] : make_int2(0, 0);
    const unsigned b = (unsigned)r.y;
    int kind = 0;  // 1 particle, 2 cell, 3 opened
    WalkNode w{0, 0u, {0.0, 0.0, 0.0}};
    const int lev = (int)(b >> 8 & 31u);
    if ((b >> o) & 1u) {
      const double l = ldexp(L, -lev);
      const double s2 = 0.25 * l * l;  // child side squared
      w = load_walk(wn, r.x + __popc(b & ((1u << o) - 1u)));
      if (w.y == (kLeafEntry | 1u))
        kind = 1;
      else if (bh_box_d2(gc, li, w.com) * th2 > s2)
        kind = 2;
      else
        kind = 3;
    }
    const bool inner = kind == 3 && !w.leaf();
    const u64 mp = __ballot(kind == 1), mc = __ballot(kind == 2), ms = __ballot(kind == 3);
    const u64 mi = __ballot(inner);
    const u64 below = (1ULL << lane) - 1ULL;
    const int opened = __popcll(ms);
    while ((tail + opened - 1) / kOpenChunk >= nch) {
      if (!grow()) return ran_out();
      lds_sync();
    }
    head += npop;
    if (kind == 1) ++np;
    if (kind == 2) ++nc;
    if (kind == 3) {
      const int k = tail + __popcll(ms & below);
      if (inner) {
        const int q = waiting + __popcll(mi & below);
        const int2 v = make_int2(w.x, (int)w.y | (lev + 1) << 8 | k << 13);
        if (q < head + kOpenRing) {
          ring[q % kOpenRing] = v;
        } else {
          pool.rec[at(k)] = make_int4(v.x, v.y, 0, 0);
          pool.wait[at(q)] = k;
        }
      } else {
        pool.rec[at(k)] = make_int4(w.x, (int)w.y, 0, 0);
        np += w.count();
      }
    }
    // places freed by this step, for entries that have waited in the pool
    if (waiting > head - npop + kOpenRing) {
      sync();
      const int q = head - npop + kOpenRing + lane;
      if (lane < npop && q < waiting) {
        const int4 v = pool.rec[at(pool.wait[at(q)])];
        ring[q % kOpenRing] = make_int2(v.x, v.y);
      }
    }
    if (valid && o == 0) {
      const unsigned m1 = (unsigned)(mp >> (8 * e)) & 0xffu, m2 = (unsigned)(mc >> (8 * e)) & 0xffu;
      pool.rec[at((int)(b >> 13))] = make_int4(r.x, (int)((b & 0xffu) | m1 << 8 | m2 << 16),
                                               tail + __popcll(ms & below), 0);
    }
    // a level's entries start where the first entry examined of the level
    // before put its opened children
    if (next < head) {
      const u64 before = (1ULL << (8 * (next - head + npop))) - 1ULL;
      if (lane == 0) level[nlev] = tail + __popcll(ms & before);
      ++nlev;
      next = waiting + __popcll(mi & before);
    }
    waiting += __popcll(mi);
    tail += opened;
  }
  for (int d = 32; d > 0; d >>= 1) {
    np += __shfl_xor(np, d);
    nc += __shfl_xor(nc, d);
  }
  if (lane == 0) {
    level[nlev] = tail;  // (the deepest level may have no entries)
    level[kOpenLevels - 1] = nlev;
    pcnt[g] = np;
    ccnt[g] = nc;
    if (tail > kListEntries) pool.used[1] = 1;
  }
}

// The lists of k_bh_open's groups, one block each: the entries of a level
// after the other, first deepest to root for what each entry's subtree lists,
// then root to deepest for where each entry's particles and cells go, then
// the lists, eight lanes per entry.  The working entries {masks, first opened
// child, particles, cells} are in LDS, or (BIG) for groups of more than
// kListEntries in the pool.
template <bool BIG>
__global__ __launch_bounds__(kListThreads) void k_bh_list(
    int ng, OpenPool pool, const int* __restrict__ item, const int* __restrict__ poff,
    const int* __restrict__ coff, int* __restrict__ plist, int* __restrict__ clist) {
  __shared__ int4 s_ent[BIG ? 1 : kListEntries];
  __shared__ int s_x[BIG ? 1 : kListEntries];  // first child or particle
  __shared__ int s_chunk[kOpenGroupChunks], s_level[kOpenLevels];
  const int g = xcd_block(blockIdx.x, gridDim.x);
  const int tid = threadIdx.x;
  if (tid < kOpenLevels) s_level[tid] = pool.level[(size_t)g * kOpenLevels + tid];
  static_assert(kOpenGroupChunks <= kListThreads, "one chunk per thread");
  if (tid < pool.width) s_chunk[tid] = pool.chunk[(size_t)g * pool.width + tid];
  __syncthreads();
  const int nlev = s_level[kOpenLevels - 1];
  if (nlev <= 0) return;  // uniform
  const int n = s_level[nlev];
  if (BIG != (n > kListEntries)) return;  // uniform
  auto at = [&](int k) { return (size_t)s_chunk[k / kOpenChunk] * kOpenChunk + k % kOpenChunk; };
  auto ent = [&](int k) -> int4& { return BIG ? pool.sum[at(k)] : s_ent[k]; };
  for (int k = tid; k < n; k += kListThreads) {
    const int4 r = pool.rec[at(k)];
    const unsigned b = (unsigned)r.y;
    ent(k) = make_int4(r.y, r.z, own_particles(b), own_cells(b));
    if (!BIG) s_x[k] = r.x;
  }
  __syncthreads();
  for (int v = nlev - 1; v >= 0; --v) {
    for (int k = s_level[v] + tid; k < s_level[v + 1]; k += kListThreads) {
      int4 r = ent(k);
      const int m = open_count((unsigned)r.x);
      for (int c = 0; c < m; ++c) {
        const int4 t = ent(r.y + c);
        r.z += t.z;
        r.w += t.w;
      }
      if (m) ent(k) = r;
    }
    __syncthreads();
  }
  if (tid == 0) {
    int4& r = ent(0);
    r.z = 0;
    r.w = 0;
  }
  __syncthreads();
  for (int v = 0; v < nlev; ++v) {
    for (int k = s_level[v] + tid; k < s_level[v + 1]; k += kListThreads) {
      const int4 r = ent(k);
      const unsigned b = (unsigned)r.x;
      const int m = open_count(b);
      int np = r.z + own_particles(b), nc = r.w + own_cells(b);
      for (int c = 0; c < m; ++c) {
        int4& t = ent(r.y + c);
        const int tp = t.z, tc = t.w;
        t.z = np;
        t.w = nc;
        np += tp;
        nc += tc;
      }
    }
    __syncthreads();
  }
  int* pl = plist + poff[g];
  int* cl = clist + coff[g];
  const int o = tid & 7;
  const unsigned above = 0xffu & ~((2u << o) - 1u);  // octants listed before this one
  for (int k0 = tid >> 3; k0 < n; k0 += 4 * (kListThreads / 8)) {
    int4 r[4];
    int x[4], w[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {  // four entries' loads in flight
      const int k = k0 + u * (kListThreads / 8);
      r[u] = k < n ? ent(k) : make_int4(0, 0, 0, 0);
      x[u] = k < n ? (BIG ? pool.rec[at(k)].x : s_x[k]) : 0;
      const unsigned b = (unsigned)r[u].x;
      if (!(b & kLeafEntry) && (((b >> 8 | b >> 16) >> o) & 1u))
        w[u] = item[x[u] + __popc(b & ((1u << o) - 1u))];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const unsigned b = (unsigned)r[u].x, m1 = b >> 8 & 0xffu, m2 = b >> 16 & 0xffu;
      if (b & kLeafEntry) {
        const int cnt = (int)(b & ~kLeafEntry);
        for (int p = o; p < cnt; p += 8) pl[r[u].z + p] = x[u] + p;
      } else if ((m1 >> o) & 1u) {
        pl[r[u].z + __popc(m1 & above)] = w[u];
      } else if ((m2 >> o) & 1u) {
        cl[r[u].w + __popc(m2 & above)] = w[u];
      }
    }
  }
}

// Lists of one cell, the whole tree (groups that k_bh_open gave no entries).
__global__ void k_bh_whole(int ng, const int* __restrict__ pcnt, const int* __restrict__ ccnt,
                           WalkNodes wn, const int* __restrict__ coff,
                           const int* __restrict__ gnode, Nodes nd, double L, double th2,
                           int* __restrict__ clist) {
#pragma clang fp contract(off)
  const int g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= ng || pcnt[g] != 0 || ccnt[g] != 1) return;
  const int gk = gnode[g];
  const double gc[3] = {nd.c[3 * gk], nd.c[3 * gk + 1], nd.c[3 * gk + 2]};
  if (bh_box_d2(gc, 0.5 * ldexp(L, -nd.lev[gk]), load_walk(wn, 0).com) * th2 >= L * L)
    clist[coff[g]] = nd.cell[0];
}

// For the groups that open more nodes than k_bh_open's pool or their table has
// left (level: of the pool), or for all of a build without a pool (level null).
//
// One wavefront per group: the depth-first walk of the host builder
// (source.cpp:832-867 order: the children of an opened node are examined in
// octant order 7..0, emitting singletons and accepted cells in that order and
// pushing the rest, so octant 0 is expanded first), counting (FILL == false)
// or writing the particle and cell lists.  Each step examines the children
// of the top 8 stack entries at once, one lane per (entry, octant), and keeps
// the work of the entries the serial walk would finish before the first one
// that pushes children: a run of entries whose children are all listed,
// ending at one that opens some, so the lists and the stack come out exactly
// as in the serial walk.  Ballots rank the emissions and pushes in the serial
// order.  A pushed entry holds what its expansion needs (the node's children
// and level, or the particle range of a leaf), so a step costs one round of
// global loads: the children's records.
template <bool FILL>
__global__ __launch_bounds__(64 * kWalkWaves) void k_bh_walk(
    int ng, const int* __restrict__ gnode, Nodes nd, WalkNodes wn, double L,
    double th2, const int* __restrict__ level, int* __restrict__ pcnt, int* __restrict__ ccnt,
    const int* __restrict__ poff, const int* __restrict__ coff, int* __restrict__ plist,
    int* __restrict__ clist) {
#pragma clang fp contract(off)
  // entry: {first child, octant mask, level} of a node to expand, or
  // {lo, hi, -1} of a leaf whose particles are listed
  __shared__ int3 s_stack[kWalkWaves][kWalkDepth];
  const int lane = threadIdx.x & 63;
  const int g = xcd_block(blockIdx.x, gridDim.x) * kWalkWaves + (threadIdx.x >> 6);
  if (g >= ng) return;  // uniform per wavefront
  if (level && level[(size_t)g * kOpenLevels + kOpenLevels - 1] != kRanOut) return;  // the same
  int3* stk = s_stack[threadIdx.x >> 6];
  const int gk = gnode[g];
  const double gc[3] = {nd.c[3 * gk], nd.c[3 * gk + 1], nd.c[3 * gk + 2]};
  const double li = 0.5 * ldexp(L, -nd.lev[gk]);
  int np = 0, nc = 0;
  int* pl = FILL ? plist + poff[g] : nullptr;
  int* cl = FILL ? clist + coff[g] : nullptr;
  const WalkNode root = load_walk(wn, 0);
  // the whole tree as one cell (source.cpp:832-840)
  if (bh_box_d2(gc, li, root.com) * th2 >= L * L) {
    if (FILL && lane == 0) cl[0] = nd.cell[0];
    nc = 1;
  } else {
    if (lane == 0)
      stk[0] = root.leaf() ? make_int3(root.x, root.x + root.count(), -1)
                           : make_int3(root.x, (int)root.y, 0);
    int sp = 1;
    while (sp > 0) {
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      // lanes 8e..8e+7 take entry e from the top (e = 0 is the top), octant
      // o = lane % 8 of it
      const int npop = sp < 8 ? sp : 8;
      const int e = lane >> 3, o = lane & 7;
      int3 ent = make_int3(0, 0, 0);
      if (e < npop) ent = stk[sp - 1 - e];
      const bool leaf = e < npop && ent.z < 0;
      int kind = 0;  // 1 particle, 2 cell, 3 push
      int lo = 0, cell = 0;
      WalkNode w{0, 0u, {0.0, 0.0, 0.0}};
      if (e < npop && !leaf && ((ent.y >> o) & 1)) {
        const double l = ldexp(L, -ent.z);
        const double s2 = 0.25 * l * l;  // child side squared
        const int k = ent.x + __popc(ent.y & ((1 << o) - 1));
        w = load_walk(wn, k);
        if (w.y == (kLeafEntry | 1u))
          kind = 1;
        else if (bh_box_d2(gc, li, w.com) * th2 > s2)
          kind = 2;
        else
          kind = 3;
        if (FILL) {
          lo = cell = wn.item[k];
        }
      }
      // The serial walk would expand the entries from the top until one
      // pushes children; those entries (ncommit of them) are done here, the
      // rest stay on the stack.
      const u64 ms = __ballot(kind == 3);
      const int ncommit = ms ? (__builtin_ctzll(ms) >> 3) + 1 : npop;
      const bool commit = e < ncommit;
      const u64 mp = __ballot(commit && kind == 1), mc = __ballot(commit && kind == 2);
      const u64 mine = 0xffULL << (8 * e);           // this entry's lanes
      const u64 before = (1ULL << (8 * e)) - 1ULL;   // entries above this one
      const u64 above = ~((2ULL << lane) - 1ULL);    // lanes > this one
      // emission order: entries from the top; octants 7..0 inside an entry;
      // a leaf entry lists its particles lo..hi-1
      const int leafcnt = commit && leaf && o == 0 ? ent.y - ent.x : 0;
      int leafpre = 0, leaftot = 0;
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const int c = __builtin_amdgcn_readlane(leafcnt, 8 * q);
        leafpre += q < e ? c : 0;
        leaftot += c;
      }
      const int pbase = np + leafpre + __popcll(mp & before);
      if (FILL && commit && kind == 1) pl[pbase + __popcll(mp & mine & above)] = lo;
      if (FILL && commit && leaf)
        for (int p = ent.x + o; p < ent.y; p += 8) pl[pbase + (p - ent.x)] = p;
      if (FILL && commit && kind == 2) cl[nc + __popcll(mc & (before | (mine & above)))] = cell;
      const u64 mpush = ms & (0xffULL << (8 * (ncommit - 1)));  // the last committed entry
      sp -= ncommit;
      if (kind == 3 && commit)
        stk[sp + __popcll(mpush & above)] = w.leaf() ? make_int3(w.x, w.x + w.count(), -1)
                                                     : make_int3(w.x, (int)w.y, ent.z + 1);
      np += __popcll(mp) + leaftot;
      nc += __popcll(mc);
      sp += __popcll(mpush);
    }
  }
  if (!FILL && lane == 0) {
    pcnt[g] = np;
    ccnt[g] = nc;
  }
}

// ------------------------------------------------------------ common tail
// Clears coff[ng + 1] and ccnt[ng] (null: neither) and the two sums of k_cost.
__global__ void k_clear(int ng, int* __restrict__ coff, int* __restrict__ ccnt,
                        unsigned long long* __restrict__ work) {
  const int g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g < 2) work[g] = 0;
  if (coff && g <= ng) coff[g] = 0;
  if (ccnt && g < ng) ccnt[g] = 0;
}

// cost key: groups by decreasing icnt * (jcnt + 2 ccnt), ties by index.  idx:
// the groups (to be sorted), or their ranks cleared.
__global__ void k_cost(int ng, const int* __restrict__ icnt, const int* __restrict__ jcnt,
                       const int* __restrict__ ccnt, u64* __restrict__ key, int* __restrict__ idx,
                       bool by_rank, unsigned long long* __restrict__ work) {
  const int g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= ng) return;
  const long long c = (long long)icnt[g] * (jcnt[g] + (ccnt ? 2 * ccnt[g] : 0));
  key[g] = (u64)(LLONG_MAX - c);
  idx[g] = by_rank ? 0 : g;
  atomicAdd(&work[0], (unsigned long long)((long long)icnt[g] * jcnt[g]));
  if (ccnt) atomicAdd(&work[1], (unsigned long long)((long long)icnt[g] * ccnt[g]));
}

// order[] of k_cost's keys for up to kRankGroups groups: rank[g] (0 before)
// gains the groups of one tile that come before g, then order[rank[g]] = g.
// Every pair is compared, 14029 groups in 25 us; the library's sort of the
// 64-bit keys took 61.
constexpr int kRankGroups = 1 << 14;
__global__ __launch_bounds__(256) void k_rank(int ng, const u64* __restrict__ key,
                                              int* __restrict__ rank) {
  __shared__ u64 s[256];
  const int h0 = blockIdx.y * 256, g = blockIdx.x * 256 + threadIdx.x;
  if (h0 + (int)threadIdx.x < ng) s[threadIdx.x] = key[h0 + threadIdx.x];
  __syncthreads();
  if (g >= ng) return;
  const u64 own = key[g];
  const int n = min(256, ng - h0);
  int r = 0;
  if (blockIdx.y == blockIdx.x) {
    for (int h = 0; h < n; ++h) r += s[h] < own || (s[h] == own && h0 + h < g);
  } else {
    // a tie goes to the lower index; keys are below 2^63
    const u64 end = own + (blockIdx.y < blockIdx.x);
#pragma unroll 8
    for (int h = 0; h < n; ++h) r += s[h] < end;
  }
  if (r) atomicAdd(&rank[g], r);
}

__global__ void k_rank_order(int ng, const int* __restrict__ rank, int* __restrict__ order) {
  const int g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g < ng) order[rank[g]] = g;
}

__global__ void k_pack(int np, const double* __restrict__ pos, const int* __restrict__ src,
                       const double* __restrict__ mass, float scale, float4* __restrict__ out) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= np) return;
  float4 v;
  v.x = (float)pos[3 * p] * scale;
  v.y = (float)pos[3 * p + 1] * scale;
  v.z = (float)pos[3 * p + 2] * scale;
  v.w = (float)mass[src[p]];
  out[p] = v;
}

__global__ void k_pack_cells(int nc, const double* __restrict__ cells, float* __restrict__ out) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= nc) return;
  for (int t = 0; t < 10; ++t) out[12 * (size_t)c + t] = (float)cells[10 * (size_t)c + t];
  out[12 * (size_t)c + 10] = 0.f;
  out[12 * (size_t)c + 11] = 0.f;
}

// ------------------------------------------------------------ host drivers
struct Octree {
  Nodes nd{};
  int nn = 0;
  LevelStarts level;  // level l occupies [v[l], v[l + 1])
};

// Sorted keys, particles in Morton order and the octree.  m may be null.
void build_octree(Build& B, Lists& R, int n, const double* x, const double* m,
                  const double lo[3], double L, int split, Octree& T, u64** skey_out,
                  double** mm_out) {
  hipStream_t st = B.st;
  split = std::min(split, n);  // no cell holds more than n: the root is not split
  u64* key = B.tmp.get<u64>(n);
  const double s = (double)(1 << kLevels) / L;
  double* mm = m ? B.tmp.get<double>(n) : nullptr;
  unsigned char* leaf = B.tmp.get<unsigned char>(n);
  unsigned char* leaf2 = split > kMaxWindow ? B.tmp.get<unsigned char>(n) : nullptr;
  const int nb = (int)grid_for(n, kTreeBlock).x;
  int* count = B.tmp.get<int>((size_t)kTreeLevels * nb);
  int* first = B.tmp.get<int>((size_t)kTreeLevels * nb + 1);
  int* long_run = B.tmp.get<int>(1);
  u64* skey = nullptr;
  for (int bits = kFirstBits;; bits = 3 * kLevels) {
    hipLaunchKernelGGL(k_keys, grid_for(n), dim3(256), 0, st, n, x, lo[0], lo[1], lo[2], s, key,
                       long_run);
    PGAMD_HIP_CHECK(hipGetLastError());
    int* perm = nullptr;
    B.sort_keys(key, n, 3 * kLevels, bits, &skey, &perm, long_run);
    hipLaunchKernelGGL(k_gather, grid_for(n), dim3(256), 0, st, n, perm, x, m, R.pos, mm, R.src);
    // leaf level of every particle: the sliding maximum over split + 1 places (all
    // are 0 where split = n)
    int w = std::min(split, kMaxWindow) + 1;
    hipLaunchKernelGGL(k_window_max, grid_for(n, kWindowOut), dim3(256), 0, st, n, split, w, skey,
                       leaf);
    for (int h; split < n && w < split + 1; w += h) {
      h = std::min(w, split + 1 - w);
      hipLaunchKernelGGL(k_window_grow, grid_for(n), dim3(256), 0, st, n, h, leaf, leaf2);
      std::swap(leaf, leaf2);
    }
    hipLaunchKernelGGL(k_tree_count, dim3(nb), dim3(256), 0, st, n, skey, leaf, count);
    PGAMD_HIP_CHECK(hipGetLastError());
    B.scan(count, first, kTreeLevels * nb, -1);
    hipLaunchKernelGGL(k_tree_levels, dim3(1), dim3(64), 0, st, nb, first, long_run,
                       host_dev(host_ints()) + kSlotLevels);
    PGAMD_HIP_CHECK(hipGetLastError());
    const volatile int* host = B.wait() + kSlotLevels;
    for (int l = 0; l < kLevels + 2; ++l) T.level.v[l] = host[l];
    if (host[kTreeLevels + 1] == 0) break;  // no long run
  }
  T.nn = T.level.v[kLevels + 1];
  Nodes& nd = T.nd;
  const size_t c = (size_t)T.nn;
  nd.lo = B.tmp.get<int>(c);
  nd.hi = B.tmp.get<int>(c);
  nd.par = B.tmp.get<int>(c);
  nd.lev = B.tmp.get<int>(c);
  nd.child = B.tmp.get<int>(8 * c);
  nd.c = B.tmp.get<double>(3 * c);
  nd.com = B.tmp.get<double>(3 * c);
  nd.m = B.tmp.get<double>(c);
  nd.q = B.tmp.get<double>(6 * c);
  nd.cell = B.tmp.get<int>(c);
  hipLaunchKernelGGL(k_fill_int4, grid_for(2 * c), dim3(256), 0, st, 2 * c, -1,
                     reinterpret_cast<int4*>(nd.child));
  hipLaunchKernelGGL(k_tree_fill, dim3(nb), dim3(256), 0, st, n, skey, leaf, first, nd);
  hipLaunchKernelGGL(k_tree_nodes, grid_for(T.nn), dim3(256), 0, st, T.nn, n, skey, L,
                     lo[0] + 0.5 * L, lo[1] + 0.5 * L, lo[2] + 0.5 * L, nd);
  PGAMD_HIP_CHECK(hipGetLastError());
  *skey_out = skey;
  *mm_out = mm;
}

// Groups of the octree sorted by first particle; fills ioff/icnt/ilist.
// flag_groups queues their count (kSlotTotal), build_groups runs after a
// wait().
struct GroupFlags {
  int *flag, *off;
};
GroupFlags flag_groups(Build& B, const Octree& T, int ncrit) {
  const int nn = T.nn;
  const GroupFlags f{B.tmp.get<int>(nn), B.tmp.get<int>(nn + 1)};
  hipLaunchKernelGGL(k_group_flag, grid_for(nn), dim3(256), 0, B.st, nn, T.nd, ncrit, f.flag);
  PGAMD_HIP_CHECK(hipGetLastError());
  B.scan(f.flag, f.off, nn, kSlotTotal);
  return f;
}

int build_groups(Build& B, Lists& R, int n, const Octree& T, const GroupFlags& f,
                 int** gnode_out) {
  hipStream_t st = B.st;
  const int nn = T.nn;
  const int *flag = f.flag, *off = f.off;
  const int ng = host_ints()[kSlotTotal];
  int* gn = B.tmp.get<int>(ng);
  int* gn_sorted = B.tmp.get<int>(ng);
  hipLaunchKernelGGL(k_compact, grid_for(nn), dim3(256), 0, st, nn, flag, off, gn);
  hipLaunchKernelGGL(k_group_order, grid_for(ng, 8), dim3(256), 0, st, ng, gn, off, T.level, T.nd,
                     gn_sorted);
  PGAMD_HIP_CHECK(hipGetLastError());
  R.ng = ng;
  R.icnt = R.mem.get<int>(ng);
  R.ioff = R.mem.get<int>(ng + 1);
  hipLaunchKernelGGL(k_group_icnt, grid_for(ng), dim3(256), 0, st, ng, gn_sorted, T.nd, R.icnt);
  PGAMD_HIP_CHECK(hipGetLastError());
  B.scan(R.icnt, R.ioff, ng, -1);
  R.ni = n;  // every particle is in one group
  R.ilist = R.mem.get<int>(R.ni);
  if (ng > 0)
    hipLaunchKernelGGL(k_group_ilist, dim3(ng), dim3(256), 0, st, ng, gn_sorted, T.nd, R.ioff,
                       R.ilist);
  PGAMD_HIP_CHECK(hipGetLastError());
  *gnode_out = gn_sorted;
  return ng;
}

void finish(Build& B, Lists& R, bool cells) {
  hipStream_t st = B.st;
  const int ng = (int)R.ng;
  u64* key = B.tmp.get<u64>(ng);
  int* idx = B.tmp.get<int>(ng);
  unsigned long long* work = B.tmp.get<unsigned long long>(2);
  hipLaunchKernelGGL(k_clear, grid_for(cells ? 1 : ng + 1), dim3(256), 0, st, ng,
                     cells ? nullptr : R.coff, cells ? nullptr : R.ccnt, work);
  R.order = R.mem.get<int>(ng);
  hipLaunchKernelGGL(k_cost, grid_for(ng), dim3(256), 0, st, ng, R.icnt, R.jcnt,
                     cells ? R.ccnt : nullptr, key, idx, ng <= kRankGroups, work);
  if (ng <= kRankGroups) {
    hipLaunchKernelGGL(k_rank, dim3(grid_for(ng).x, grid_for(ng).x), dim3(256), 0, st, ng, key,
                       idx);
    hipLaunchKernelGGL(k_rank_order, grid_for(ng), dim3(256), 0, st, ng, idx, R.order);
  } else {
    u64* skey = B.tmp.get<u64>(ng);
    B.sort_pairs(key, skey, idx, R.order, ng, 64);
  }
  hipLaunchKernelGGL(k_copy_ints, dim3(1), dim3(64), 0, st, 4, reinterpret_cast<int*>(work),
                     host_dev(host_ints()) + kSlotWork);
  PGAMD_HIP_CHECK(hipGetLastError());
  unsigned long long w[2];
  const volatile int* h = B.wait() + kSlotWork;
  for (int k = 0; k < 2; ++k)
    w[k] = (unsigned)h[2 * k] | (unsigned long long)(unsigned)h[2 * k + 1] << 32;
  R.work_pp = (long long)w[0];
  R.work_pc = cells ? (long long)w[1] : 0;
}

Lists* treepm_build(int n, const double* x, double rcut, int ncrit, hipStream_t st) {
  Lists* R = new Lists();
  Build B(st);
  // positions: originals then ghosts (at most 7 per particle)
  double* pos_all = R->mem.get<double>(3 * (size_t)n * 8);
  int* src_all = R->mem.get<int>((size_t)n * 8);
  R->pos = pos_all;
  R->src = src_all;
  Octree T;
  u64* skey = nullptr;
  double* mm = nullptr;
  const double lo[3] = {0, 0, 0};
  build_octree(B, *R, n, x, nullptr, lo, 1.0, std::max(1, ncrit), T, &skey, &mm);
  const GroupFlags gf = flag_groups(B, T, ncrit);
  // ghosts
  const int gblocks = (int)grid_for(n, kGhostBlock).x;
  int* gcnt = B.tmp.get<int>(gblocks);
  int* goff = B.tmp.get<int>(gblocks + 1);
  hipLaunchKernelGGL(k_ghost_count, dim3(gblocks), dim3(256), 0, st, n, R->pos, rcut, gcnt);
  PGAMD_HIP_CHECK(hipGetLastError());
  B.scan(gcnt, goff, gblocks, kSlotTotal2);
  hipLaunchKernelGGL(k_ghost_fill, dim3(gblocks), dim3(256), 0, st, n, goff, rcut, R->pos, R->src);
  PGAMD_HIP_CHECK(hipGetLastError());
  const int nghost = B.wait()[kSlotTotal2];
  int* gnode = nullptr;
  const int ng = build_groups(B, *R, n, T, gf, &gnode);
  const int np = n + nghost;
  R->np = np;
  // grid over [-rcut, 1 + rcut) with cells of side >= rcut
  Grid gr;
  gr.glo = -rcut;
  const double gL = 1.0 + 2 * rcut;
  gr.nc = std::max(1, (int)std::floor(gL / rcut));
  gr.h = gL / gr.nc;
  const int ncell = gr.nc * gr.nc * gr.nc;
  unsigned* cell = B.tmp.get<unsigned>(np);
  unsigned* scell = nullptr;
  int* cpart = nullptr;
  int* cstart = B.tmp.get<int>(ncell + 1);
  hipLaunchKernelGGL(k_cell_of, grid_for(np), dim3(256), 0, st, np, R->pos, gr, cell);
  PGAMD_HIP_CHECK(hipGetLastError());
  const int cell_bits = bits_for(ncell);
  B.sort_keys(cell, np, cell_bits, cell_bits, &scell, &cpart, nullptr);
  hipLaunchKernelGGL(k_cell_start, grid_for(ncell + 1), dim3(256), 0, st, ncell, np, scell,
                     cstart);
  PGAMD_HIP_CHECK(hipGetLastError());
  // j-lists: count, offsets, fill (cell order)
  double* box = B.tmp.get<double>(6 * (size_t)std::max(ng, 1));
  hipLaunchKernelGGL(k_group_box, grid_for(ng, 4), dim3(256), 0, st, ng, gnode, T.nd, R->pos, box);
  R->jcnt = R->mem.get<int>(ng);
  R->joff = R->mem.get<int>(ng + 1);
  float4* cpos = B.tmp.get<float4>(np);
  int* wide = B.tmp.get<int>(1);
  hipLaunchKernelGGL(k_fill_int, dim3(1), dim3(64), 0, st, 1, 0, wide);
  hipLaunchKernelGGL(k_cell_pos, grid_for(np), dim3(256), 0, st, np, cpart, R->pos, cpos, wide);
  // One walk: each group writes its list at its candidate offset (the
  // candidate count bounds the list length), then the lists are packed.
  int* ccand = B.tmp.get<int>(ng);
  int* soff = B.tmp.get<int>(ng + 1);
  hipLaunchKernelGGL(k_treepm_cand, grid_for(ng, 4), dim3(256), 0, st, ng, box, gr, cstart, rcut,
                     ccand);
  PGAMD_HIP_CHECK(hipGetLastError());
  B.scan(ccand, soff, ng, kSlotTotal);
  const int ncand = B.wait()[kSlotTotal];
  int* scratch = B.tmp.get<int>(std::max(ncand, 1));
  hipLaunchKernelGGL(k_treepm_jlist, grid_for(ng, 4), dim3(256), 0, st, ng, box, cpos,
                     gr, cstart, R->pos, wide, fine_reach(rcut), rcut, R->jcnt, soff, scratch);
  PGAMD_HIP_CHECK(hipGetLastError());
  B.scan(R->jcnt, R->joff, ng, kSlotTotal);
  R->nj = B.wait()[kSlotTotal];
  R->jlist = R->mem.get<int>(R->nj);
  hipLaunchKernelGGL(k_pack_lists, grid_for(ng, 4), dim3(256), 0, st, ng, soff, R->jcnt, R->joff,
                     scratch, R->jlist);
  PGAMD_HIP_CHECK(hipGetLastError());
  R->coff = R->mem.get<int>(ng + 1);
  R->ccnt = R->mem.get<int>(ng);
  R->clist = R->mem.get<int>(1);
  R->cells = R->mem.get<double>(10);
  finish(B, *R, false);
  return R;
}

// The pool of a build of ng groups over nn nodes; rec is null where the
// depth-first walk is to do it alone.
//
// Opened nodes of a group on average (halo of 2^21 particles, groups of up to 512,
// leaves of 8): 793 at theta = 0.5, 2206 at 0.3, 5858 at 0.2, 8666 at 0.17, about
// theta^-2.25; in groups of up to 16 444 at 0.5.  The pool has room for 1280 (768)
// of them and as much more for smaller theta, and a group for 16384 or 65536.
// Where most groups would open more than that the walk takes all of them.
OpenPool open_pool(Build& B, int ng, int nn, double theta, int ncrit) {
  OpenPool p{};
  const double all = std::ceil(nn / (double)kOpenChunk);  // chunks of all nodes
  const double each =
      std::min(all, (ncrit < 128 ? 3.0 : 5.0) * std::max(1.0, std::pow(0.5 / theta, 2.25)));
  if (each > kOpenGroupChunks) return p;
  p.width = each > 40 ? kOpenGroupChunks : 64;
  // a power of two, as the cache's blocks; a group's table can be filled from the
  // parts it asks
  size_t chunks = (size_t)kPoolParts / kPoolTries * p.width;
  while (chunks < std::min(64 + ng * each, kPoolMost)) chunks *= 2;
  p.chunks = (int)(chunks / kPoolParts);
  p.rec = B.pool.try_get<int4>(chunks * kOpenChunk);
  p.wait = B.pool.try_get<int>(chunks * kOpenChunk);
  p.chunk = B.pool.try_get<int>((size_t)ng * p.width);
  p.level = B.pool.try_get<int>((size_t)ng * kOpenLevels);
  p.used = B.pool.try_get<int>(kPoolUsed);
  if (!p.rec || !p.wait || !p.chunk || !p.level || !p.used) {
    B.pool.free_all();
    p.rec = nullptr;
  }
  return p;
}

Lists* bh_build(int n, const double* x, const double* m, double theta, int ncrit, int nleaf,
                hipStream_t st) {
  Lists* R = new Lists();
  Build B(st);
  // bounding box -> cube side, as the host builder
  const int nb = 256;
  double* part = B.tmp.get<double>(6 * nb);
  hipLaunchKernelGGL(k_bbox_part, dim3(nb), dim3(256), 0, st, n, x, part);
  hipLaunchKernelGGL(k_bbox_final, dim3(1), dim3(64), 0, st, nb, part,
                     reinterpret_cast<double*>(host_dev(host_ints()) + kSlotBox));
  PGAMD_HIP_CHECK(hipGetLastError());
  double h[6];
  const volatile double* box = reinterpret_cast<const volatile double*>(B.wait() + kSlotBox);
  for (int k = 0; k < 6; ++k) h[k] = box[k];
  const double lo[3] = {h[0], h[1], h[2]};
  double L = 0;
  for (int d = 0; d < 3; ++d) L = std::max(L, h[3 + d] - h[d]);
  L *= 1.0 + 1e-9;
  R->pos = R->mem.get<double>(3 * (size_t)n);
  R->src = R->mem.get<int>(n);
  R->np = n;
  Octree T;
  u64* skey = nullptr;
  double* mm = nullptr;
  build_octree(B, *R, n, x, m, lo, L, std::max(1, std::min(ncrit, nleaf)), T, &skey, &mm);
  // moments: all leaves at once, then the inner nodes, deepest level first
  // (2^21 particles: 54 + 103 + 29 us; 16 launches over whole levels took 240)
  hipLaunchKernelGGL(k_leaf_moments, grid_for(T.nn), dim3(256), 0, st, T.nn, T.nd, R->pos, mm);
  int top = 0;
  while (top <= kLevels && T.level.v[top + 1] - T.level.v[top] <= kTopNodes) ++top;
  for (int lev = kLevels; lev >= top; --lev) {
    const int a = T.level.v[lev], b = T.level.v[lev + 1];
    if (b > a)
      hipLaunchKernelGGL(k_inner_moments, grid_for(b - a, 64), dim3(64), 0, st, a, b, T.nd);
  }
  hipLaunchKernelGGL(k_top_moments, dim3(1), dim3(kTopNodes), 0, st, top, T.level, T.nd);
  PGAMD_HIP_CHECK(hipGetLastError());
  // cells: nodes with more than one particle, in node order
  int* flag = B.tmp.get<int>(T.nn);
  int* off = B.tmp.get<int>(T.nn + 1);
  hipLaunchKernelGGL(k_cell_flag, grid_for(T.nn), dim3(256), 0, st, T.nn, T.nd, flag);
  PGAMD_HIP_CHECK(hipGetLastError());
  B.scan(flag, off, T.nn, kSlotTotal2);
  const GroupFlags gf = flag_groups(B, T, ncrit);
  R->ncells = B.wait()[kSlotTotal2];
  R->cells = R->mem.get<double>(10 * (size_t)R->ncells);
  hipLaunchKernelGGL(k_cell_fill, grid_for(T.nn), dim3(256), 0, st, T.nn, T.nd, flag, off,
                     R->cells);
  PGAMD_HIP_CHECK(hipGetLastError());
  int* gnode = nullptr;
  const int ng = build_groups(B, *R, n, T, gf, &gnode);
  const double th2 = theta * theta;
  R->jcnt = R->mem.get<int>(ng);
  R->joff = R->mem.get<int>(ng + 1);
  R->ccnt = R->mem.get<int>(ng);
  R->coff = R->mem.get<int>(ng + 1);
  WalkNodes wn;
  wn.item = B.tmp.get<int>(T.nn);
  wn.ex = B.tmp.get<int4>(T.nn);
  wn.yz = B.tmp.get<double2>(T.nn);
  hipLaunchKernelGGL(k_walk_nodes, grid_for(T.nn), dim3(256), 0, st, T.nn, nleaf, T.nd, wn);
  PGAMD_HIP_CHECK(hipGetLastError());
  const dim3 wgrid((ng + kWalkWaves - 1) / kWalkWaves), wblock(64 * kWalkWaves);
  auto offsets = [&] {
    B.scan(R->jcnt, R->joff, ng, kSlotTotal);
    B.scan(R->ccnt, R->coff, ng, kSlotTotal2);
    const volatile int* host = B.wait();
    R->nj = host[kSlotTotal];
    R->nc = host[kSlotTotal2];
    return host;
  };
  OpenPool pool = open_pool(B, ng, T.nn, theta, ncrit);
  bool opened = pool.rec != nullptr, walks = !opened, big = false;
  // without the pool (its kernels have ended) the walk lists all groups
  auto give_up = [&] {
    B.pool.free_all();
    opened = false;
    walks = true;
  };
  if (opened) {
    hipLaunchKernelGGL(k_fill_int, dim3(1), dim3(1024), 0, st, kPoolUsed, 0, pool.used);
    hipLaunchKernelGGL(k_bh_open, wgrid, wblock, 0, st, ng, gnode, T.nd, wn, L, th2, pool,
                       R->jcnt, R->ccnt);
    hipLaunchKernelGGL(k_copy_ints, dim3(1), dim3(64), 0, st, 2, pool.used,
                       host_dev(host_ints()) + kSlotPool);
    PGAMD_HIP_CHECK(hipGetLastError());
    const volatile int* host = offsets();
    walks = host[kSlotPool] != 0;
    big = host[kSlotPool + 1] != 0;
    if (big) pool.sum = B.pool.try_get<int4>((size_t)pool.chunks * kPoolParts * kOpenChunk);
    if (big && !pool.sum) give_up();
  }
  if (walks) {
    hipLaunchKernelGGL((k_bh_walk<false>), wgrid, wblock, 0, st, ng, gnode, T.nd, wn, L, th2,
                       opened ? pool.level : nullptr, R->jcnt, R->ccnt, nullptr, nullptr, nullptr,
                       nullptr);
    PGAMD_HIP_CHECK(hipGetLastError());
    offsets();
  }
  R->jlist = R->mem.try_get<int>(R->nj);
  R->clist = R->jlist ? R->mem.try_get<int>(R->nc) : nullptr;
  if (!R->clist && opened) give_up();
  if (!R->jlist) R->jlist = R->mem.get<int>(R->nj);
  if (!R->clist) R->clist = R->mem.get<int>(R->nc);
  if (opened) {
    hipLaunchKernelGGL(k_bh_list<false>, dim3(ng), dim3(kListThreads), 0, st, ng, pool, wn.item,
                       R->joff, R->coff, R->jlist, R->clist);
    if (big)
      hipLaunchKernelGGL(k_bh_list<true>, dim3(ng), dim3(kListThreads), 0, st, ng, pool, wn.item,
                         R->joff, R->coff, R->jlist, R->clist);
    hipLaunchKernelGGL(k_bh_whole, grid_for(ng), dim3(256), 0, st, ng, R->jcnt, R->ccnt, wn,
                       R->coff, gnode, T.nd, L, th2, R->clist);
  }
  if (walks)
    hipLaunchKernelGGL((k_bh_walk<true>), wgrid, wblock, 0, st, ng, gnode, T.nd, wn, L, th2,
                       opened ? pool.level : nullptr, nullptr, nullptr, R->joff, R->coff, R->jlist,
                       R->clist);
  PGAMD_HIP_CHECK(hipGetLastError());
  finish(B, *R, true);
  return R;
}

}  // namespace

// ------------------------------------------------------------ C ABI
namespace {
hipStream_t g_stream = nullptr;
std::mutex g_mutex;

hipStream_t pick_stream(void* s) {
  if (s) return (hipStream_t)s;
  if (!g_stream) PGAMD_HIP_CHECK(hipStreamCreateWithFlags(&g_stream, hipStreamNonBlocking));
  return g_stream;
}
}  // namespace

// TreePM lists of pgt_treepm_build (libpgtree.so), built on the GPU.
// x: device [n][3] FP64 positions in the periodic unit box [0, 1).  Returns
// a handle (null after an API error).  Synchronous on `stream` (null = the
// library's stream).
PGAMD_API void* pgt_dev_treepm_build(int n, const double* x, double rcut, int ncrit, void* stream) {
  std::lock_guard<std::mutex> lk(g_mutex);
  ensure_device();
  if (n <= 0 || !x || !(rcut > 0.0 && rcut < 0.5) || ncrit < 1) {
    api_error(3, "pgt_dev_treepm_build: n=%d rcut=%g ncrit=%d (need n > 0, 0 < rcut < 0.5, "
                 "ncrit >= 1, x non-null)", n, rcut, ncrit);
    return nullptr;
  }
  return treepm_build(n, x, rcut, ncrit, pick_stream(stream));
}

// Barnes-Hut lists of pgt_bh_build (libpgtree.so), built on the GPU.
// x: device [n][3], m: device [n], FP64.
PGAMD_API void* pgt_dev_bh_build(int n, const double* x, const double* m, double theta, int ncrit,
                                 int nleaf, void* stream) {
  std::lock_guard<std::mutex> lk(g_mutex);
  ensure_device();
  if (n <= 1 || !x || !m || !(theta > 0.0) || ncrit < 1 || nleaf < 1) {
    api_error(3, "pgt_dev_bh_build: n=%d theta=%g ncrit=%d nleaf=%d (need n > 1, theta > 0, "
                 "ncrit, nleaf >= 1, x and m non-null)", n, theta, ncrit, nleaf);
    return nullptr;
  }
  return bh_build(n, x, m, theta, ncrit, nleaf, pick_stream(stream));
}

// info[8] = {np, ngroups, len(ilist), len(jlist), len(clist), ncells,
//            sum ni*nj, sum ni*ncells}, as pgt_info.
PGAMD_API int pgt_dev_info(void* h, long long* info) {
  if (!h || !info) {
    api_error(3, "pgt_dev_info: null argument");
    return -1;
  }
  const Lists* r = static_cast<Lists*>(h);
  info[0] = r->np;
  info[1] = r->ng;
  info[2] = r->ni;
  info[3] = r->nj;
  info[4] = r->nc;
  info[5] = r->ncells;
  info[6] = r->work_pp;
  info[7] = r->work_pc;
  return 0;
}

namespace {
// Device pointer and byte size of array `what` (codes of pgt_get).
const void* array_of(const Lists* r, int what, size_t* bytes) {
  const size_t ng = (size_t)r->ng;
  switch (what) {
    case 0: *bytes = 3 * sizeof(double) * (size_t)r->np; return r->pos;
    case 1: *bytes = sizeof(int) * (size_t)r->np; return r->src;
    case 2: *bytes = sizeof(int) * ng; return r->ioff;
    case 3: *bytes = sizeof(int) * ng; return r->icnt;
    case 4: *bytes = sizeof(int) * (size_t)r->ni; return r->ilist;
    case 5: *bytes = sizeof(int) * ng; return r->joff;
    case 6: *bytes = sizeof(int) * ng; return r->jcnt;
    case 7: *bytes = sizeof(int) * (size_t)r->nj; return r->jlist;
    case 8: *bytes = sizeof(int) * ng; return r->coff;
    case 9: *bytes = sizeof(int) * ng; return r->ccnt;
    case 10: *bytes = sizeof(int) * (size_t)r->nc; return r->clist;
    case 11: *bytes = sizeof(int) * ng; return r->order;
    case 12: *bytes = 10 * sizeof(double) * (size_t)r->ncells; return r->cells;
    default: *bytes = 0; return nullptr;
  }
}
}  // namespace

// Device pointer of array `what` (0 pos, 1 src, 2 ioff, 3 icnt, 4 ilist,
// 5 joff, 6 jcnt, 7 jlist, 8 coff, 9 ccnt, 10 clist, 11 order, 12 cells),
// valid until pgt_dev_free.
PGAMD_API const void* pgt_dev_ptr(void* h, int what) {
  size_t b = 0;
  const void* p = h ? array_of(static_cast<Lists*>(h), what, &b) : nullptr;
  if (!p) api_error(3, "pgt_dev_ptr: bad handle or array code %d", what);
  return p;
}

// Copies array `what` to host memory `out` (sized as pgt_get's).  Synchronous.
PGAMD_API int pgt_dev_get(void* h, int what, void* out) {
  size_t b = 0;
  const void* p = h ? array_of(static_cast<Lists*>(h), what, &b) : nullptr;
  if (!p || !out) {
    api_error(3, "pgt_dev_get: bad handle, array code %d or output", what);
    return -1;
  }
  if (b) PGAMD_HIP_CHECK(hipMemcpy(out, p, b, hipMemcpyDeviceToHost));
  return 0;
}

// Packs the batch-call inputs on the device: pos4[np] = float4 {float(x) *
// float(scale), ..., float(mass[src])} and, for Barnes-Hut lists, cells12
// [ncells] = 12 floats {x, y, z, M, Qxx, Qxy, Qxz, Qyy, Qyz, Qzz, 0, 0}
// (either output may be null).  mass: device [n] FP64 of the original
// particles.  Asynchronous on `stream`.
PGAMD_API int pgt_dev_pack(void* h, const double* mass, double scale, void* pos4, void* cells12,
                           void* stream) {
  if (!h || (pos4 && !mass)) {
    api_error(3, "pgt_dev_pack: null handle or mass");
    return -1;
  }
  const Lists* r = static_cast<Lists*>(h);
  hipStream_t st = pick_stream(stream);
  if (pos4 && r->np > 0)
    hipLaunchKernelGGL(k_pack, grid_for(r->np), dim3(256), 0, st, (int)r->np, r->pos, r->src,
                       mass, (float)scale, (float4*)pos4);
  if (cells12 && r->ncells > 0)
    hipLaunchKernelGGL(k_pack_cells, grid_for(r->ncells), dim3(256), 0, st, (int)r->ncells,
                       r->cells, (float*)cells12);
  PGAMD_HIP_CHECK(hipGetLastError());
  return 0;
}

PGAMD_API void pgt_dev_free(void* h) {
  if (!h) return;
  std::lock_guard<std::mutex> lk(g_mutex);
  Lists* r = static_cast<Lists*>(h);
  PGAMD_HIP_CHECK(hipDeviceSynchronize());
  r->mem.free_all();
  delete r;
}
