// Device-wide primitives for the graph build, written for gfx950 (wave64):
// an exclusive prefix sum and a stable LSD radix sort.  Both are plain
// integer, HBM-bound kernels; tiles are sized for 256-thread workgroups.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include <cstdint>
#include <stdexcept>
#include <string>
#include <vector>

namespace gx {

#define GX_HIP(call)                                                                               \
  do {                                                                                             \
    hipError_t _e = (call);                                                                        \
    if (_e != hipSuccess)                                                                          \
      throw ::gx::HipError(std::string(#call) + ": " + hipGetErrorString(_e), (int)_e);            \
  } while (0)

struct HipError : std::runtime_error {
  int code;
  HipError(const std::string& m, int c) : std::runtime_error(m), code(c) {}
};

struct DevBuf;

// Buffers that the running build reads no more.  They stay allocated for the
// next build on the handle and are freed only when an allocation would
// otherwise fail; ensure() of a listed buffer takes it off the list.
struct ReclaimList {
  hipStream_t st = nullptr;
  hipStream_t st2 = nullptr;  // a second stream of the same handle (drained too before a free)
  std::vector<DevBuf*> dead;
  uint64_t allocs = 0;  // device allocations made while the list was installed
  uint64_t freed = 0;   // listed buffers freed to make room
};
inline thread_local ReclaimList* tl_reclaim = nullptr;

// Growable device allocation, reused across builds on one handle.
struct DevBuf {
  void* p = nullptr;
  size_t cap = 0;
  DevBuf() = default;
  DevBuf(const DevBuf&) = delete;
  DevBuf& operator=(const DevBuf&) = delete;
  ~DevBuf() { release(); }
  void release() {
    if (p) (void)hipFree(p);
    p = nullptr;
    cap = 0;
  }
  inline void* ensure(size_t bytes);
  template <class T>
  T* as() const { return static_cast<T*>(p); }
};

// Frees one listed buffer other than `self` (after the stream has drained:
// kernels in flight may still read it) toward an allocation of `need`
// bytes: the smallest that covers what free memory lacks, else the
// largest; false if none is left.  Callers free one at a time until their
// allocation fits, so a build short of memory gives up as little of the
// next build's buffers as it can.
inline bool reclaim_dead(const DevBuf* self, size_t need) {
  ReclaimList* r = tl_reclaim;
  if (!r) return false;
  size_t fr = 0, tot = 0;
  if (hipMemGetInfo(&fr, &tot) != hipSuccess) fr = 0;
  const size_t lack = need > fr ? need - fr : 0;
  const size_t none = r->dead.size();
  size_t fit = none, big = none;
  for (size_t i = 0; i < r->dead.size(); i++) {
    const DevBuf* d = r->dead[i];
    if (d == self || !d->p) continue;
    if (d->cap >= lack && (fit == none || d->cap < r->dead[fit]->cap)) fit = i;
    if (big == none || d->cap > r->dead[big]->cap) big = i;
  }
  const size_t pick = fit != none ? fit : big;
  if (pick == none) return false;
  (void)hipStreamSynchronize(r->st);
  if (r->st2) (void)hipStreamSynchronize(r->st2);
  r->dead[pick]->release();
  r->dead[pick] = r->dead.back();
  r->dead.pop_back();
  r->freed++;
  return true;
}

// Takes a buffer in use again off the list (every listing: a buffer may be
// listed by several phases).
inline void reclaim_forget(const DevBuf* d) {
  if (!tl_reclaim) return;
  auto& v = tl_reclaim->dead;
  for (size_t i = 0; i < v.size();)
    if (v[i] == d) {
      v[i] = v.back();
      v.pop_back();
    } else {
      i++;
    }
}

inline void* DevBuf::ensure(size_t bytes) {
  reclaim_forget(this);
  if (bytes == 0) bytes = 256;
  if (bytes > cap) {
    release();
    hipError_t e = hipMalloc(&p, bytes);
    while (e == hipErrorOutOfMemory && reclaim_dead(this, bytes)) {
      (void)hipGetLastError();
      e = hipMalloc(&p, bytes);
    }
    if (tl_reclaim) tl_reclaim->allocs++;
    if (e != hipSuccess) {
      (void)hipGetLastError();
      p = nullptr;
      throw HipError("hipMalloc of " + std::to_string(bytes) + " bytes: " + hipGetErrorString(e), (int)e);
    }
    cap = bytes;
  }
  return p;
}

// Installs a handle's reclaim list for the calling thread while a build
// phase runs.
struct ReclaimScope {
  ReclaimList* prev;
  ReclaimScope(ReclaimList* r, hipStream_t st) : prev(tl_reclaim) {
    r->st = st;
    tl_reclaim = r;
  }
  ~ReclaimScope() { tl_reclaim = prev; }
  ReclaimScope(const ReclaimScope&) = delete;
  ReclaimScope& operator=(const ReclaimScope&) = delete;
};

constexpr int kBlock = 256;

static inline unsigned grid_for(size_t n, size_t per_block, unsigned cap = 1u << 20) {
  size_t g = (n + per_block - 1) / per_block;
  if (g == 0) g = 1;
  return (unsigned)(g > cap ? cap : g);
}

// ---------------------------------------------------------------------------
// Exclusive scan: out[i] = sum(in[0..i)), out[n] = total.  out may not alias
// what in reads.  `in` is any device functor of the element number, so that
// a value made of a few others needs no array and launch of its own; it is
// called twice per element.
// ---------------------------------------------------------------------------

constexpr int kScanItems = 8;
constexpr int kScanTile = kBlock * kScanItems;

template <class Tin>
struct ScanArray {
  const Tin* __restrict__ p;
  __device__ inline Tin operator()(size_t i) const { return p[i]; }
};

template <class T, int kThreads = kBlock>
__device__ inline T block_exclusive_scan(T v, T* total) {
  __shared__ T wsum[kThreads / 64];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  T x = v;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    T y = __shfl_up(x, d, 64);
    if (lane >= d) x += y;
  }
  if (lane == 63) wsum[wid] = x;
  __syncthreads();
  T before = 0, all = 0;
#pragma unroll
  for (int w = 0; w < kThreads / 64; w++) {
    if (w < wid) before += wsum[w];
    all += wsum[w];
  }
  __syncthreads();
  *total = all;
  return before + x - v;
}

template <class In, class T>
__global__ void __launch_bounds__(kBlock) k_scan_reduce(In in, size_t n, T* __restrict__ part) {
  size_t base = (size_t)blockIdx.x * kScanTile;
  T s = 0;
#pragma unroll
  for (int i = 0; i < kScanItems; i++) {
    size_t j = base + (size_t)i * kBlock + threadIdx.x;
    if (j < n) s += (T)in(j);
  }
  T tot;
  (void)block_exclusive_scan<T>(s, &tot);
  if (threadIdx.x == 0) part[blockIdx.x] = tot;
}

// The tile passes through LDS twice: loaded and stored with consecutive
// threads on consecutive elements (whole lines per wave instruction), and
// scanned with each thread on kScanItems consecutive elements.  Tile
// position q sits at LDS slot q + q / kScanItems, so the threads' runs of
// kScanItems fall on different banks.
// part: the tiles' sums, scanned, or (kSumParts) as they are: each block
// then adds up those before its own.
template <class In, class T, bool kSumParts>
__global__ void __launch_bounds__(kBlock) k_scan_apply(In in, size_t n, const T* __restrict__ part,
                                                       T* __restrict__ out) {
  __shared__ T tile[kScanTile + kBlock];
  const size_t base = (size_t)blockIdx.x * kScanTile;
#pragma unroll
  for (int i = 0; i < kScanItems; i++) {
    const uint32_t q = (uint32_t)(i * kBlock + threadIdx.x);
    const size_t j = base + q;
    tile[q + q / kScanItems] = j < n ? (T)in(j) : (T)0;
  }
  __syncthreads();
  const uint32_t run = threadIdx.x * (kScanItems + 1);  // slot of this thread's first element
  T v[kScanItems];
  T s = 0;
#pragma unroll
  for (int i = 0; i < kScanItems; i++) {
    v[i] = tile[run + i];
    s += v[i];
  }
  T tot, before = 0;
  if constexpr (kSumParts) {
    T mine = 0;
    for (uint32_t q = threadIdx.x; q < blockIdx.x; q += kBlock) mine += part[q];
    (void)block_exclusive_scan<T>(mine, &before);
  } else {
    before = part[blockIdx.x];
  }
  T ex = block_exclusive_scan<T>(s, &tot) + before;
#pragma unroll
  for (int i = 0; i < kScanItems; i++) {  // the thread's own slots: no other thread reads them
    tile[run + i] = ex;
    ex += v[i];
  }
  if (blockIdx.x == gridDim.x - 1 && threadIdx.x == kBlock - 1) out[n] = ex;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kScanItems; i++) {
    const uint32_t q = (uint32_t)(i * kBlock + threadIdx.x);
    const size_t j = base + q;
    if (j < n) out[j] = tile[q + q / kScanItems];
  }
}

// Scratch needed by exclusive_scan for n elements (bytes), all levels.
template <class T>
static size_t scan_scratch_bytes(size_t n) {
  size_t b = 0;
  while (n > (size_t)kScanTile) {
    n = (n + kScanTile - 1) / kScanTile;
    b += (n + 1) * sizeof(T) * 2 + 256;
  }
  return b + 256;
}

// Short inputs: one block, tile after tile.
constexpr int kScanOneThreads = 1024;
constexpr size_t kScanOne = 2 * (size_t)kScanOneThreads * kScanItems;
template <class In, class T>
__global__ void __launch_bounds__(kScanOneThreads) k_scan_one(In in, size_t n, T* __restrict__ out) {
  T carry = 0;
  for (size_t base = 0; base < n; base += (size_t)kScanOneThreads * kScanItems) {
    const size_t j0 = base + (size_t)threadIdx.x * kScanItems;
    T v[kScanItems], s = 0, tot;
#pragma unroll
    for (int i = 0; i < kScanItems; i++) {
      v[i] = j0 + i < n ? (T)in(j0 + i) : (T)0;
      s += v[i];
    }
    T ex = block_exclusive_scan<T, kScanOneThreads>(s, &tot) + carry;
#pragma unroll
    for (int i = 0; i < kScanItems; i++) {
      if (j0 + i < n) out[j0 + i] = ex;
      ex += v[i];
    }
    carry += tot;
  }
  if (threadIdx.x == 0) out[n] = carry;
}

// One launch up to kScanOne elements, two (the tiles' sums, then the tiles)
// while a block can add up the sums before its own, 2048 at most; beyond
// that the sums are scanned in between.  (A launch costs 2.5 us: three of
// them bounded every scan of a small graph.)
constexpr size_t kSumTiles = 2048;
template <class T, class In>
static void exclusive_scan_of(In in, T* out, size_t n, char* scratch, hipStream_t st) {
  if (n <= kScanOne) {
    hipLaunchKernelGGL((k_scan_one<In, T>), dim3(1), dim3(kScanOneThreads), 0, st, in, n, out);
    GX_HIP(hipGetLastError());
    return;
  }
  const size_t tiles = (n + kScanTile - 1) / kScanTile;
  T* part = reinterpret_cast<T*>(scratch);
  T* partscan = part + (tiles + 1);
  char* next = reinterpret_cast<char*>(partscan + tiles + 1);
  next = reinterpret_cast<char*>(((uintptr_t)next + 255) & ~(uintptr_t)255);
  hipLaunchKernelGGL((k_scan_reduce<In, T>), dim3((unsigned)tiles), dim3(kBlock), 0, st, in, n, part);
  GX_HIP(hipGetLastError());
  if (tiles <= kSumTiles) {
    hipLaunchKernelGGL((k_scan_apply<In, T, true>), dim3((unsigned)tiles), dim3(kBlock), 0, st, in, n, (const T*)part,
                       out);
  } else {
    exclusive_scan_of<T>(ScanArray<T>{part}, partscan, tiles, next, st);
    hipLaunchKernelGGL((k_scan_apply<In, T, false>), dim3((unsigned)tiles), dim3(kBlock), 0, st, in, n,
                       (const T*)partscan, out);
  }
  GX_HIP(hipGetLastError());
}

template <class Tin, class T>
static void exclusive_scan(const Tin* in, T* out, size_t n, char* scratch, hipStream_t st) {
  exclusive_scan_of<T>(ScanArray<Tin>{in}, out, n, scratch, st);
}

// ---------------------------------------------------------------------------
// Stable LSD radix sort, 8-bit digits.  Keys are up to 128 bits (KeyT =
// uint32_t, uint64_t or Key128); the digits sorted are bytes
// [byte_lo, byte_hi) of the key's integer value.  Values are uint32_t or
// uint64_t.
// ---------------------------------------------------------------------------

struct Key128 {
  uint64_t lo, hi;
};

__device__ __host__ inline uint32_t key_byte(uint32_t k, int b) { return (k >> (8 * b)) & 0xff; }
__device__ __host__ inline uint32_t key_byte(uint64_t k, int b) { return (uint32_t)(k >> (8 * b)) & 0xff; }
__device__ __host__ inline uint32_t key_byte(const Key128& k, int b) {
  return b < 8 ? (uint32_t)(k.lo >> (8 * b)) & 0xff : (uint32_t)(k.hi >> (8 * (b - 8))) & 0xff;
}

// A tile of the sort: kSortThreads threads with kPer elements each.  4096
// elements over 256 digits leave runs of 16 on average, 128 bytes of 8-byte
// keys (2048 left half a line each and twice the digit counts to scan); of
// 16-byte keys 2048 do.
constexpr int kSortThreads = 512, kSortWaves = kSortThreads / 64;
template <class KeyT>
struct SortTile {
  static constexpr int kPer = sizeof(KeyT) > 8 ? 4 : 8;
  static constexpr int kTile = kSortThreads * kPer;
};

// Rank of each lane's digit among the wave's elements so far: count holds
// the wave's elements of each digit (raised here), so successive calls rank
// successive elements with no barrier between them.  All lanes call it.
// (The match takes four vector instructions a bit, with the three-input one;
// selects between a ballot and its complement took six: the scatters are
// bound by them, 10 Mbp build 29.8 -> 28.8 ms with branch-free loads of the
// k-mers' words.)
__device__ inline uint32_t wave_rank(uint16_t* count, uint32_t d, bool valid, uint64_t lt) {
  const uint64_t v = __ballot(valid);
  uint32_t lo = (uint32_t)v, hi = (uint32_t)(v >> 32);
#pragma unroll
  for (int b = 0; b < 8; b++) {
    const uint32_t s = (uint32_t)((int32_t)(d << (31 - b)) >> 31);  // the lane's bit in every place
    const uint64_t m = __ballot(s != 0);
    lo = __builtin_amdgcn_bitop3_b32(lo, (uint32_t)m, s, 0x90);  // lo & ~(m ^ s)
    hi = __builtin_amdgcn_bitop3_b32(hi, (uint32_t)(m >> 32), s, 0x90);
  }
  const uint64_t match = ((uint64_t)hi << 32) | lo;
  // the wave's LDS accesses run in order: read by every lane, then raised
  // by the group's first
  const uint32_t before = count[d];
  __builtin_amdgcn_wave_barrier();
  if (valid && (match & lt) == 0) count[d] = (uint16_t)(before + __popcll(match));
  __builtin_amdgcn_wave_barrier();
  return before + __popcll(match & lt);
}

// The waves' digit counts of a tile turned into each wave's first position
// of each digit, in digit order and then wave order; returns (threads below
// 256) the first position of digit threadIdx.x.  wsum: [4].  Barriers before
// and after by the caller.
template <int kWaves>
__device__ inline uint32_t tile_digit_starts(uint16_t (*wcnt)[256], uint32_t* wsum) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  uint32_t c[kWaves], tot = 0, incl = 0;
  if (threadIdx.x < 256) {
#pragma unroll
    for (int w = 0; w < kWaves; w++) {
      c[w] = tot;
      tot += wcnt[w][threadIdx.x];
    }
    incl = tot;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t y = __shfl_up(incl, o);
      if (lane >= o) incl += y;
    }
    if (lane == 63) wsum[wid] = incl;
  }
  __syncthreads();
  if (threadIdx.x >= 256) return 0;
  uint32_t b = incl - tot;
  for (int w = 0; w < wid; w++) b += wsum[w];
#pragma unroll
  for (int w = 0; w < kWaves; w++) wcnt[w][threadIdx.x] = (uint16_t)(b + c[w]);
  return b;
}

// Sorts of few elements: one block, every pass in LDS, one launch (three per
// pass otherwise, 2.5 us each with nothing in between: 12 passes over the
// 1600 heads of a 5 kbp genome took 100 us).  A wave holds a contiguous run
// of the elements in registers, so its ranks need no barrier: a match over
// the digit's bits plus the wave's own count of earlier equal digits; the
// waves' counts are then summed per digit.
constexpr int kSmallThreads = 1024, kSmallPer = 4;
constexpr size_t kSmallSort = (size_t)kSmallThreads * kSmallPer;
template <class KeyT, bool kVals, class ValT>
__global__ void __launch_bounds__(kSmallThreads) k_radix_small(KeyT* __restrict__ keys, ValT* __restrict__ vals,
                                                               uint32_t n, int byte_lo, int byte_hi) {
  constexpr int kWaves = kSmallThreads / 64;
  __shared__ KeyT sk[kSmallSort];
  __shared__ ValT sv[kVals ? kSmallSort : 1];
  __shared__ uint16_t wcnt[kWaves][256];
  __shared__ uint32_t wsum[4];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const uint64_t lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  const uint32_t first = (uint32_t)wid * 64 * kSmallPer;
  KeyT key[kSmallPer];
  ValT val[kSmallPer];
#pragma unroll
  for (int r = 0; r < kSmallPer; r++) {
    const uint32_t j = first + r * 64 + lane;
    if (j < n) {
      key[r] = keys[j];
      if (kVals) val[r] = vals[j];
    }
  }
  for (int byte = byte_lo; byte < byte_hi; byte++) {
#pragma unroll
    for (int q = 0; q < 4; q++) wcnt[wid][q * 64 + lane] = 0;
    __builtin_amdgcn_wave_barrier();
    uint32_t rank[kSmallPer], dig[kSmallPer];
#pragma unroll
    for (int r = 0; r < kSmallPer; r++) {
      const bool valid = first + r * 64 + lane < n;
      dig[r] = valid ? key_byte(key[r], byte) : 0;
      rank[r] = wave_rank(wcnt[wid], dig[r], valid, lt);
    }
    __syncthreads();
    tile_digit_starts<kWaves>(wcnt, wsum);
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kSmallPer; r++)
      if (first + r * 64 + lane < n) {
        const uint32_t pos = wcnt[wid][dig[r]] + rank[r];
        sk[pos] = key[r];
        if (kVals) sv[pos] = val[r];
      }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kSmallPer; r++) {
      const uint32_t j = first + r * 64 + lane;
      if (j < n) {
        key[r] = sk[j];
        if (kVals) val[r] = sv[j];
      }
    }
  }
#pragma unroll
  for (int r = 0; r < kSmallPer; r++) {
    const uint32_t j = first + r * 64 + lane;
    if (j < n) {
      keys[j] = key[r];
      if (kVals) vals[j] = val[r];
    }
  }
}

// First output position of digit threadIdx.x (threads below 256) for a tile
// from the tiles' counts themselves (hist, digit-major, not scanned): with
// few tiles every block adds up the counts before its own, which saves the
// launches of a scan.  wsum: [4].  All threads call it.
constexpr unsigned kDirectTiles = 64;
__device__ inline uint64_t direct_digit_start(const uint32_t* __restrict__ hist, unsigned ntiles, uint32_t* wsum) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  uint32_t before = 0, all = 0, incl = 0;
  if (threadIdx.x < 256) {
#pragma unroll 8
    for (unsigned t = 0; t < ntiles; t++) {
      const uint32_t c = hist[(size_t)threadIdx.x * ntiles + t];
      before += t < blockIdx.x ? c : 0;
      all += c;
    }
    incl = all;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t y = __shfl_up(incl, o);
      if (lane >= o) incl += y;
    }
    if (lane == 63) wsum[wid] = incl;
  }
  __syncthreads();
  if (threadIdx.x >= 256) return 0;
  uint32_t b = incl - all;
  for (int w = 0; w < wid; w++) b += wsum[w];
  return (uint64_t)b + before;
}

template <class KeyT>
__global__ void __launch_bounds__(kSortThreads) k_radix_hist(const KeyT* __restrict__ keys, size_t n, int byte,
                                                             uint32_t* __restrict__ hist, unsigned ntiles) {
  __shared__ uint32_t h[256];
  if (threadIdx.x < 256) h[threadIdx.x] = 0;
  __syncthreads();
  const size_t base = (size_t)blockIdx.x * SortTile<KeyT>::kTile;
#pragma unroll
  for (int i = 0; i < SortTile<KeyT>::kPer; i++) {
    const size_t j = base + (size_t)i * kSortThreads + threadIdx.x;
    if (j < n) atomicAdd(&h[key_byte(keys[j], byte)], 1u);
  }
  __syncthreads();
  if (threadIdx.x < 256) hist[(size_t)threadIdx.x * ntiles + blockIdx.x] = h[threadIdx.x];
}

// A load of data read once, in order: nontemporal for integer words, so
// the stream does not evict lines other accesses reuse.
template <class T>
__device__ inline T load_stream(const T* p) {
  if constexpr (std::is_integral<T>::value) return __builtin_nontemporal_load(p);
  else return *p;
}

// Scatter with stable ranks.  Each wave of the tile holds a contiguous run
// of its elements in registers and ranks them by itself (wave_rank), so the
// tile has five barriers in all; ranked in rounds of 256 elements with the
// waves' counts exchanged in each, it had three per round and waited on them
// (the records of 10 Mbp, k = 31: 3.9 -> 3.0 ms; of 4 x 20 M at k = 55 3.5 ->
// 2.7 ms).  The elements then go through an LDS stage in digit order and leave as one
// contiguous run per digit (the tile's share of that digit's output range):
// scattered element stores would leave lines partly written, and the partial
// lines cost extra HBM writes.
// offs: the scanned counts, or (kDirect) the counts themselves.
template <class KeyT, bool kVals, class ValT, bool kDirect>
__global__ void __launch_bounds__(kSortThreads) k_radix_scatter(const KeyT* __restrict__ keys, const ValT* __restrict__ vals,
                                                          size_t n, int byte,
                                                          const typename std::conditional<kDirect, uint32_t, uint64_t>::type* __restrict__ offs,
                                                          unsigned ntiles, KeyT* __restrict__ okeys,
                                                          ValT* __restrict__ ovals) {
  constexpr int kPer = SortTile<KeyT>::kPer, kTile = SortTile<KeyT>::kTile;
  __shared__ uint64_t run[256];  // output position of a digit's elements less their place in the stage
  __shared__ uint32_t wsum[4];
  __shared__ uint16_t wcnt[kSortWaves][256];
  __shared__ KeyT sk[kTile];
  __shared__ ValT sv[kVals ? kTile : 1];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const uint64_t lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  const size_t base = (size_t)blockIdx.x * kTile;
  const uint32_t tn = (uint32_t)(n - base < (size_t)kTile ? n - base : (size_t)kTile);
  const uint32_t first = (uint32_t)wid * 64 * kPer + lane;
  KeyT key[kPer];
  ValT val[kPer];
  uint32_t rank[kPer];
#pragma unroll
  for (int r = 0; r < kPer; r++) {
    const uint32_t i = first + r * 64;
    key[r] = KeyT{};
    if (i < tn) {
      key[r] = load_stream(keys + base + i);
      if (kVals) val[r] = load_stream(vals + base + i);
    }
  }
  uint64_t out;
  if constexpr (kDirect) {
    out = direct_digit_start(offs, ntiles, wsum);
  } else {
    out = threadIdx.x < 256 ? offs[(size_t)threadIdx.x * ntiles + blockIdx.x] : 0;
  }
#pragma unroll
  for (int q = 0; q < 4; q++) wcnt[wid][q * 64 + lane] = 0;
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int r = 0; r < kPer; r++) rank[r] = wave_rank(wcnt[wid], key_byte(key[r], byte), first + r * 64 < tn, lt);
  __syncthreads();
  const uint32_t start = tile_digit_starts<kSortWaves>(wcnt, wsum);
  if (threadIdx.x < 256) run[threadIdx.x] = out - start;
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kPer; r++)
    if (first + r * 64 < tn) {
      const uint32_t pos = wcnt[wid][key_byte(key[r], byte)] + rank[r];
      sk[pos] = key[r];
      if (kVals) sv[pos] = val[r];
    }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kPer; r++) {
    const uint32_t i = r * kSortThreads + threadIdx.x;
    if (i < tn) {
      const KeyT k = sk[i];
      const uint64_t pos = run[key_byte(k, byte)] + i;
      okeys[pos] = k;
      if (kVals) ovals[pos] = sv[i];
    }
  }
}

template <class KeyT>
static size_t radix_scratch_bytes(size_t n) {
  size_t ntiles = (n + SortTile<KeyT>::kTile - 1) / SortTile<KeyT>::kTile;
  if (ntiles == 0) ntiles = 1;
  size_t h = 256 * ntiles;
  return h * 4 + (h + 1) * 8 + scan_scratch_bytes<uint64_t>(h) + 1024;
}

// Sorts (keys, vals) by bytes [byte_lo, byte_hi).  Uses (k2, v2) as the
// ping-pong buffers; returns true when the result ended in (k2, v2).
template <class KeyT, bool kVals, class ValT>
static bool radix_sort_impl(KeyT* k1, ValT* v1, KeyT* k2, ValT* v2, size_t n, int byte_lo, int byte_hi, char* scratch,
                            hipStream_t st) {
  if (n <= 1 || byte_lo >= byte_hi) return false;
  if (n <= kSmallSort) {
    hipLaunchKernelGGL((k_radix_small<KeyT, kVals, ValT>), dim3(1), dim3(kSmallThreads), 0, st, k1, v1, (uint32_t)n,
                       byte_lo, byte_hi);
    GX_HIP(hipGetLastError());
    return false;
  }
  unsigned ntiles = (unsigned)((n + SortTile<KeyT>::kTile - 1) / SortTile<KeyT>::kTile);
  size_t h = (size_t)256 * ntiles;
  uint32_t* hist = reinterpret_cast<uint32_t*>(scratch);
  uint64_t* offs = reinterpret_cast<uint64_t*>(((uintptr_t)(hist + h) + 255) & ~(uintptr_t)255);
  char* sc = reinterpret_cast<char*>(((uintptr_t)(offs + h + 1) + 255) & ~(uintptr_t)255);
  bool flip = false;
  for (int b = byte_lo; b < byte_hi; b++) {
    KeyT* ik = flip ? k2 : k1;
    KeyT* ok = flip ? k1 : k2;
    ValT* iv = flip ? v2 : v1;
    ValT* ov = flip ? v1 : v2;
    hipLaunchKernelGGL((k_radix_hist<KeyT>), dim3(ntiles), dim3(kSortThreads), 0, st, ik, n, b, hist, ntiles);
    GX_HIP(hipGetLastError());
    if (ntiles <= kDirectTiles) {
      hipLaunchKernelGGL((k_radix_scatter<KeyT, kVals, ValT, true>), dim3(ntiles), dim3(kSortThreads), 0, st, ik, iv, n, b,
                         hist, ntiles, ok, ov);
    } else {
      exclusive_scan<uint32_t, uint64_t>(hist, offs, h, sc, st);
      hipLaunchKernelGGL((k_radix_scatter<KeyT, kVals, ValT, false>), dim3(ntiles), dim3(kSortThreads), 0, st, ik, iv, n, b,
                         offs, ntiles, ok, ov);
    }
    GX_HIP(hipGetLastError());
    flip = !flip;
  }
  return flip;
}

template <class KeyT, class ValT = uint32_t>
static bool radix_sort(KeyT* k1, ValT* v1, KeyT* k2, ValT* v2, size_t n, int byte_lo, int byte_hi,
                       char* scratch, hipStream_t st) {
  return v1 ? radix_sort_impl<KeyT, true, ValT>(k1, v1, k2, v2, n, byte_lo, byte_hi, scratch, st)
            : radix_sort_impl<KeyT, false, ValT>(k1, v1, k2, v2, n, byte_lo, byte_hi, scratch, st);
}

}  // namespace gx
