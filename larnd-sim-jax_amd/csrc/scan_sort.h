// Deterministic device-wide exclusive scan and stable LSD radix sort (key, value) pairs.
// Hand-written instead of a library call so that every launch is a plain kernel (no memset or
// host synchronisation inside), which keeps the forward capturable into a hipGraph.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace lsim {

constexpr int kScanThreads = 256;
constexpr int kScanItems = 16;
constexpr int kScanTile = kScanThreads * kScanItems;  // 4096

template <typename T>
__device__ __forceinline__ T shfl_up_t(T v, int d) {
  return __shfl_up(v, d, kWave);
}

// Block-wide exclusive scan of one value per thread (256 threads).  Returns the exclusive
// prefix; `total` receives the block sum.  Uses `sh` (>= 4 entries of T) as scratch.
template <typename T>
__device__ __forceinline__ T block_exclusive_scan(T v, T* sh, T& total) {
  const int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
  T inc = v;
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    T u = shfl_up_t(inc, d);
    if (lane >= d) inc += u;
  }
  // the exclusive prefix is the previous lane's inclusive one (not inc - v: that would round, and
  // a NaN or inf of this thread's own values would reach its prefix, which a cumulative sum's
  // earlier entries never see)
  T exc = shfl_up_t(inc, 1);
  if (lane == 0) exc = 0;
  if (lane == kWave - 1) sh[wid] = inc;
  __syncthreads();
  const int nw = blockDim.x / kWave;
  T base = 0, tot = 0;
  for (int w = 0; w < nw; ++w) {
    if (w < wid) base += sh[w];
    tot += sh[w];
  }
  total = tot;
  __syncthreads();
  return base + exc;
}

// 1) per-tile sums
template <typename T>
__global__ __launch_bounds__(kScanThreads) void k_scan_reduce(const T* __restrict__ in, int64_t n, T* __restrict__ tile_sums) {
  __shared__ T sh[kScanThreads / kWave];
  const int64_t base = (int64_t)blockIdx.x * kScanTile + (int64_t)threadIdx.x * kScanItems;
  T s = 0;
#pragma unroll
  for (int k = 0; k < kScanItems; ++k)
    if (base + k < n) s += in[base + k];
  T tot;
  (void)block_exclusive_scan<T>(s, sh, tot);
  if (threadIdx.x == 0) tile_sums[blockIdx.x] = tot;
}

// 2) exclusive scan of the tile sums in place (one block, loops over chunks); total -> *total
template <typename T, typename TT>
__global__ __launch_bounds__(kScanThreads) void k_scan_tiles(T* __restrict__ sums, int64_t ntiles, TT* __restrict__ total) {
  __shared__ T sh[kScanThreads / kWave];
  T carry = 0;
  for (int64_t c0 = 0; c0 < ntiles; c0 += kScanThreads) {
    const int64_t i = c0 + threadIdx.x;
    T v = i < ntiles ? sums[i] : T(0);
    T tot;
    T ex = block_exclusive_scan<T>(v, sh, tot);
    if (i < ntiles) sums[i] = carry + ex;
    carry += tot;
  }
  if (threadIdx.x == 0 && total) *total = (TT)carry;
}

// 3) scan within each tile plus the tile offset
template <typename T>
__global__ __launch_bounds__(kScanThreads) void k_scan_apply(const T* __restrict__ in, T* __restrict__ out, int64_t n,
                                                            const T* __restrict__ tile_off) {
  __shared__ T sh[kScanThreads / kWave];
  const int64_t base = (int64_t)blockIdx.x * kScanTile + (int64_t)threadIdx.x * kScanItems;
  T v[kScanItems];
  T s = 0;
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    v[k] = (base + k < n) ? in[base + k] : T(0);
    s += v[k];
  }
  T tot;
  T ex = block_exclusive_scan<T>(s, sh, tot) + tile_off[blockIdx.x];
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    if (base + k < n) out[base + k] = ex;
    ex += v[k];
  }
}

inline int64_t scan_tiles(int64_t n) { return (n + kScanTile - 1) / kScanTile; }

// Small inputs (up to 16 values per thread of one 1024-thread workgroup): the whole scan in one
// launch instead of three (the radix sort's digit histograms and the per-row counts are this
// size, and each launch costs a few microseconds on its own).
constexpr int kScanSmallThreads = 1024;
constexpr int kScanSmallItems = 16;
constexpr int64_t kScanSmallMax = (int64_t)kScanSmallThreads * kScanSmallItems;

template <typename T, typename TT>
__global__ __launch_bounds__(kScanSmallThreads) void k_scan_small(const T* in, T* out, int64_t n,
                                                                 TT* __restrict__ total) {  // in may equal out
  __shared__ T sh[kScanSmallThreads / kWave];
  const int per = (int)((n + kScanSmallThreads - 1) / kScanSmallThreads);  // <= kScanSmallItems
  const int64_t base = (int64_t)threadIdx.x * per;
  T v[kScanSmallItems];
  T s = 0;
#pragma unroll
  for (int k = 0; k < kScanSmallItems; ++k) {
    v[k] = (k < per && base + k < n) ? in[base + k] : T(0);
    s += v[k];
  }
  T tot;
  T ex = block_exclusive_scan<T>(s, sh, tot);
#pragma unroll
  for (int k = 0; k < kScanSmallItems; ++k) {
    if (k < per && base + k < n) out[base + k] = ex;
    ex += v[k];
  }
  if (threadIdx.x == 0 && total) *total = (TT)tot;
}

// Exclusive scan of n values (in may equal out).  tmp holds scan_tiles(n) values of T.
template <typename T, typename TT>
inline hipError_t exclusive_scan(const T* in, T* out, int64_t n, T* tmp, TT* total, hipStream_t st) {
  const int64_t nt = scan_tiles(n);
  if (nt == 0) {
    return hipSuccess;
  }
  if (n <= kScanSmallMax) {
    hipLaunchKernelGGL((k_scan_small<T, TT>), dim3(1), dim3(kScanSmallThreads), 0, st, in, out, n, total);
    return hipGetLastError();
  }
  hipLaunchKernelGGL((k_scan_reduce<T>), dim3((unsigned)nt), dim3(kScanThreads), 0, st, in, n, tmp);
  hipLaunchKernelGGL((k_scan_tiles<T, TT>), dim3(1), dim3(kScanThreads), 0, st, tmp, nt, total);
  hipLaunchKernelGGL((k_scan_apply<T>), dim3((unsigned)nt), dim3(kScanThreads), 0, st, in, out, n, tmp);
  return hipGetLastError();
}

// ------------------------------------------------------------------------------------------
// stable LSD radix sort, 8-bit digits
// ------------------------------------------------------------------------------------------
//
// Every wave owns 64 R consecutive items and ranks them by itself (ballots give the peers of a digit, a
// per-wave counter in LDS carries over its R rounds), so a tile costs a fixed few barriers whatever R is.
// Three sizes, each bound by the latency of its steps rather than by the 16 bytes an item moves per pass:
//   n <= 4096            all passes in one workgroup with the items in LDS: one launch instead of 3 a pass
//                        (the sorts of a 1k-segment call 124 -> 34 us);
//   up to 524288 (256 tiles of 8 rounds)
//                        two launches a pass, R = 1 .. 8 such that there are at most 256 tiles (many small
//                        tiles in flight); a tile sums the histograms of those before it as it starts
//                        (256 KB from L2 at most), which saves the scan's one to three launches
//                        (200k segments 190 -> 98 us, 30k 128 -> 62);
//   above                histogram, device-wide scan, scatter (that sum would grow as the square of n).

constexpr int kSortThreads = 256;
constexpr int kSortWaves = kSortThreads / kWave;
constexpr int kSortRounds = 8;  // the most
constexpr int kRadix = 256;
constexpr int kSortSumTiles = 256;
constexpr int kSumBatch = 32;
constexpr int kSmallThreads = 1024;
constexpr int kSmallRounds = 4;
constexpr int kSmallMax = kSmallThreads * kSmallRounds;

__device__ __forceinline__ int radix_digit(uint32_t key, int shift) { return (key >> shift) & (kRadix - 1); }

// Ranks of a wave's items (item r of lane l is the (64 r + l)-th) among its items of the same digit;
// cnt[digit] (this wave's, zero before) ends as the digit's count.
template <int R>
__device__ __forceinline__ void radix_rank(const uint32_t (&key)[R], const bool (&valid)[R], int shift, int* cnt,
                                           int (&rank)[R]) {
  const int lane = threadIdx.x & (kWave - 1);
  const uint64_t lt = (lane == 0) ? 0ull : ((~0ull) >> (64 - lane));
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int dg = radix_digit(key[r], shift);
    uint64_t peers = __ballot(valid[r]);
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      const bool bit = (dg >> b) & 1;
      const uint64_t bb = __ballot(bit);
      peers &= bit ? bb : ~bb;
    }
    const int below = __popcll(peers & lt);
    const int before = valid[r] ? cnt[dg] : 0;
    __builtin_amdgcn_wave_barrier();
    if (valid[r] && below == 0) cnt[dg] = before + __popcll(peers);
    __builtin_amdgcn_wave_barrier();
    rank[r] = before + below;
  }
}

// hist[digit * dstride + tile * tstride] = the tile's count of the digit
template <int R>
__global__ __launch_bounds__(kSortThreads) void k_radix_hist(const uint32_t* __restrict__ keys, int64_t n, int shift,
                                                             int64_t dstride, int64_t tstride, int* __restrict__ hist) {
  __shared__ int h[kRadix];
  h[threadIdx.x] = 0;
  __syncthreads();
  const int64_t base = (int64_t)blockIdx.x * (kSortThreads * R);
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int64_t i = base + r * kSortThreads + threadIdx.x;
    if (i < n) atomicAdd(&h[radix_digit(keys[i], shift)], 1);
  }
  __syncthreads();
  hist[threadIdx.x * dstride + blockIdx.x * tstride] = h[threadIdx.x];
}

// SUM: `hist` holds the tiles' histograms ([tile][digit]) and this tile derives its digits' first
// positions from them; otherwise the scanned ones ([digit][tile]).
template <int R, bool SUM>
__global__ __launch_bounds__(kSortThreads) void k_radix_scatter(const uint32_t* __restrict__ kin,
                                                                const uint32_t* __restrict__ vin,
                                                                uint32_t* __restrict__ kout,
                                                                uint32_t* __restrict__ vout, int64_t n, int shift,
                                                                int ntiles, const int* __restrict__ hist) {
  __shared__ int cnt[kSortWaves][kRadix];
  __shared__ int s_scan[kSortWaves];
  const int t = threadIdx.x, lane = t & (kWave - 1), wid = t / kWave;
  const int64_t i0 = (int64_t)blockIdx.x * (kSortThreads * R) + wid * (kWave * R) + lane;
  uint32_t key[R], val[R];
  bool valid[R];
  int rank[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    valid[r] = i0 + r * kWave < n;
    key[r] = valid[r] ? kin[i0 + r * kWave] : 0;
    val[r] = valid[r] ? vin[i0 + r * kWave] : 0;
  }
#pragma unroll
  for (int w = 0; w < kSortWaves; ++w) cnt[w][t] = 0;
  __syncthreads();
  radix_rank<R>(key, valid, shift, cnt[wid], rank);
  int base;
  if (SUM) {
    int before = 0, total = 0;
    const int me = blockIdx.x;
    for (int t0 = 0; t0 < ntiles; t0 += kSumBatch) {  // (a batch's loads in flight together)
      int v[kSumBatch];
#pragma unroll
      for (int k = 0; k < kSumBatch; ++k) v[k] = hist[min(t0 + k, ntiles - 1) * kRadix + t];
#pragma unroll
      for (int k = 0; k < kSumBatch; ++k) {
        total += t0 + k < ntiles ? v[k] : 0;
        before += t0 + k < me ? v[k] : 0;
      }
    }
    int tot;
    base = block_exclusive_scan<int>(total, s_scan, tot) + before;
  } else {
    base = hist[(int64_t)t * ntiles + blockIdx.x];
  }
  __syncthreads();
  // (thread t: the first positions of digit t in each wave)
#pragma unroll
  for (int w = 0; w < kSortWaves; ++w) {
    const int c = cnt[w][t];
    cnt[w][t] = base;
    base += c;
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if (valid[r]) {
      const int pos = cnt[wid][radix_digit(key[r], shift)] + rank[r];
      kout[pos] = key[r];
      vout[pos] = val[r];
    }
  }
}

// All passes over n <= kSmallMax items in one workgroup.
__global__ __launch_bounds__(kSmallThreads) void k_radix_small(const uint32_t* kin, const uint32_t* vin,
                                                               uint32_t* kout, uint32_t* vout,  // may equal kin, vin
                                                               int n, int bits) {
  constexpr int NW = kSmallThreads / kWave, R = kSmallRounds;
  __shared__ uint32_t s_key[kSmallMax], s_val[kSmallMax];
  __shared__ int cnt[NW][kRadix];
  __shared__ int s_scan[NW];
  const int t = threadIdx.x, lane = t & (kWave - 1), wid = t / kWave;
  const int i0 = wid * (kWave * R) + lane;
  uint32_t key[R], val[R];
  bool valid[R];
  int rank[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    valid[r] = i0 + r * kWave < n;
    key[r] = valid[r] ? kin[i0 + r * kWave] : 0;
    val[r] = valid[r] ? vin[i0 + r * kWave] : 0;
  }
  for (int shift = 0; shift < bits; shift += 8) {
#pragma unroll
    for (int k = 0; k < NW * kRadix / kSmallThreads; ++k) (&cnt[0][0])[k * kSmallThreads + t] = 0;
    __syncthreads();  // (and the pass before has been read back)
    radix_rank<R>(key, valid, shift, cnt[wid], rank);
    __syncthreads();
    int total = 0;
    if (t < kRadix) {
#pragma unroll
      for (int w = 0; w < NW; ++w) total += cnt[w][t];
    }
    int tot;
    int base = block_exclusive_scan<int>(total, s_scan, tot);
    if (t < kRadix) {
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        const int c = cnt[w][t];
        cnt[w][t] = base;
        base += c;
      }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if (valid[r]) {
        const int pos = cnt[wid][radix_digit(key[r], shift)] + rank[r];
        s_key[pos] = key[r];
        s_val[pos] = val[r];
      }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if (valid[r]) {
        key[r] = s_key[i0 + r * kWave];
        val[r] = s_val[i0 + r * kWave];
      }
    }
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if (valid[r]) {
      kout[i0 + r * kWave] = key[r];
      vout[i0 + r * kWave] = val[r];
    }
  }
}

inline int sort_tiles(int64_t n, int rounds) { return (int)((n + (int64_t)kSortThreads * rounds - 1) / (kSortThreads * rounds)); }

// Rounds of a tile for n items: the fewest that leave no more than kSortSumTiles tiles.
inline int sort_rounds(int64_t n) {
  int r = 1;
  while (r < kSortRounds && sort_tiles(n, r) > kSortSumTiles) r *= 2;
  return r;
}

// Bytes of scratch the sort of up to n items needs (histogram + scan tiles).
inline size_t radix_sort_scratch(int64_t n) {
  int64_t nt = sort_tiles(n, sort_rounds(n));
  const int64_t fine = (n + kSortThreads - 1) / kSortThreads;  // (fewer items may have more, smaller tiles)
  if (nt < kSortSumTiles) nt = fine < kSortSumTiles ? fine : kSortSumTiles;
  const int64_t hist = nt * kRadix;
  return (size_t)(hist + scan_tiles(hist) + 4) * sizeof(int);
}

template <int R>
inline hipError_t radix_pass(const uint32_t* ki, const uint32_t* vi, uint32_t* ko, uint32_t* vo, int64_t n, int shift,
                             int* hist, hipStream_t st) {
  const int nt = sort_tiles(n, R);
  if (nt <= kSortSumTiles) {
    hipLaunchKernelGGL(k_radix_hist<R>, dim3(nt), dim3(kSortThreads), 0, st, ki, n, shift, (int64_t)1, (int64_t)kRadix, hist);
    hipLaunchKernelGGL((k_radix_scatter<R, true>), dim3(nt), dim3(kSortThreads), 0, st, ki, vi, ko, vo, n, shift, nt, hist);
    return hipSuccess;
  }
  hipLaunchKernelGGL(k_radix_hist<R>, dim3(nt), dim3(kSortThreads), 0, st, ki, n, shift, (int64_t)nt, (int64_t)1, hist);
  const hipError_t err = exclusive_scan<int, int>(hist, hist, (int64_t)nt * kRadix, hist + (int64_t)nt * kRadix, (int*)nullptr, st);
  if (err != hipSuccess) return err;
  hipLaunchKernelGGL((k_radix_scatter<R, false>), dim3(nt), dim3(kSortThreads), 0, st, ki, vi, ko, vo, n, shift, nt, hist);
  return hipSuccess;
}

// Sort (keys, vals) by the low `bits` bits of the key.  Ping-pongs between (k0, v0) and (k1, v1); returns
// the buffer index (0 or 1) holding the result: the parity of the passes, whatever n is.
inline int radix_sort_pairs(uint32_t* k0, uint32_t* v0, uint32_t* k1, uint32_t* v1, int64_t n, int bits, void* scratch,
                            hipStream_t st, hipError_t* err) {
  int* hist = (int*)scratch;
  int cur = 0;
  *err = hipSuccess;
  if (n == 0) return 0;
  if (n <= kSmallMax) {
    const int odd = ((bits + 7) / 8) & 1;
    hipLaunchKernelGGL(k_radix_small, dim3(1), dim3(kSmallThreads), 0, st, k0, v0, odd ? k1 : k0, odd ? v1 : v0, (int)n, bits);
    *err = hipGetLastError();
    return odd;
  }
  const int R = sort_rounds(n);
  for (int shift = 0; shift < bits; shift += 8) {
    uint32_t* ki = cur ? k1 : k0;
    uint32_t* vi = cur ? v1 : v0;
    uint32_t* ko = cur ? k0 : k1;
    uint32_t* vo = cur ? v0 : v1;
    *err = R == 1   ? radix_pass<1>(ki, vi, ko, vo, n, shift, hist, st)
           : R == 2 ? radix_pass<2>(ki, vi, ko, vo, n, shift, hist, st)
           : R == 4 ? radix_pass<4>(ki, vi, ko, vo, n, shift, hist, st)
                    : radix_pass<8>(ki, vi, ko, vo, n, shift, hist, st);
    if (*err != hipSuccess) return cur;
    cur ^= 1;
  }
  *err = hipGetLastError();
  return cur;
}

}  // namespace lsim
