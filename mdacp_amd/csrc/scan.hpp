// scan.hpp -- exclusive prefix sum on the device in one launch.  Each workgroup
// scans kScanItems items and publishes its total; it takes the sum of those
// before it by looking back over their published totals and prefixes (Merrill
// and Garland, "Single-pass Parallel Prefix Scan with Decoupled Look-back",
// 2016), 64 of them at a time.  Workgroups take their places from a counter,
// so each waits only for ones that have started.  A construction runs six
// scans; as three or four launches each (blocks, their totals, offsets, the
// sum) they were 20 of its 50 launches.
//
// What is scanned comes from a functor F:
//   long long in(i)            item i
//   void out(i, excl, v)       its exclusive prefix, and the item again
//   void total(sum)            once
#pragma once
#include "device_common.hpp"

namespace mdgpu {

constexpr int kScanThreads = 256;
constexpr int kScanPerThread = 8;
constexpr int kScanItems = kScanThreads * kScanPerThread;

// A published word: a flag (1: the workgroup's total, 2: the prefix up to its
// end), the launch's number, so that words of earlier launches do not count
// and nothing is cleared in between, and the value.
constexpr int kScanEpochBits = 20;
constexpr unsigned kScanEpochs = 1u << kScanEpochBits;

struct ScanCtx {
  unsigned long long *status;  // a word per workgroup
  unsigned *ticket;            // counts the workgroups of all launches
  unsigned base;               // its value before this launch
  unsigned epoch;              // this launch's number, 1 .. kScanEpochs - 1
};

__device__ __forceinline__ unsigned long long scan_word(unsigned flag, unsigned epoch, long long v) {
  return (unsigned long long)flag | (unsigned long long)epoch << 2 | (unsigned long long)v << (2 + kScanEpochBits);
}

// skip (optional): nothing to do when it is set (a workgroup still takes its place)
template <class F>
__global__ __launch_bounds__(kScanThreads) void k_scan(F f, long long n, ScanCtx c, const int *skip) {
  __shared__ long long wsum[kScanThreads / kWave];
  __shared__ long long before;
  __shared__ int place, skipped;
  if (threadIdx.x == 0) {
    place = (int)(atomicAdd(c.ticket, 1u) - c.base);
    skipped = skip != nullptr && *skip != 0;
  }
  __syncthreads();
  if (skipped) return;
  const int b = place, lane = threadIdx.x % kWave, wv = threadIdx.x / kWave;
  const long long first = (long long)b * kScanItems + (long long)threadIdx.x * kScanPerThread;
  long long v[kScanPerThread];
  long long sum = 0;
#pragma unroll
  for (int k = 0; k < kScanPerThread; k++) {
    v[k] = first + k < n ? f.in(first + k) : 0;
    sum += v[k];
  }
  long long inc = sum;  // inclusive over the wavefront
  for (int o = 1; o < kWave; o <<= 1) {
    const long long y = __shfl_up(inc, o, kWave);
    if (lane >= o) inc += y;
  }
  if (lane == kWave - 1) wsum[wv] = inc;
  __syncthreads();
  long long excl = inc - sum, all = 0;
#pragma unroll
  for (int k = 0; k < kScanThreads / kWave; k++) {
    if (k < wv) excl += wsum[k];
    all += wsum[k];
  }
  if (wv == 0) {
    if (lane == 0)
      __hip_atomic_store(&c.status[b], scan_word(b == 0 ? 2 : 1, c.epoch, all), __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
    long long pre = 0;
    for (int top = b - 1; top >= 0; top -= kWave) {
      const int at = top - lane;  // the nearest workgroup in lane 0
      unsigned long long w = scan_word(2, c.epoch, 0);
      if (at >= 0) do {
          w = __hip_atomic_load(&c.status[at], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        } while ((w & 3ull) == 0 || ((w >> 2) & (kScanEpochs - 1)) != c.epoch);
      const unsigned long long whole = __ballot((w & 3ull) == 2);
      const int stop = whole ? __ffsll((long long)whole) - 1 : kWave - 1;  // the nearest prefix
      long long x = lane <= stop ? (long long)(w >> (2 + kScanEpochBits)) : 0;
      for (int o = kWave / 2; o > 0; o >>= 1) x += __shfl_xor(x, o, kWave);
      pre += x;
      if (whole) break;
    }
    if (lane == 0) {
      if (b > 0)
        __hip_atomic_store(&c.status[b], scan_word(2, c.epoch, pre + all), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
      before = pre;
    }
  }
  __syncthreads();
  excl += before;
#pragma unroll
  for (int k = 0; k < kScanPerThread; k++) {
    if (first + k < n) f.out(first + k, excl, v[k]);
    excl += v[k];
  }
  if (b == (int)gridDim.x - 1 && threadIdx.x == 0) f.total(before + all);
}

// dst = exclusive prefix sums of src, *sum (optional) their total
template <class Tin, class Tout>
struct ScanArray {
  const Tin *src;
  Tout *dst;
  long long *sum;
  __device__ __forceinline__ long long in(long long i) const { return (long long)src[i]; }
  __device__ __forceinline__ void out(long long i, long long x, long long) const { dst[i] = (Tout)x; }
  __device__ __forceinline__ void total(long long t) const {
    if (sum) *sum = t;
  }
};

}  // namespace mdgpu
