// Key -> members association map (CSR) on the device: the cluster -> points map
// of get_clusters (utils/detail/get_clusters.hpp:24-49) and the event -> clusters
// map of getSampleAssociations (core/detail/Clusterer.hpp:219-241), both built by
// make_associator (data_structures/internal/MakeAssociator.hpp:15-45):
//   bins     = max key + 1;
//   members  = the indices whose key is >= 0, grouped by key;
//   offsets  = bins + 1 boundaries.
// Members of one key are in ascending index order (a stable sort), which is the
// host map's fill order; the reference's device fill orders them by atomics.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>

#include "clue_assoc.h"
#include "clue_device.h"

namespace clue_dev {
namespace {

constexpr int kBlock = 256;

// Largest key and number of keys >= 0 of each workgroup's share, stats[2 * block] on
// (the host combines them: results kept in one place took an atomic update per
// workgroup, 50 us for 2^20 keys).
__global__ __launch_bounds__(kBlock) void k_assoc_stats(const int32_t* __restrict__ keys, int n,
                                                        int32_t* __restrict__ stats) {
  __shared__ int32_t smax[kBlock / kWave], scnt[kBlock / kWave];
  int mx = INT32_MIN, cnt = 0;
#pragma unroll 8
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x; i < n;
       i += static_cast<int64_t>(gridDim.x) * kBlock) {
    const int k = keys[i];
    mx = max(mx, k);
    cnt += k >= 0 ? 1 : 0;
  }
  mx = wave_max_i(mx);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) cnt += __shfl_xor(cnt, off, 64);
  const int w = threadIdx.x / kWave;
  if (lane_id() == 0) {
    smax[w] = mx;
    scnt[w] = cnt;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    int m = INT32_MIN, c = 0;
    for (int k = 0; k < kBlock / kWave; ++k) {
      m = max(m, smax[k]);
      c += scnt[k];
    }
    stats[2 * blockIdx.x] = m;
    stats[2 * blockIdx.x + 1] = c;
  }
}

// Sort key: the key itself, negative keys after every bin; with the first digits'
// counts per block of the sort.
__global__ __launch_bounds__(kBlock) void k_assoc_keys(const int32_t* __restrict__ keys, int n,
                                                       int bins, uint32_t* __restrict__ k0,
                                                       int digit_bits, int32_t* __restrict__ hist) {
  __shared__ int32_t cnt[kRsMaxBins];
  const int digits = 1 << digit_bits;
  for (int d = threadIdx.x; d < digits; d += kBlock) cnt[d] = 0;
  __syncthreads();
  const int64_t b = static_cast<int64_t>(blockIdx.x) * kRsTileKeys;
  const int64_t e = b + kRsTileKeys < n ? b + kRsTileKeys : n;
#pragma unroll 8
  for (int64_t i = b + threadIdx.x; i < e; i += kBlock) {
    const int k = keys[i];
    const uint32_t key = static_cast<uint32_t>(k >= 0 ? k : bins);
    k0[i] = key;
    atomicAdd(&cnt[key & (digits - 1)], 1);
  }
  __syncthreads();
  for (int d = threadIdx.x; d < digits; d += kBlock)
    hist[static_cast<int64_t>(d) * gridDim.x + blockIdx.x] = cnt[d];
}

// offsets[b] = first sorted position whose key is >= b (lower bound), b in [0, bins].
__global__ __launch_bounds__(kBlock) void k_assoc_offsets(const uint32_t* __restrict__ sk, int n,
                                                          int bins, int32_t* __restrict__ offsets) {
  const int b = blockIdx.x * kBlock + threadIdx.x;
  if (b > bins) return;
  int lo = 0, hi = n;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (static_cast<int>(sk[mid]) < b)
      lo = mid + 1;
    else
      hi = mid;
  }
  offsets[b] = lo;
}

}  // namespace

int64_t assoc_hist_elems(int64_t n) {
  return radix_hist_elems((n + kRsTileKeys - 1) / kRsTileKeys, kRsMaxBits);
}

hipError_t assoc_stats(const int32_t* keys, int n, int32_t* stats_dev, int* blocks, hipStream_t s) {
  *blocks = static_cast<int>(
      std::min<int64_t>((static_cast<int64_t>(n) + 8 * kBlock - 1) / (8 * kBlock), kAssocStatBlocks));
  if (n > 0)
    hipLaunchKernelGGL(k_assoc_stats, dim3(*blocks), dim3(kBlock), 0, s, keys, n, stats_dev);
  return hipGetLastError();
}

hipError_t assoc_build(const int32_t* keys, int n, int bins, const AssocScratch& w,
                       int32_t* offsets, int32_t* members, int n_members, hipStream_t s) {
  if (n > 0) {
    int bits = 0;
    while ((int64_t(1) << bits) <= bins) ++bits;  // keys lie in [0, bins]
    const unsigned blocks =
        static_cast<unsigned>((static_cast<int64_t>(n) + kRsTileKeys - 1) / kRsTileKeys);
    hipLaunchKernelGGL(k_assoc_keys, dim3(blocks), dim3(kBlock), 0, s, keys, n, bins, w.k0,
                       radix_plan(bits).bits, w.hist);
    bool in_first = true;
    // The last pass leaves the members, which are the sorted values but for the
    // negative keys' behind them, where the caller wants them.
    radix_sort_pairs(w.k0, w.v0, w.k1, w.v1, n, bits, w.hist, true, nullptr, 0, members, n_members,
                     &in_first, s);
    const uint32_t* sk = in_first ? w.k0 : w.k1;
    hipLaunchKernelGGL(k_assoc_offsets, dim3((bins + 1 + kBlock - 1) / kBlock), dim3(kBlock), 0,
                       s, sk, n, bins, offsets);
  } else {
    hipLaunchKernelGGL(k_assoc_offsets, dim3(1), dim3(kBlock), 0, s, w.k0, 0, 0, offsets);
  }
  return hipGetLastError();
}

}  // namespace clue_dev
