// Device-wide primitives written for CDNA4 wave64: exclusive scan and a stable
// LSD radix sort of (key, value) pairs. No rocPRIM/rocThrust.
#include <hip/hip_runtime.h>

#include <utility>

#include "clue_device.h"
#include "clue_internal.h"

namespace clue_dev {

// ---------------------------------------------------------------------------
// Block reductions / scans (256 threads = 4 waves).
// ---------------------------------------------------------------------------
constexpr int kBlock = 256;
constexpr int kWavesPerBlock = kBlock / kWave;

__device__ __forceinline__ int wave_sum_i(int v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

__device__ __forceinline__ int block_excl_scan(int v, int* total) {
  return block_excl_scan<kBlock>(v, total);
}

// ---------------------------------------------------------------------------
// Exclusive scan of int32 (reduce -> scan partials -> downsweep).
// ---------------------------------------------------------------------------
constexpr int kScanItems = 16;
constexpr int kScanTile = kBlock * kScanItems;
static_assert(kScanTile == kScanTileElems, "scan workspace sizing");

__global__ __launch_bounds__(kBlock) void k_scan_reduce(const int32_t* __restrict__ in, int64_t n,
                                                        int32_t* __restrict__ partial) {
  const int64_t base = static_cast<int64_t>(blockIdx.x) * kScanTile;
  int s = 0;
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    const int64_t i = base + k * kBlock + threadIdx.x;
    if (i < n) s += in[i];
  }
  __shared__ int wsum[kWavesPerBlock];
  s = wave_sum_i(s);
  if (lane_id() == 0) wsum[threadIdx.x / kWave] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    int t = 0;
    for (int k = 0; k < kWavesPerBlock; ++k) t += wsum[k];
    partial[blockIdx.x] = t;
  }
}

// One block scans the partials in place (exclusive), in chunks with a carry.
__global__ __launch_bounds__(kBlock) void k_scan_partials(int32_t* __restrict__ partial, int64_t nb,
                                                          int32_t* __restrict__ total_out) {
  int carry = 0;
  for (int64_t base = 0; base < nb; base += kBlock) {
    const int64_t i = base + threadIdx.x;
    const int v = i < nb ? partial[i] : 0;
    int tot;
    const int ex = block_excl_scan(v, &tot);
    if (i < nb) partial[i] = carry + ex;
    carry += tot;
  }
  if (threadIdx.x == 0 && total_out) *total_out = carry;
}

__global__ __launch_bounds__(kBlock) void k_scan_down(const int32_t* in, int32_t* out, int64_t n,
                                                      const int32_t* __restrict__ partial) {
  const int64_t base = static_cast<int64_t>(blockIdx.x) * kScanTile + threadIdx.x * kScanItems;
  int v[kScanItems];
  int s = 0;
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    const int64_t i = base + k;
    v[k] = i < n ? in[i] : 0;
    s += v[k];
  }
  int tot;
  int run = block_excl_scan(s, &tot) + partial[blockIdx.x];
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    const int64_t i = base + k;
    if (i < n) out[i] = run;
    run += v[k];
  }
}

// One block for n <= kScanTile: the downsweep with no partials, and the total
// (small scans, such as one event's tiles or a batch's per-event seed counts,
// then take one launch instead of three).
__global__ __launch_bounds__(kBlock) void k_scan_single(const int32_t* in, int32_t* out, int64_t n,
                                                        int32_t* __restrict__ total_out) {
  const int64_t base = static_cast<int64_t>(threadIdx.x) * kScanItems;
  int v[kScanItems];
  int s = 0;
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    const int64_t i = base + k;
    v[k] = i < n ? in[i] : 0;
    s += v[k];
  }
  int tot;
  int run = block_excl_scan(s, &tot);
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    const int64_t i = base + k;
    if (i < n) out[i] = run;
    run += v[k];
  }
  if (threadIdx.x == 0 && total_out) *total_out = tot;
}

void scan_exclusive(const int32_t* in, int32_t* out, int64_t n, int32_t* temp, int32_t* total,
                    hipStream_t s) {
  if (n <= 0) return;
  if (n <= kScanTile) {
    hipLaunchKernelGGL(k_scan_single, dim3(1), dim3(kBlock), 0, s, in, out, n, total);
    return;
  }
  const int64_t nb = (n + kScanTile - 1) / kScanTile;
  hipLaunchKernelGGL(k_scan_reduce, dim3(static_cast<unsigned>(nb)), dim3(kBlock), 0, s, in, n, temp);
  hipLaunchKernelGGL(k_scan_partials, dim3(1), dim3(kBlock), 0, s, temp, nb, total);
  hipLaunchKernelGGL(k_scan_down, dim3(static_cast<unsigned>(nb)), dim3(kBlock), 0, s, in, out, n, temp);
}

// ---------------------------------------------------------------------------
// Stable LSD radix sort of (uint32 key, int32 value), digits of up to 10 bits.
//
// Each block owns a contiguous range of at most kRsTile keys; each of its sixteen
// waves owns a contiguous sixteenth, walked in rounds of 64 (two: a wave alone takes
// 23 us for the sixteen rounds of a 256-thread block). Within a round, lanes with the
// same digit are found with one ballot per digit bit and ranked by lane order;
// per-wave digit counters live in LDS. Ranges, rounds and lanes are all visited in
// index order, so the pass is stable. Between the counts and the placement one
// workgroup per digit scans the digit's counts over the blocks; the digits' totals
// are scanned by every placing block for itself.
// ---------------------------------------------------------------------------
constexpr int kRsWaves = 16;
constexpr int kRsBlock = kRsWaves * kWave;
constexpr int kRsTile = kRsTileKeys;
constexpr int kRsRounds = kRsTile / kRsBlock;
static_assert(kRsMaxBins <= kRsBlock, "one digit per thread in the scan of the totals");

__device__ __forceinline__ void rs_range(const Chunk* chunks, int64_t n, int64_t* begin,
                                         int64_t* end) {
  if (chunks) {
    *begin = chunks[blockIdx.x].begin;
    *end = chunks[blockIdx.x].end;
  } else {
    *begin = static_cast<int64_t>(blockIdx.x) * kRsTile;
    *end = *begin + kRsTile < n ? *begin + kRsTile : n;
  }
}

// hist[digit][block]
__global__ __launch_bounds__(kBlock) void k_rs_hist(const uint32_t* __restrict__ keys, int64_t n,
                                                    const Chunk* __restrict__ chunks, int shift,
                                                    int bits, int32_t* __restrict__ hist) {
  __shared__ int cnt[kRsMaxBins];
  const int bins = 1 << bits;
  for (int k = threadIdx.x; k < bins; k += kBlock) cnt[k] = 0;
  __syncthreads();
  int64_t b, e;
  rs_range(chunks, n, &b, &e);
  for (int64_t i = b + threadIdx.x; i < e; i += kBlock)
    atomicAdd(&cnt[(keys[i] >> shift) & (bins - 1)], 1);
  __syncthreads();
  for (int d = threadIdx.x; d < bins; d += kBlock)
    hist[static_cast<int64_t>(d) * gridDim.x + blockIdx.x] = cnt[d];
}

// One workgroup per digit: its counts become an exclusive scan over the blocks, and
// total[digit] their sum.
__global__ __launch_bounds__(kBlock) void k_rs_rows(int32_t* __restrict__ hist, int64_t nblocks,
                                                    int32_t* __restrict__ total) {
  int32_t* row = hist + static_cast<int64_t>(blockIdx.x) * nblocks;
  int carry = 0;
  for (int64_t base = 0; base < nblocks; base += kBlock * 4) {
    int v[4], sum = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int64_t i = base + threadIdx.x * 4 + k;
      v[k] = i < nblocks ? row[i] : 0;
      sum += v[k];
    }
    int tot;
    int run = carry + block_excl_scan(sum, &tot);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int64_t i = base + threadIdx.x * 4 + k;
      if (i < nblocks) row[i] = run;
      run += v[k];
    }
    carry += tot;
  }
  if (threadIdx.x == 0) total[blockIdx.x] = carry;
}

// MaxBits: room for the counters (16 KB of LDS at 8 bits, 64 KB at 10).
template <int MaxBits>
__global__ __launch_bounds__(kRsBlock) void k_rs_scatter(
    const uint32_t* __restrict__ kin, const int32_t* __restrict__ vin, uint32_t* __restrict__ kout,
    int32_t* __restrict__ vout, int64_t n_out, int64_t n, const Chunk* __restrict__ chunks,
    int shift, int bits,
    const int32_t* __restrict__ rows, const int32_t* __restrict__ total) {
  __shared__ int cnt[kRsWaves << MaxBits];  // [kRsWaves][bins]
  const int bins = 1 << bits;
  const int w = threadIdx.x / kWave;
  const int l = lane_id();
  int64_t b, e;
  rs_range(chunks, n, &b, &e);
  const int64_t wb = b + static_cast<int64_t>(w) * (kRsTile / kRsWaves);
  uint32_t key[kRsRounds];
  uint64_t peers[kRsRounds];
#pragma unroll
  for (int r = 0; r < kRsRounds; ++r) {
    const int64_t i = wb + r * kWave + l;
    key[r] = i < e ? kin[i] : 0u;
  }
  const int d0 = static_cast<int>(threadIdx.x);
  const int mine = d0 < bins ? total[d0] : 0;
  const int row = d0 < bins ? rows[static_cast<int64_t>(d0) * gridDim.x + blockIdx.x] : 0;
  for (int k = threadIdx.x; k < kRsWaves * bins; k += kRsBlock) cnt[k] = 0;
  int all;
  const int before = block_excl_scan<kRsBlock>(mine, &all);  // keys of smaller digits
  const uint64_t lt = lanemask_lt();
  int* my = cnt + w * bins;
  // Per-wave digit counts.
#pragma unroll
  for (int r = 0; r < kRsRounds; ++r) {
    const bool valid = wb + r * kWave + l < e;
    const uint32_t dgt = (key[r] >> shift) & (bins - 1);
    peers[r] = match_peers(dgt, bits, valid);
    if (valid && (peers[r] & lt) == 0) my[dgt] += __popcll(peers[r]);
    __builtin_amdgcn_wave_barrier();
  }
  __syncthreads();
  // Per digit: global offset of this block, then the waves in order.
  if (d0 < bins) {
    int run = before + row;
#pragma unroll
    for (int k = 0; k < kRsWaves; ++k) {
      const int c = cnt[k * bins + d0];
      cnt[k * bins + d0] = run;
      run += c;
    }
  }
  __syncthreads();
  // Place keys.
#pragma unroll
  for (int r = 0; r < kRsRounds; ++r) {
    const int64_t i = wb + r * kWave + l;
    const bool valid = i < e;
    const uint32_t dgt = (key[r] >> shift) & (bins - 1);
    int pos = 0;
    if (valid) pos = my[dgt] + __popcll(peers[r] & lt);
    __builtin_amdgcn_wave_barrier();
    if (valid && (peers[r] & lt) == 0) my[dgt] += __popcll(peers[r]);
    __builtin_amdgcn_wave_barrier();
    if (valid) {
      kout[pos] = key[r];
      if (pos < n_out) vout[pos] = vin ? vin[i] : static_cast<int32_t>(i);
    }
  }
}

void radix_sort_pairs(uint32_t* k0, int32_t* v0, uint32_t* k1, int32_t* v1, int64_t n, int key_bits,
                      int32_t* hist, bool counted, const Chunk* chunks, int n_chunks,
                      int32_t* last_values, int64_t last_count, bool* in_first, hipStream_t s) {
  *in_first = true;
  if (n <= 0) return;
  const RadixPlan plan = radix_plan(key_bits);
  const unsigned nblocks =
      chunks ? static_cast<unsigned>(n_chunks) : static_cast<unsigned>((n + kRsTile - 1) / kRsTile);
  const int bins = 1 << plan.bits;
  int32_t* total = hist + static_cast<int64_t>(bins) * nblocks;
  uint32_t *ka = k0, *kb = k1;
  int32_t *va = v0, *vb = v1;
  for (int pass = 0; pass < plan.passes; ++pass) {
    const int shift = pass * plan.bits;
    const bool last = last_values && pass + 1 == plan.passes;
    if (pass > 0 || !counted)
      hipLaunchKernelGGL(k_rs_hist, dim3(nblocks), dim3(kBlock), 0, s, ka, n, chunks, shift,
                         plan.bits, hist);
    hipLaunchKernelGGL(k_rs_rows, dim3(static_cast<unsigned>(bins)), dim3(kBlock), 0, s, hist,
                       static_cast<int64_t>(nblocks), total);
    hipLaunchKernelGGL(plan.bits <= 8 ? k_rs_scatter<8> : k_rs_scatter<kRsMaxBits>, dim3(nblocks),
                       dim3(kRsBlock), 0, s, ka, pass == 0 ? nullptr : va, kb,
                       last ? last_values : vb, last ? last_count : n, n, chunks, shift, plan.bits,
                       hist, total);
    std::swap(ka, kb);
    std::swap(va, vb);
    *in_first = !*in_first;
  }
}

}  // namespace clue_dev
