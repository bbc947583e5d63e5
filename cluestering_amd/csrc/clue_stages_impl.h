// The five CLUE stages on gfx950:
//   (a) tile construction: per-event extremes, tile keys, stable radix sort into a
//       tile-sorted SoA copy, tile offsets, work items;
//   (b) local density and (c) nearest-higher: one wave per work item (up to 64
//       points of one tile, one lane each) walks the union of the lanes' search
//       boxes in the reference's lexicographic tile order; candidates are
//       wave-uniform and come through the scalar cache. With the default tags,
//       (c) instead scans each tile's candidates in Hilbert-ordered blocks and
//       skips the blocks that cannot hold the answer (its result does not
//       depend on the visiting order);
//   (d) seeds, numbered by an exclusive scan in input order;
//   (e) follower labels: a few hops along the links, or pointer jumping in LDS, then a
//       chase to the seed.
// Launches of few points have (b) and (c) done by teams of waves (clue_team.h).
//
// Semantics follow the reference's serial backend:
//   geometry  core/detail/SetupTiles.hpp:23-57, core/detail/ComputeTiles.hpp:17-37
//   bins/box  data_structures/internal/TilesView.hpp:38-104
//   density   core/detail/ClusteringKernels.hpp:29-140
//   NH        core/detail/ClusteringKernels.hpp:142-291
//   seeds     core/detail/ClusteringKernels.hpp:293-343
//
// Included by one translation unit per point type (clue_stages_f32.hip,
// clue_stages_f64.hip), which compile in parallel.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <limits>
#include <type_traits>

#include "clue_device.h"
#include "clue_internal.h"

namespace clue_dev {

constexpr int kBlock = 256;
constexpr int kWaves = kBlock / kWave;
// The neighbour stages take 1 to 16 waves per workgroup (a tuning choice): a
// workgroup runs on one CU, so its consecutive work items (neighbouring tiles)
// share that CU's scalar cache, while smaller workgroups spread more evenly.
constexpr int kMaxNeighbourBlock = 1024;

enum { M_EUCLID = 0, M_WEUCLID = 1, M_PERIODIC = 2, M_MANHATTAN = 3, M_CHEBYSHEV = 4,
       M_WCHEBYSHEV = 5, M_MAHALANOBIS = 6, M_PERIODIC_LAST = kMetricPeriodicLast };
enum { K_FLAT = 0, K_EXP = 1, K_GAUSS = 2 };

// Workgroups are dispatched round-robin over the 8 XCDs (block b runs on XCD
// b mod 8), each with its own L2. The neighbour stages deal chunks of G = 2^k
// consecutive work-item blocks to the XCDs in turn: an XCD's L2 then sees runs
// of neighbouring tiles, while the work stays spread evenly over the XCDs (a
// contiguous eighth per XCD leaves them unequal, since events differ in cost).
// Blocks past the last whole round of chunks keep their index.
constexpr int kXcds = 8;
__device__ __forceinline__ int xcd_block(int b, int nb, int log2_chunk) {
  if (log2_chunk < 0) return b;
  const int round = kXcds << log2_chunk;
  if (b >= nb / round * round) return b;
  const int xcd = b % kXcds;
  const int k = b / kXcds;  // b is the k-th block on its XCD
  return ((((k >> log2_chunk) * kXcds) + xcd) << log2_chunk) + (k & ((1 << log2_chunk) - 1));
}

// Work items of a neighbour stage. In the grid form each wave takes one item (its
// workgroup mapped by xcd_block). In the persistent form (rp.persistent waves per
// CU) waves pull items from device queues: the item space is dealt to the XCDs in
// chunks of 2^k items, as xcd_block deals workgroups, each XCD counts off its own
// chunks (ctl[x], zeroed by k_tile_setup), and a wave whose XCD has no items left
// takes them from the next XCDs in turn. A queue's items come in increasing order,
// so a wave stops once every one of the eight counters has passed the last item.
constexpr int kQueueDensity = 8;  // counters in the n_items block: density
constexpr int kQueueNh = 16;      // nearest-higher
constexpr int kQueueWords = 24;   // words of the block k_tile_setup zeroes
struct ItemCursor {
  int32_t* ctl;
  int n;
  int log2c;
  int home;

  template <class P>
  __device__ ItemCursor(int32_t* n_items, int queue, const P& rp)
      : ctl(n_items + queue), n(*n_items), log2c(rp.xcd_chunk_log2), home(blockIdx.x % kXcds) {}

  __device__ int pull() {
    for (int t = 0; t < kXcds; ++t) {
      const int x = (home + t) & (kXcds - 1);
      int j = 0;
      if (lane_id() == 0) j = atomicAdd(&ctl[x], 1);
      j = uniform(j);
      const int item = log2c < 0 ? j * kXcds + x
                                 : ((x + kXcds * (j >> log2c)) << log2c) + (j & ((1 << log2c) - 1));
      if (item < n) return item;
    }
    return -1;
  }
};

template <int M>
struct MetricTraits {
  // Metrics ending in a square root are compared through the squared sum against
  // the largest float whose correctly rounded square root is within the radius.
  static constexpr bool kSqrt =
      (M == M_EUCLID || M == M_WEUCLID || M == M_PERIODIC || M == M_PERIODIC_LAST ||
       M == M_MAHALANOBIS);
};

// ---------------------------------------------------------------------------
// (a1) Per-event coordinate extremes (ComputeTiles.hpp:17-36). NaN coordinates
// are skipped, as the reference's std::max/std::min fold skips them.
// ---------------------------------------------------------------------------
template <class T>
struct CoordPtrs {
  const T* x[kMaxDim];
};

// One workgroup per chunk, or per `group` consecutive chunks of an event (at the first
// of them), each with its own result: a common one took as many atomic updates of one
// address as there are workgroups (18 us for 2^20 points, 9 us this way).
template <class T>
__global__ __launch_bounds__(kBlock) void k_extremes(CoordPtrs<T> c, int D,
                                                     const LoneEvent lone,
                                                     Chunk* __restrict__ chunks,
                                                     EventDesc* __restrict__ events, int group,
                                                     typename FloatBits<T>::Int* __restrict__ ext) {
  using I = typename FloatBits<T>::Int;
  constexpr I kHi = std::numeric_limits<I>::max(), kLo = std::numeric_limits<I>::min();
  Chunk ch;
  if (lone.is) {  // its descriptors, for the stages that follow
    ch = lone_chunk(lone, blockIdx.x);
    if (threadIdx.x == 0) {
      chunks[blockIdx.x] = ch;
      if (blockIdx.x == 0) events[0] = lone.ev;
    }
  } else {
    ch = chunks[blockIdx.x];
  }
  int end = ch.end;
  if (group > 1) {
    const EventDesc ev = lone.is ? lone.ev : events[ch.event];
    if ((ch.begin - ev.p_off) / kPointChunk % group != 0) return;
    end = min(ev.p_off + ev.n, ch.begin + group * kPointChunk);
  }
  __shared__ I smin[kWaves][kMaxDim], smax[kWaves][kMaxDim];
  const int w = threadIdx.x / kWave;
  for (int d = 0; d < D; ++d) {
    I lo = kHi, hi = kLo;
#pragma unroll 8
    for (int i = ch.begin + threadIdx.x; i < end; i += kBlock) {
      const T v = c.x[d][i];
      const I o = float_to_ordered(v);
      const bool ok = v == v;
      lo = (ok && o < lo) ? o : lo;
      hi = (ok && o > hi) ? o : hi;
    }
    lo = wave_min_i(lo);
    hi = wave_max_i(hi);
    if (lane_id() == 0) {
      smin[w][d] = lo;
      smax[w][d] = hi;
    }
  }
  __syncthreads();
  if (threadIdx.x < D) {
    const int d = threadIdx.x;
    I lo = kHi, hi = kLo;
    for (int k = 0; k < kWaves; ++k) {
      lo = smin[k][d] < lo ? smin[k][d] : lo;
      hi = smax[k][d] > hi ? smax[k][d] : hi;
    }
    ext[(static_cast<int64_t>(blockIdx.x) * D + d) * 2 + 0] = lo;
    ext[(static_cast<int64_t>(blockIdx.x) * D + d) * 2 + 1] = hi;
  }
}

template <class T>
__device__ __forceinline__ GeoT<T> event_geo(const T* geo, const RunParamsT<T>& rp, int e,
                                             int nper) {
  GeoT<T> g;
  g.D = rp.D;
  g.nper = nper;
  g.mn = geo + static_cast<int64_t>(e) * 3 * rp.D;
  g.mx = g.mn + rp.D;
  g.side = g.mn + 2 * rp.D;
  g.wrapped = rp.wrapped;
  return g;
}

// ---------------------------------------------------------------------------
// (a2) Tile key of every point: t_base + sum_d nper^(D-1-d) * bin_d
// (TilesView.hpp:54-64). Every workgroup takes its event's extremes and geometry from
// the chunks' results, side = (max - min) / nper (ComputeTiles.hpp:33-34); the
// event's first chunk stores the geometry, geo[e] = {mn[D], mx[D], side[D]}. The keys'
// lowest digits are counted as they are made: the histogram of the first sort pass.
// A thread has two points of the chunk, whose loads it issues together; with 256
// threads of eight points, one after the other, the chain of loads set the time
// (16,384 points in 2-D: 8.8 -> 6.2 us; 20,011 in 6-D: 17.6 -> 8.3; 2^20 in 2-D: 12.2 ->
// 9.1).
// ---------------------------------------------------------------------------
// Where the sort's blocks are not the chunks (small events, sort_by_chunk), nothing is
// counted and a workgroup has 256 threads.
template <class T, bool Count>
__global__ __launch_bounds__(Count ? 1024 : 256) void k_tile_keys(
    CoordPtrs<T> c, const RunParamsT<T> rp, const Chunk* __restrict__ chunks,
    const EventDesc* __restrict__ events, int group,
    const typename FloatBits<T>::Int* __restrict__ ext, T* __restrict__ geo,
    uint32_t* __restrict__ keys, int digit_bits, int32_t* __restrict__ hist) {
  using I = typename FloatBits<T>::Int;
  constexpr I kHi = std::numeric_limits<I>::max(), kLo = std::numeric_limits<I>::min();
  constexpr int kKeysBlock = Count ? 1024 : 256;
  constexpr int kKeysWaves = kKeysBlock / kWave;
  __shared__ int32_t cnt[Count ? kRsMaxBins : 1];
  __shared__ I smin[kKeysWaves][kMaxDim], smax[kKeysWaves][kMaxDim];
  __shared__ T sgeo[3 * kMaxDim];
  const Chunk ch = chunks[blockIdx.x];
  const EventDesc ev = events[ch.event];
  const int D = rp.D;
  const int bins = Count ? 1 << digit_bits : 0;
  for (int k = threadIdx.x; k < bins; k += kKeysBlock) cnt[k] = 0;
  const int first = static_cast<int>(blockIdx.x) - (ch.begin - ev.p_off) / kPointChunk;
  const int n_ext = ((ev.n + kPointChunk - 1) / kPointChunk + group - 1) / group;
  const int w = threadIdx.x / kWave;
  for (int d = 0; d < D; ++d) {
    I lo = kHi, hi = kLo;
    for (int k = threadIdx.x; k < n_ext; k += kKeysBlock) {
      const int64_t q = (static_cast<int64_t>(first + k * group) * D + d) * 2;
      const I l = ext[q], h = ext[q + 1];
      lo = l < lo ? l : lo;
      hi = h > hi ? h : hi;
    }
    lo = wave_min_i(lo);
    hi = wave_max_i(hi);
    if (lane_id() == 0) {
      smin[w][d] = lo;
      smax[w][d] = hi;
    }
  }
  __syncthreads();
  if (threadIdx.x < D) {
    const int d = threadIdx.x;
    I lo = kHi, hi = kLo;
    for (int k = 0; k < kKeysWaves; ++k) {
      lo = smin[k][d] < lo ? smin[k][d] : lo;
      hi = smax[k][d] > hi ? smax[k][d] : hi;
    }
    const T mn = lo == kHi ? std::numeric_limits<T>::max() : ordered_to_float(lo);
    const T mx = hi == kLo ? std::numeric_limits<T>::lowest() : ordered_to_float(hi);
    const T side = (mx - mn) / static_cast<T>(ev.nper);
    sgeo[d] = mn;
    sgeo[D + d] = mx;
    sgeo[2 * D + d] = side;
    if (ch.begin == ev.p_off) {
      T* g = geo + static_cast<int64_t>(ch.event) * 3 * D;
      g[d] = mn;
      g[D + d] = mx;
      g[2 * D + d] = side;
    }
  }
  __syncthreads();
  GeoT<T> g;
  g.D = D;
  g.nper = ev.nper;
  g.mn = sgeo;
  g.mx = sgeo + D;
  g.side = sgeo + 2 * D;
  g.wrapped = rp.wrapped;
  constexpr int kPer = 2;
  for (int i0 = ch.begin + static_cast<int>(threadIdx.x); i0 < ch.end; i0 += kPer * kKeysBlock) {
    int t[kPer] = {};
    for (int d = 0; d < D; ++d) {
      T v[kPer];
#pragma unroll
      for (int u = 0; u < kPer; ++u) v[u] = c.x[d][min(i0 + u * kKeysBlock, ch.end - 1)];
#pragma unroll
      for (int u = 0; u < kPer; ++u) t[u] = t[u] * ev.nper + get_bin(g, v[u], d);
    }
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      const int i = i0 + u * kKeysBlock;
      if (i >= ch.end) break;
      const uint32_t key = static_cast<uint32_t>(ev.t_base + t[u]);
      keys[i] = key;
      if constexpr (Count) atomicAdd(&cnt[key & (bins - 1)], 1);
    }
  }
  if constexpr (!Count) return;
  __syncthreads();
  for (int k = threadIdx.x; k < bins; k += kKeysBlock)
    hist[static_cast<int64_t>(k) * gridDim.x + blockIdx.x] = cnt[k];
}

// ---------------------------------------------------------------------------
// (a3) Gather the tile-sorted SoA copy and the tile offsets. toff[k] is the first
// sorted position whose key is >= k, so tile k spans [toff[k], toff[k+1]).
// ---------------------------------------------------------------------------
template <class T>
struct GatherArgs {
  PointArraysT<T> in;
  SortedArraysT<T> out;
  int64_t cs;  // column stride of the sorted coordinate block
};

template <class T>
__global__ __launch_bounds__(kBlock) void k_gather(const GatherArgs<T> a, const RunParamsT<T> rp,
                                                   const uint32_t* __restrict__ keys,
                                                   const int32_t* __restrict__ perm, int n,
                                                   int n_tiles_total, int32_t* __restrict__ toff,
                                                   uint32_t* __restrict__ bits) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n) return;
  if (s < (n + 31) / 32) bits[s] = 0u;  // no seeds yet (k_results)
  const int i = perm[s];
  for (int d = 0; d < rp.D; ++d) a.out.x[d][s] = a.in.x[d][i];
  const T wi = a.in.w[i];
  a.out.w[s] = wi;
  if (a.out.fw) a.out.fw[s] = rp.kp0 * wi;  // flat kernel: K * w for j != i
  if (rp.has_sigma)
    for (int d = 0; d < rp.D; ++d) a.out.sigma[d][s] = a.in.sigma[d][i];
  if (rp.has_u) a.out.u[s] = a.in.u[i];
  a.out.tag[s] = rp.has_tags ? a.in.tags[i] : static_cast<uint32_t>(i);
  a.out.perm[s] = i;
  const int key = static_cast<int>(keys[s]);
  const int prev = s == 0 ? -1 : static_cast<int>(keys[s - 1]);
  for (int k = prev + 1; k <= key; ++k) toff[k] = s;
  if (s == n - 1)
    for (int k = key + 1; k <= n_tiles_total; ++k) toff[k] = n;
}

// ---------------------------------------------------------------------------
// (a1-a3 fused) One workgroup per event when every event of the batch has at
// most kEvtMaxTiles tiles: extremes and geometry, tile ids, a stable counting
// sort by tile into the sorted SoA copy and the tile offsets, all in one
// kernel. Same results as k_extremes + k_tile_keys + the radix
// sort + k_gather: the extremes are the same ordered-integer min/max (NaN
// skipped), the bins the same get_bin, and the order (tile, input index).
// Each wave owns a contiguous sixteenth of the event, walked in
// rounds of 64; lanes with the same tile are ranked by ballot, per-wave tile
// counters live in LDS, and waves, rounds and lanes go in index order, so the
// sort is stable. Events are taken largest first (order[]).
// ---------------------------------------------------------------------------
constexpr int kEvtWaves = 16;
constexpr int kEvtBlock = kEvtWaves * kWave;
static_assert(kEvtMaxTiles <= kEvtBlock, "one tile per thread in the offset scan");

// Rounds of 64 points whose loads a wave issues together (memory-level
// parallelism; the rounds are still ranked in order).
constexpr int kEvtRounds = 4;

template <int D, class T>
__global__ __launch_bounds__(kEvtBlock) void k_event_tiles(
    const RunParamsT<T> rp, const EventDesc* __restrict__ events,
    const int32_t* __restrict__ order, const PointArraysT<T> in, const SortedArraysT<T> out,
    T* __restrict__ geo,
    int32_t* __restrict__ toff, int32_t* __restrict__ iperm, int n_tiles_total, int n_total) {
  using I = typename FloatBits<T>::Int;
  constexpr I kHi = std::numeric_limits<I>::max(), kLo = std::numeric_limits<I>::min();
  __shared__ int32_t cnt[kEvtWaves][kEvtMaxTiles];
  __shared__ I red[kEvtWaves][2 * D];
  __shared__ T sgeo[3 * D];
  __shared__ int32_t wsum[kEvtWaves];
  const int e = order[blockIdx.x];
  const EventDesc ev = events[e];
  const int w = threadIdx.x / kWave;
  const int lane = lane_id();
  const int b0 = ev.p_off, n = ev.n;

  // Extremes (ComputeTiles.hpp:17-36) and geometry (:33-34).
#pragma unroll
  for (int d = 0; d < D; ++d) {
    I lo = kHi, hi = kLo;
#pragma unroll 4
    for (int k = threadIdx.x; k < n; k += kEvtBlock) {
      const T v = in.x[d][b0 + k];
      const I o = float_to_ordered(v);
      const bool ok = v == v;  // NaN coordinates are skipped
      lo = (ok && o < lo) ? o : lo;
      hi = (ok && o > hi) ? o : hi;
    }
    lo = wave_min_i(lo);
    hi = wave_max_i(hi);
    if (lane == 0) {
      red[w][2 * d] = lo;
      red[w][2 * d + 1] = hi;
    }
  }
  __syncthreads();
  if (threadIdx.x < D) {
    const int d = threadIdx.x;
    I lo = kHi, hi = kLo;
    for (int k = 0; k < kEvtWaves; ++k) {
      lo = red[k][2 * d] < lo ? red[k][2 * d] : lo;
      hi = red[k][2 * d + 1] > hi ? red[k][2 * d + 1] : hi;
    }
    const T mn = lo == kHi ? std::numeric_limits<T>::max() : ordered_to_float(lo);
    const T mx = hi == kLo ? std::numeric_limits<T>::lowest() : ordered_to_float(hi);
    const T side = (mx - mn) / static_cast<T>(ev.nper);
    sgeo[d] = mn;
    sgeo[D + d] = mx;
    sgeo[2 * D + d] = side;
    T* gq = geo + static_cast<int64_t>(e) * 3 * D;
    gq[d] = mn;
    gq[D + d] = mx;
    gq[2 * D + d] = side;
  }
  if (static_cast<int>(threadIdx.x) < ev.ntiles)
#pragma unroll
    for (int k = 0; k < kEvtWaves; ++k) cnt[k][threadIdx.x] = 0;
  __syncthreads();
  GeoT<T> g;
  g.D = D;
  g.nper = ev.nper;
  g.mn = sgeo;
  g.mx = sgeo + D;
  g.side = sgeo + 2 * D;
  g.wrapped = rp.wrapped;
  // Tile id (TilesView.hpp:54-64) of the point with coordinates x.
  auto tile_of = [&](const T (&x)[D]) {
    int t = 0;
#pragma unroll
    for (int d = 0; d < D; ++d) t = t * g.nper + get_bin(g, x[d], d);
    return static_cast<uint32_t>(t);
  };

  int bits = 0;
  while ((1 << bits) < ev.ntiles) ++bits;
  const int per_wave = (n + kEvtWaves - 1) / kEvtWaves;
  const int wb = w * per_wave;
  const int we = min(n, wb + per_wave);
  const uint64_t lt = lanemask_lt();
  // Per-wave tile counts (LDS atomics; by ballots, as the ranks below, the kernel
  // took 1,010 us on the 4096-event batch, against 973).
  for (int k0 = wb; k0 < we; k0 += kWave * kEvtRounds) {
    uint32_t t[kEvtRounds];
    bool valid[kEvtRounds];
#pragma unroll
    for (int u = 0; u < kEvtRounds; ++u) {
      const int k = k0 + u * kWave + lane;
      valid[u] = k < we;
      T x[D];
#pragma unroll
      for (int d = 0; d < D; ++d) x[d] = valid[u] ? in.x[d][b0 + k] : T(0);
      t[u] = valid[u] ? tile_of(x) : 0u;
    }
#pragma unroll
    for (int u = 0; u < kEvtRounds; ++u)
      if (valid[u]) atomicAdd(&cnt[w][t[u]], 1);
  }
  __syncthreads();
  // Tile offsets: exclusive scan over tiles (one per thread), then each wave's
  // first position within each tile.
  {
    const int t = threadIdx.x;
    int tot = 0;
    if (t < ev.ntiles)
      for (int k = 0; k < kEvtWaves; ++k) tot += cnt[k][t];
    int incl = tot;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
      const int y = __shfl_up(incl, off, 64);
      if (lane >= off) incl += y;
    }
    if (lane == kWave - 1) wsum[w] = incl;
    __syncthreads();
    int before = 0;
    for (int k = 0; k < w; ++k) before += wsum[k];
    const int base = before + incl - tot;
    if (t < ev.ntiles) {
      toff[ev.t_base + t] = b0 + base;
      int run = base;
      for (int k = 0; k < kEvtWaves; ++k) {
        const int c = cnt[k][t];
        cnt[k][t] = run;
        run += c;
      }
    }
    if (t == 0 && ev.t_base + ev.ntiles == n_tiles_total) toff[n_tiles_total] = n_total;
  }
  __syncthreads();
  // Stable placement: rounds in order, lanes ranked by ballot. Only the
  // permutation is scattered (perm[s] = i, and iperm[i] = s in input order);
  // the sorted columns are then gathered in sorted order, so their writes are
  // whole lines instead of one scattered word per column.
  for (int k0 = wb; k0 < we; k0 += kWave * kEvtRounds) {
    uint32_t t[kEvtRounds];
    bool valid[kEvtRounds];
#pragma unroll
    for (int u = 0; u < kEvtRounds; ++u) {
      const int k = k0 + u * kWave + lane;
      valid[u] = k < we;
      T x[D];
#pragma unroll
      for (int d = 0; d < D; ++d) x[d] = valid[u] ? in.x[d][b0 + k] : T(0);
      t[u] = valid[u] ? tile_of(x) : 0u;
    }
#pragma unroll
    for (int u = 0; u < kEvtRounds; ++u) {
      const uint64_t peers = match_peers(t[u], bits, valid[u]);
      int pos = 0;
      if (valid[u]) pos = cnt[w][t[u]] + __popcll(peers & lt);
      __builtin_amdgcn_wave_barrier();
      if (valid[u] && (peers & lt) == 0) cnt[w][t[u]] += __popcll(peers);
      if (valid[u]) {
        const int i = b0 + k0 + u * kWave + lane;
        out.perm[b0 + pos] = i;
        iperm[i] = b0 + pos;
      }
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");  // perm of the whole event
  __syncthreads();
#pragma unroll 4
  for (int k = threadIdx.x; k < n; k += kEvtBlock) {
    const int s = b0 + k;
    const int i = out.perm[s];
#pragma unroll
    for (int d = 0; d < D; ++d) out.x[d][s] = in.x[d][i];
    const T wt = in.w[i];
    out.w[s] = wt;
    if (out.fw) out.fw[s] = rp.kp0 * wt;  // flat kernel: K * w for j != i
    if (rp.has_sigma)
#pragma unroll
      for (int d = 0; d < D; ++d) out.sigma[d][s] = in.sigma[d][i];
    if (rp.has_u) out.u[s] = in.u[i];
    out.tag[s] = rp.has_tags ? in.tags[i] : static_cast<uint32_t>(i);
  }
}

// The same for a lone event of at most kLoneMaxPoints points: every thread has at most
// kLoneRounds of them, so each pass issues all its loads together and what a pass needs
// again stays in registers (coordinates of up to 16 bytes per point, tile ids, sorted
// positions). One workgroup waits out every load of its chain alone: the kernel
// above took 21.8 us for 5,003 points in 2-D and 9.0 for 300, this one 14.2 and 6.3.
constexpr int kLoneRounds = kLoneMaxPoints / kEvtBlock;
static_assert(kLoneMaxPoints == kLoneRounds * kEvtBlock && kLoneMaxPoints <= 1 << 15,
              "whole rounds; 16-bit positions");

template <int D, class T>
__global__ __launch_bounds__(kEvtBlock) void k_lone_tiles(
    const RunParamsT<T> rp, const EventDesc ev, EventDesc* __restrict__ events,
    const PointArraysT<T> in, const SortedArraysT<T> out, T* __restrict__ geo,
    int32_t* __restrict__ toff, int32_t* __restrict__ iperm) {
  using I = typename FloatBits<T>::Int;
  constexpr I kHi = std::numeric_limits<I>::max(), kLo = std::numeric_limits<I>::min();
  constexpr int R = kLoneRounds;
  constexpr bool kKeep = D * sizeof(T) <= 16;
  __shared__ alignas(8) int32_t cnt[kEvtWaves][kEvtMaxTiles];
  static_assert(sizeof(cnt) >= kLoneMaxPoints * sizeof(T), "a column fits the counters' space");
  __shared__ I red[kEvtWaves][2 * D];
  __shared__ T sgeo[3 * D];
  __shared__ int32_t wsum[kEvtWaves];
  if (threadIdx.x == 0) events[0] = ev;  // for the stages that follow
  const int w = threadIdx.x / kWave;
  const int lane = lane_id();
  const int n = ev.n;
  // Each wave owns a contiguous sixteenth of the event, R rounds of 64 (loads past the
  // event read its last point, which the extremes see anyway).
  const int per_wave = (n + kEvtWaves - 1) / kEvtWaves;
  const int k0 = w * per_wave + lane;
  const int we = min(n, (w + 1) * per_wave);
  const int rounds = (n + kEvtBlock - 1) / kEvtBlock;
  T x[kKeep ? D : 1][R], wt[R];
  auto load = [&](const auto* src, auto& v) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if (r >= rounds) break;
      v[r] = src[min(k0 + r * kWave, n - 1)];
    }
  };
  auto column = [&](int d) -> T (&)[R] {
    load(in.x[d], x[kKeep ? d : 0]);
    return x[kKeep ? d : 0];
  };
  if constexpr (kKeep)
#pragma unroll
    for (int d = 0; d < D; ++d) column(d);
  load(in.w, wt);
#pragma unroll
  for (int d = 0; d < D; ++d) {
    const T(&v)[R] = kKeep ? x[kKeep ? d : 0] : column(d);
    I lo = kHi, hi = kLo;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if (r >= rounds) break;
      const I o = float_to_ordered(v[r]);
      const bool ok = v[r] == v[r];  // NaN coordinates are skipped
      lo = (ok && o < lo) ? o : lo;
      hi = (ok && o > hi) ? o : hi;
    }
    lo = wave_min_i(lo);
    hi = wave_max_i(hi);
    if (lane == 0) {
      red[w][2 * d] = lo;
      red[w][2 * d + 1] = hi;
    }
  }
  if (static_cast<int>(threadIdx.x) < ev.ntiles)
#pragma unroll
    for (int k = 0; k < kEvtWaves; ++k) cnt[k][threadIdx.x] = 0;
  __syncthreads();
  if (threadIdx.x < D) {
    const int d = threadIdx.x;
    I lo = kHi, hi = kLo;
#pragma unroll
    for (int k = 0; k < kEvtWaves; ++k) {
      lo = red[k][2 * d] < lo ? red[k][2 * d] : lo;
      hi = red[k][2 * d + 1] > hi ? red[k][2 * d + 1] : hi;
    }
    const T mn = lo == kHi ? std::numeric_limits<T>::max() : ordered_to_float(lo);
    const T mx = hi == kLo ? std::numeric_limits<T>::lowest() : ordered_to_float(hi);
    const T side = (mx - mn) / static_cast<T>(ev.nper);
    sgeo[d] = geo[d] = mn;
    sgeo[D + d] = geo[D + d] = mx;
    sgeo[2 * D + d] = geo[2 * D + d] = side;
  }
  __syncthreads();
  GeoT<T> g;
  g.D = D;
  g.nper = ev.nper;
  g.mn = sgeo;
  g.mx = sgeo + D;
  g.side = sgeo + 2 * D;
  g.wrapped = rp.wrapped;
  uint32_t t[R];
#pragma unroll
  for (int r = 0; r < R; ++r) t[r] = 0u;
#pragma unroll
  for (int d = 0; d < D; ++d) {
    const T(&v)[R] = kKeep ? x[kKeep ? d : 0] : column(d);
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if (r >= rounds) break;
      t[r] = t[r] * g.nper + get_bin(g, v[r], d);
    }
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if (r >= rounds) break;
    if (k0 + r * kWave < we) atomicAdd(&cnt[w][t[r]], 1);
  }
  __syncthreads();
  {
    const int tile = threadIdx.x;
    int c[kEvtWaves], tot = 0;
#pragma unroll
    for (int k = 0; k < kEvtWaves; ++k) {
      c[k] = tile < ev.ntiles ? cnt[k][tile] : 0;
      tot += c[k];
    }
    int incl = tot;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
      const int y = __shfl_up(incl, off, 64);
      if (lane >= off) incl += y;
    }
    if (lane == kWave - 1) wsum[w] = incl;
    __syncthreads();
    int run = incl - tot;
    for (int k = 0; k < w; ++k) run += wsum[k];
    if (tile < ev.ntiles) {
      toff[tile] = run;
#pragma unroll
      for (int k = 0; k < kEvtWaves; ++k) {
        cnt[k][tile] = run;
        run += c[k];
      }
    }
    if (tile == 0) toff[ev.ntiles] = n;
  }
  __syncthreads();
  int bits = 0;
  while ((1 << bits) < ev.ntiles) ++bits;
  const uint64_t lt = lanemask_lt();
  int pos[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if (r >= rounds) break;
    const int k = k0 + r * kWave;
    const bool valid = k < we;
    const uint64_t peers = match_peers(t[r], bits, valid);
    pos[r] = 0;
    if (valid) pos[r] = cnt[w][t[r]] + __popcll(peers & lt);
    __builtin_amdgcn_wave_barrier();
    if (valid && (peers & lt) == 0) cnt[w][t[r]] += __popcll(peers);
    if (valid) iperm[k] = pos[r];
  }
  // The columns go to their sorted places through LDS (the counters' space), so that
  // global loads and stores are whole lines (gathered: 15.4 us for 5,003 points).
  auto place = [&](const auto& v, auto&& store) {
    auto* col = reinterpret_cast<std::remove_cv_t<std::remove_reference_t<decltype(v[0])>>*>(cnt);
    __syncthreads();  // the counters, or the column before, are done with
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if (r >= rounds) break;
      if (k0 + r * kWave < we) col[pos[r]] = v[r];
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int s = static_cast<int>(threadIdx.x) + r * kEvtBlock;
      if (s >= n) break;
      store(s, col[s]);
    }
  };
#pragma unroll
  for (int d = 0; d < D; ++d)
    place(kKeep ? x[kKeep ? d : 0] : column(d), [&](int s, T v) { out.x[d][s] = v; });
  place(wt, [&](int s, T v) {
    out.w[s] = v;
    if (out.fw) out.fw[s] = rp.kp0 * v;  // flat kernel: K * w for j != i
  });
  if (rp.has_sigma)
#pragma unroll
    for (int d = 0; d < D; ++d) {
      load(in.sigma[d], wt);
      place(wt, [&](int s, T v) { out.sigma[d][s] = v; });
    }
  if (rp.has_u) {
    load(in.u, wt);
    place(wt, [&](int s, T v) { out.u[s] = v; });
  }
  int index[R];
  if (rp.has_tags) {
    uint32_t tags[R];
    load(in.tags, tags);
    place(tags, [&](int s, uint32_t v) { out.tag[s] = v; });
  }
#pragma unroll
  for (int r = 0; r < R; ++r) index[r] = k0 + r * kWave;
  place(index, [&](int s, int v) {
    out.perm[s] = v;
    if (!rp.has_tags) out.tag[s] = static_cast<uint32_t>(v);
  });
}

template <int D, class T>
static void launch_event_tiles_d(const RunParamsT<T>& rp, const PointArraysT<T>& in,
                                 const BatchBuffersT<T>& bb, hipStream_t s) {
  if (bb.lone.is) {
    hipLaunchKernelGGL((k_lone_tiles<D, T>), dim3(1), dim3(kEvtBlock), 0, s, rp, bb.lone.ev,
                       bb.events, in, bb.sorted, bb.geo, bb.toff, bb.iperm);
    return;
  }
  hipLaunchKernelGGL((k_event_tiles<D, T>), dim3(static_cast<unsigned>(bb.n_events)),
                     dim3(kEvtBlock), 0, s, rp, bb.events, bb.event_order, in, bb.sorted, bb.geo,
                     bb.toff, bb.iperm, bb.n_tiles_total, bb.n_total);
}

template <class T>
static void launch_event_tiles(const RunParamsT<T>& rp, const PointArraysT<T>& in,
                               const BatchBuffersT<T>& bb, hipStream_t s) {
  switch (rp.D) {
    case 1: launch_event_tiles_d<1>(rp, in, bb, s); break;
    case 2: launch_event_tiles_d<2>(rp, in, bb, s); break;
    case 3: launch_event_tiles_d<3>(rp, in, bb, s); break;
    case 4: launch_event_tiles_d<4>(rp, in, bb, s); break;
    case 5: launch_event_tiles_d<5>(rp, in, bb, s); break;
    case 6: launch_event_tiles_d<6>(rp, in, bb, s); break;
    case 7: launch_event_tiles_d<7>(rp, in, bb, s); break;
    case 8: launch_event_tiles_d<8>(rp, in, bb, s); break;
    case 9: launch_event_tiles_d<9>(rp, in, bb, s); break;
    default: launch_event_tiles_d<10>(rp, in, bb, s); break;
  }
}

// Work items: ceil(count / 64) per tile, from slot ioff[t] on (an exclusive scan of
// the counts), or, without that scan (ioff NULL), from slot toff[t] / 64 + t on: a
// tile then has at most one slot more than items, and such slots hold empty items.
// Small launches save four kernels by it; in large ones the empty items, a seventh of
// the slots of the 4096-event batch, cost the neighbour stages 1-3 %.
__device__ __forceinline__ int first_item(const int32_t* __restrict__ ioff, int b, int t) {
  return ioff ? ioff[t] : b / kWave + t;
}
// Exclusive scan of n <= kRankWords counts and their total, by one workgroup: four
// consecutive counts per thread and row (count(w, c) gives those from w on, 0 past the
// end), the rows' loads all in flight together.
constexpr int kRankBlock = 1024;
constexpr int kRankRows = 8;
constexpr int kRankWords = 4 * kRankBlock * kRankRows;
template <class Count>
__device__ __forceinline__ void rank_counts(Count&& count, int n, int32_t* __restrict__ before,
                                            int32_t* __restrict__ total) {
  constexpr int kW = kRankBlock / kWave;
  static_assert(kRankRows * kW == 2 * kWave, "two row totals per lane of the scanning wave");
  __shared__ int32_t part[kRankRows * kW];
  const int wave = threadIdx.x / kWave, lane = lane_id();
  int c[kRankRows][4], incl[kRankRows];
#pragma unroll
  for (int r = 0; r < kRankRows; ++r)
    count((r * kRankBlock + static_cast<int>(threadIdx.x)) * 4, c[r]);
#pragma unroll
  for (int r = 0; r < kRankRows; ++r) {
    incl[r] = wave_incl_scan(c[r][0] + c[r][1] + c[r][2] + c[r][3]);
    if (lane == kWave - 1) part[r * kW + wave] = incl[r];
  }
  __syncthreads();
  if (wave == 0) {
    const int p0 = part[2 * lane], p1 = part[2 * lane + 1];
    const int upto = wave_incl_scan(p0 + p1);
    part[2 * lane] = upto - p0 - p1;
    part[2 * lane + 1] = upto - p1;
    if (lane == kWave - 1) *total = upto;
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kRankRows; ++r) {
    int run = part[r * kW + wave] + incl[r] - (c[r][0] + c[r][1] + c[r][2] + c[r][3]);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int w = (r * kRankBlock + static_cast<int>(threadIdx.x)) * 4 + k;
      if (w < n) before[w] = run;
      run += c[r][k];
    }
  }
}

// The scan of the items per tile (the slots' number is n_items): up to kRankWords tiles
// by one workgroup, more by k_item_count and the general scan (8,281 tiles of 2^20
// points: 8.7 us against four launches of 17; 14,000 tiles in 48 events 12 against 20).
static __global__ __launch_bounds__(kRankBlock) void k_item_ranks(const int32_t* __restrict__ toff,
                                                                  int n_tiles,
                                                                  int32_t* __restrict__ before,
                                                                  int32_t* __restrict__ total) {
  rank_counts(
      [&](int t, int (&c)[4]) {
        int o[5];
#pragma unroll
        for (int k = 0; k < 5; ++k) o[k] = toff[min(t + k, n_tiles)];
#pragma unroll
        for (int k = 0; k < 4; ++k) c[k] = (o[k + 1] - o[k] + kWave - 1) / kWave;
      },
      n_tiles, before, total);
}
static __global__ void k_item_count(const int32_t* __restrict__ toff, int n_tiles,
                                    int32_t* __restrict__ icount) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n_tiles) return;
  icount[k] = (toff[k + 1] - toff[k] + kWave - 1) / kWave;
}

// Event of tile t: the last with t_base <= t (one wave, 64 events per step).
__device__ __forceinline__ int tile_event(const EventDesc* __restrict__ events, int n_events, int t) {
  int lo = 0, n = n_events;  // the answer lies in [lo, lo + n)
  while (n > 1) {
    const int step = (n + kWave - 1) / kWave;
    const int k = lane_id() * step;
    const bool at_or_before = k < n && events[lo + k].t_base <= t;
    const int last = 63 - __builtin_clzll(ballot(at_or_before));  // lane 0 always is
    lo += last * step;
    n = min(step, n - last * step);
  }
  return lo;
}

__device__ __forceinline__ float fmin_t(float a, float b) { return __builtin_fminf(a, b); }
__device__ __forceinline__ double fmin_t(double a, double b) { return __builtin_fmin(a, b); }
__device__ __forceinline__ float fmax_t(float a, float b) { return __builtin_fmaxf(a, b); }
__device__ __forceinline__ double fmax_t(double a, double b) { return __builtin_fmax(a, b); }

// ---------------------------------------------------------------------------
// Distances (DistanceMetrics.hpp), right fold over dimensions
// (internal/meta/accumulate.hpp): t0 + (t1 + (... + (t_{D-1} + 0))).
// For square-root metrics the value returned is the sum under the root.
// ---------------------------------------------------------------------------
template <int D, int M, class T>
__device__ __forceinline__ T metric_pair(const T (&xi)[D], const T (&si)[D], const T (&xj)[D],
                                         const T (&sj)[D], const RunParamsT<T>& rp) {
  if constexpr (M == M_EUCLID) {
    T s;
#pragma unroll
    for (int d = D - 1; d >= 0; --d) {
      const T dx = xi[d] - xj[d];
      s = (d == D - 1) ? dx * dx : dx * dx + s;  // t + 0 == t for t = dx*dx >= +0
    }
    return s;
  } else if constexpr (M == M_WEUCLID) {
    T s = T(0);
#pragma unroll
    for (int d = D - 1; d >= 0; --d) {
      const T dx = xi[d] - xj[d];
      s = rp.mparam[d] * dx * dx + s;
    }
    return s;
  } else if constexpr (M == M_PERIODIC || M == M_PERIODIC_LAST) {
    T s;
#pragma unroll
    for (int d = D - 1; d >= 0; --d) {
      T m = xi[d] - xj[d];
      if (M == M_PERIODIC || d == D - 1) {
        // std::min(a, P - a) by one instruction: NaN in a is NaN in P - a too, a NaN
        // period leaves a on both, and the sign of a zero is lost in the square.
        const T a = __builtin_fabs(m);
        m = fmin_t(a, rp.mparam[d] - a);
      }
      s = (d == D - 1) ? m * m : m * m + s;
    }
    return s;
  } else if constexpr (M == M_MANHATTAN) {
    T s;
#pragma unroll
    for (int d = D - 1; d >= 0; --d) {
      const T a = __builtin_fabs(xi[d] - xj[d]);
      s = (d == D - 1) ? a : a + s;
    }
    return s;
  } else if constexpr (M == M_CHEBYSHEV) {
    T m = T(0);
#pragma unroll
    for (int d = 0; d < D; ++d) {
      const T a = __builtin_fabs(xi[d] - xj[d]);
      m = (m < a) ? a : m;  // std::max(m, a)
    }
    return m;
  } else if constexpr (M == M_WCHEBYSHEV) {
    T m = T(0);
#pragma unroll
    for (int d = 0; d < D; ++d) {
      const T a = rp.mparam[d] * __builtin_fabs(xi[d] - xj[d]);
      m = (m < a) ? a : m;
    }
    return m;
  } else {  // M_MAHALANOBIS: (dx*dx) / (si*si + sj*sj)
    T s = T(0);
#pragma unroll
    for (int d = D - 1; d >= 0; --d) {
      const T dx = xi[d] - xj[d];
      s = dx * dx / (si[d] * si[d] + sj[d] * sj[d]) + s;
    }
    return s;
  }
}

// The same for candidate j read from the sorted columns.
template <int D, int M, class T>
__device__ __forceinline__ T metric_value(const T (&xi)[D], const T (&si)[D],
                                          const T* __restrict__ sx, int64_t cs, int j,
                                          const T* __restrict__ ssig, const RunParamsT<T>& rp) {
  T xj[D], sj[D];
#pragma unroll
  for (int d = 0; d < D; ++d) {
    xj[d] = sx[d * cs + j];
    sj[d] = (M == M_MAHALANOBIS) ? ssig[d * cs + j] : T(0);
  }
  return metric_pair<D, M>(xi, si, xj, sj, rp);
}

// Normal: the caller has shown v >= 2^-96 or v == 0 (float sqrt without its
// tiny-input branch).
template <int M, bool Normal = false, class T>
__device__ __forceinline__ T finish_distance(T v) {
  if constexpr (MetricTraits<M>::kSqrt) {
    if constexpr (Normal && sizeof(T) == 4)
      return sqrt_rn_normal(v);
    else
      return sqrt_rn(v);
  } else {
    return v;
  }
}

// Search box of one point (ClusteringKernels.hpp:111-121, TilesView.hpp:77-87).
// sqrt(2) correctly rounded in each precision (std::sqrt of 2 in the reference).
template <class T>
struct Sqrt2;
template <>
struct Sqrt2<float> {
  static constexpr float v = 0x1.6a09e6p+0f;
};
template <>
struct Sqrt2<double> {
  static constexpr double v = 0x1.6a09e667f3bcdp+0;
};

template <int D, class T>
__device__ __forceinline__ void search_box(const GeoT<T>& g, const T (&xi)[D], const T (&si)[D],
                                           T R, int (&lo)[D], int (&hi)[D]) {
#pragma unroll
  for (int d = 0; d < D; ++d) {
    const T rs = R * si[d] * Sqrt2<T>::v;
    const T r = (R < rs) ? rs : R;  // std::max(R, R * sigma * sqrt(2))
    int a = get_bin(g, xi[d] - r, d);
    int b = get_bin(g, xi[d] + r, d);
    if (g.wrapped[d] && a > b) b += g.nper;
    lo[d] = a;
    hi[d] = b;
  }
}

// Walks the union of the wave's search boxes in lexicographic order (dim 0
// outermost). For every tile that at least one lane's own box contains, calls
// visit(tile_key, in_box) with in_box true on the lanes whose box contains it.
// Each lane thus sees exactly its own boxes' tiles, in the reference's order.
template <int D, class F>
__device__ __forceinline__ void walk_tiles(const int (&lo)[D], const int (&hi)[D], int nper,
                                           const int32_t* wrapped, int t_base, F&& visit) {
  int ulo[D], uhi[D], b[D];
#pragma unroll
  for (int d = 0; d < D; ++d) {
    ulo[d] = wave_min_uniform(lo[d]);
    uhi[d] = wave_max_uniform(hi[d]);
    b[d] = ulo[d];
  }
  if (ulo[0] > uhi[0]) return;  // no active lane
  while (true) {
    bool in = true;
#pragma unroll
    for (int d = 0; d < D; ++d) in = in && (lo[d] <= b[d]) && (b[d] <= hi[d]);
    if (ballot(in) != 0ull) {
      int t = 0;
#pragma unroll
      for (int d = 0; d < D; ++d) t = t * nper + (wrapped[d] ? b[d] % nper : b[d]);
      visit(uniform(t_base + t), in);
    }
    int d = D - 1;
    for (; d >= 0; --d) {
      if (b[d] < uhi[d]) {
        ++b[d];
        break;
      }
      b[d] = ulo[d];
    }
    if (d < 0) break;
  }
}

// ---------------------------------------------------------------------------
// Query order within a tile. A wave pays for the candidates that any of its lanes can
// reach, so the points of every tile with more than one wave's worth are ordered by
// the Hilbert index of their sub-cell of the tile; items then take 64 consecutive
// entries. Results do not depend on the order: a point's traversal is its own,
// whichever lane runs it. (An order by which neighbouring tiles a point's search box
// reaches, kept within the Hilbert order, measured no faster once candidates were
// culled by the wave's box.)
// ---------------------------------------------------------------------------
constexpr int kQueryDims = 3;  // dimensions that enter the keys

// Hilbert index of the point's sub-cell over the first (up to) three dimensions of the
// tile, kCellBits bits per dimension: the curve's steps between neighbouring cells keep
// the 64 consecutive points of an item in a smaller box than a Morton order's jumps
// (4096-event batch, 4 bits: density 23.0 -> 22.4 ms, nearest-higher 7.6 -> 6.8 ms).
// Fine cells order dense tiles further (5 bits: 22.1 and 6.5 ms; 2^20 points in 2-D,
// nearest-higher 404 -> 275 us; 6 bits gain no more and sort slower); small launches
// take the coarse ones, whose sort is shorter (5,003 points: 12 against 15 us). The
// index follows Skilling's transform ("Programming the Hilbert curve", AIP Conf. Proc. 707,
// 2004): rotations undone from the top bit down, a Gray code, the bits interleaved.
template <int D, bool Fine>
struct QueryCells {
  static constexpr int kDims = D < kQueryDims ? D : kQueryDims;
  static constexpr int kCellBits = kDims == 1 ? 8 : kDims == 2 ? (Fine ? 5 : 4) : (Fine ? 3 : 2);
  static constexpr int kBins = 1 << (kDims * kCellBits);
};
template <int D, bool Fine, class T>
__device__ __forceinline__ uint32_t query_cell(const GeoT<T>& g, const T (&xi)[D],
                                               const int (&tb)[D]) {
  constexpr int kD = QueryCells<D, Fine>::kDims;
  constexpr int kB = QueryCells<D, Fine>::kCellBits;
  constexpr int kS = 1 << kB;
  uint32_t q[kD];
#pragma unroll
  for (int d = 0; d < kD; ++d) {
    const T c = g.wrapped[d] ? normalize(g, xi[d], d) : xi[d];
    const T f = ((c - g.mn[d]) / g.side[d] - static_cast<T>(tb[d])) * static_cast<T>(kS);
    q[d] = (f >= T(0)) ? (f < static_cast<T>(kS) ? static_cast<uint32_t>(f) : kS - 1u) : 0u;
  }
  if constexpr (kD > 1) {
#pragma unroll
    for (int b = kB - 1; b > 0; --b) {
      const uint32_t low = (1u << b) - 1u;
#pragma unroll
      for (int d = 0; d < kD; ++d) {
        const bool set = (q[d] >> b) & 1u;
        const uint32_t t = (q[0] ^ q[d]) & low;
        q[d] = set ? q[d] : q[d] ^ t;
        q[0] = set ? q[0] ^ low : (d == 0 ? q[0] : q[0] ^ t);
      }
    }
#pragma unroll
    for (int d = 1; d < kD; ++d) q[d] ^= q[d - 1];
    uint32_t t = 0;
#pragma unroll
    for (int b = kB - 1; b > 0; --b) t ^= ((q[kD - 1] >> b) & 1u) ? (1u << b) - 1u : 0u;
#pragma unroll
    for (int d = 0; d < kD; ++d) q[d] ^= t;
  }
  uint32_t key = 0;
#pragma unroll
  for (int b = kB - 1; b >= 0; --b)
#pragma unroll
    for (int d = 0; d < kD; ++d) key = (key << 1) | ((q[d] >> b) & 1u);
  return key;
}

// What a coordinate adds to a bounding box under the Chebyshev distances. They leave a
// NaN difference out of their maximum, so a point with a NaN may be near any other in
// that dimension, and it adds every value. (Under the other metrics it is near none, and
// their boxes leave it out.)
template <class T>
__device__ __forceinline__ T box_low(T x) {
  return x == x ? x : -std::numeric_limits<T>::infinity();
}
template <class T>
__device__ __forceinline__ T box_high(T x) {
  return x == x ? x : std::numeric_limits<T>::infinity();
}

// Wave-wide minimum and maximum of floating-point values.
template <class T>
__device__ __forceinline__ T wave_min_f(T v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = fmin_t(v, __shfl_xor(v, off, 64));
  return v;
}
template <class T>
__device__ __forceinline__ T wave_max_f(T v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = fmax_t(v, __shfl_xor(v, off, 64));
  return v;
}
// The same, wave-uniform, float through DPP lane moves (no LDS round trips).
__device__ __forceinline__ float wave_min_uniform(float v) {
  return __int_as_float(wave_reduce_dpp(__float_as_int(v), 0x7f800000, [](int a, int b) {
    return __float_as_int(__builtin_fminf(__int_as_float(a), __int_as_float(b)));
  }));
}
__device__ __forceinline__ float wave_max_uniform(float v) {
  return __int_as_float(wave_reduce_dpp(__float_as_int(v), static_cast<int>(0xff800000u), [](int a, int b) {
    return __float_as_int(__builtin_fmaxf(__int_as_float(a), __int_as_float(b)));
  }));
}
__device__ __forceinline__ double wave_min_uniform(double v) {
  v = wave_min_f(v);
  return __longlong_as_double(
      (static_cast<long long>(uniform(static_cast<int>(__double_as_longlong(v) >> 32))) << 32) |
      static_cast<uint32_t>(uniform(static_cast<int>(__double_as_longlong(v)))));
}
__device__ __forceinline__ double wave_max_uniform(double v) { return -wave_min_uniform(-v); }

// Minimum and maximum over each group of N = 8 or 16 lanes (a half row or a row),
// in every lane of the group (float through DPP lane moves: pair swap, quad swap,
// half-row mirror, then for 16 the row mirror; lanes a move does not write take
// the identity, so each move fuses into its operation).
template <int N, class F>
__device__ __forceinline__ float row_reduce_dpp(float v, float id, F op) {
  static_assert(N == 8 || N == 16, "a half row or a row");
  const int i = __float_as_int(id);
  int x = __float_as_int(v);
  x = __float_as_int(op(__int_as_float(x), __int_as_float(__builtin_amdgcn_update_dpp(i, x, 0xB1, 0xF, 0xF, false))));
  x = __float_as_int(op(__int_as_float(x), __int_as_float(__builtin_amdgcn_update_dpp(i, x, 0x4E, 0xF, 0xF, false))));
  x = __float_as_int(op(__int_as_float(x), __int_as_float(__builtin_amdgcn_update_dpp(i, x, 0x141, 0xF, 0xF, false))));
  if constexpr (N == 16)
    x = __float_as_int(op(__int_as_float(x), __int_as_float(__builtin_amdgcn_update_dpp(i, x, 0x140, 0xF, 0xF, false))));
  return __int_as_float(x);
}
template <int N = 16>
__device__ __forceinline__ float row_min(float v) {
  return row_reduce_dpp<N>(v, __builtin_inff(), [](float a, float b) { return __builtin_fminf(a, b); });
}
template <int N = 16>
__device__ __forceinline__ float row_max(float v) {
  return row_reduce_dpp<N>(v, -__builtin_inff(), [](float a, float b) { return __builtin_fmaxf(a, b); });
}
template <int N = 16>
__device__ __forceinline__ double row_min(double v) {
#pragma unroll
  for (int off = 1; off < N; off <<= 1) v = fmin_t(v, __shfl_xor(v, off, 64));
  return v;
}
template <int N = 16>
__device__ __forceinline__ double row_max(double v) {
#pragma unroll
  for (int off = 1; off < N; off <<= 1) v = fmax_t(v, __shfl_xor(v, off, 64));
  return v;
}
// Largest 64-bit key over each group of N = 8 or 16 lanes (both halves moved by DPP).
template <int Ctrl>
__device__ __forceinline__ uint64_t max_dpp_u64(uint64_t v) {
  const int lo = static_cast<int>(static_cast<uint32_t>(v));
  const int hi = static_cast<int>(static_cast<uint32_t>(v >> 32));
  const uint32_t olo = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, lo, Ctrl, 0xF, 0xF, false));
  const uint32_t ohi = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, hi, Ctrl, 0xF, 0xF, false));
  const uint64_t o = (static_cast<uint64_t>(ohi) << 32) | olo;
  return o > v ? o : v;
}
template <int N = 16>
__device__ __forceinline__ uint64_t row_max_u64(uint64_t v) {
  static_assert(N == 8 || N == 16, "a half row or a row");
  v = max_dpp_u64<0xB1>(v);   // quad_perm 1,0,3,2
  v = max_dpp_u64<0x4E>(v);   // quad_perm 2,3,0,1
  v = max_dpp_u64<0x141>(v);  // row_half_mirror
  if constexpr (N == 16) v = max_dpp_u64<0x140>(v);  // row_mirror
  return v;
}

// First layout block of tile t whose candidates begin at sorted position b:
// tile starts rounded up to whole blocks, one spare block per tile, so that the
// tiles' block ranges never overlap.
__device__ __forceinline__ int64_t nh_first_block(int b, int t) {
  return static_cast<int64_t>((b + kNhBlock - 1) / kNhBlock) + t;
}

// The nearest-higher layout of tile t, written by the query-order pass (wave w of
// n_waves takes every n_waves-th 64 slots): the tile's candidates in Hilbert order (order[k], k < cnt) from block
// nh_first_block on, padded to whole blocks (index -1), with each block's
// bounding box. The keys, known after the density stage, are written by the
// density stage itself (k_density, from the same Hilbert order).
template <int D, class T>
__device__ __forceinline__ void write_nh_layout(int t, int b, int cnt, const int32_t* order,
                                                int w, int n_waves, int nan_widens,
                                                const T* __restrict__ sx, int64_t cs,
                                                T* __restrict__ hx, int64_t hs,
                                                int32_t* __restrict__ hidx, T* __restrict__ hbox) {
  static_assert(kWave % kNhBlock == 0, "blocks must not straddle waves");
  static_assert(kNhBlock == 8 || kNhBlock == 16, "block boxes are reduced over DPP half rows or rows");
  const int lane = lane_id();
  const int64_t blk0 = nh_first_block(b, t);
  const int span = (cnt + kNhBlock - 1) / kNhBlock * kNhBlock;
  for (int k0 = w * kWave; k0 < span; k0 += n_waves * kWave) {
    const int k = k0 + lane;
    const bool real = k < cnt;
    T x[D];
    int s = -1;
    if (real) s = order ? order[b + k] : b + k;
#pragma unroll
    for (int d = 0; d < D; ++d) x[d] = real ? sx[d * cs + s] : T(0);
    const int64_t p = blk0 * kNhBlock + k;
    if (k < span) {
#pragma unroll
      for (int d = 0; d < D; ++d) hx[d * hs + p] = x[d];
      hidx[p] = s;
    }
    T lo[D], hi[D];
#pragma unroll
    for (int d = 0; d < D; ++d) {
      lo[d] = real ? x[d] : std::numeric_limits<T>::infinity();
      hi[d] = real ? x[d] : -std::numeric_limits<T>::infinity();
    }
    if (nan_widens) {
#pragma unroll
      for (int d = 0; d < D; ++d) {
        lo[d] = box_low(lo[d]);
        hi[d] = box_high(hi[d]);
      }
    }
#pragma unroll
    for (int d = 0; d < D; ++d) {
      lo[d] = row_min<kNhBlock>(lo[d]);
      hi[d] = row_max<kNhBlock>(hi[d]);
    }
    if (k < span && (k % kNhBlock) == 0) {
      const int64_t q = blk0 + k / kNhBlock;
#pragma unroll
      for (int d = 0; d < D; ++d) {
        hbox[q * 2 * D + d] = lo[d];
        hbox[q * 2 * D + D + d] = hi[d];
      }
    }
  }
}

// Tile t (one wave): its work items and (tbox) its points' bounding box, by which the
// density stage leaves out the tiles none of a wave's queries can reach.
struct TileSetup {
  const EventDesc* events;
  int n_events;
  Item* items;
  const int32_t* ioff;
  int32_t max_items;
  int32_t nan_widens;  // the metric is one of the Chebyshev distances (box_low)
};
template <int D, class T>
__device__ __forceinline__ void tile_setup(const TileSetup& a, int t, int n_tiles, int b, int e,
                                           const T* __restrict__ sx, int64_t cs,
                                           T* __restrict__ tbox) {
  // The first points' loads go out before the search for the event.
  T x0[D];
#pragma unroll
  for (int d = 0; d < D; ++d)
    x0[d] = (tbox && b + lane_id() < e) ? sx[d * cs + b + lane_id()] : std::numeric_limits<T>::quiet_NaN();
  const int e_t = tile_event(a.events, a.n_events, t);
  const int first = first_item(a.ioff, b, t);
  const int slots = a.ioff ? (e - b + kWave - 1) / kWave
                         : (t + 1 < n_tiles ? first_item(a.ioff, e, t + 1) : a.max_items) - first;
  for (int k = lane_id(); k < slots; k += kWave) {
    Item it;
    it.tile = t;
    it.begin = min(e, b + k * kWave);
    it.end = min(e, it.begin + kWave);
    it.event = e_t;
    a.items[first + k] = it;
  }
  if (!tbox) return;
  T mn[D], mx[D];
#pragma unroll
  for (int d = 0; d < D; ++d) {
    mn[d] = fmin_t(std::numeric_limits<T>::infinity(), x0[d]);
    mx[d] = fmax_t(-std::numeric_limits<T>::infinity(), x0[d]);
  }
#pragma unroll 4
  for (int s = b + kWave + lane_id(); s < e; s += kWave)
#pragma unroll
    for (int d = 0; d < D; ++d) {
      const T x = sx[d * cs + s];
      mn[d] = fmin_t(mn[d], x);
      mx[d] = fmax_t(mx[d], x);
    }
  if (a.nan_widens) {
    for (int s = b + lane_id(); s < e; s += kWave)
#pragma unroll
      for (int d = 0; d < D; ++d) {
        const T x = sx[d * cs + s];
        mn[d] = fmin_t(mn[d], box_low(x));
        mx[d] = fmax_t(mx[d], box_high(x));
      }
  }
#pragma unroll
  for (int d = 0; d < D; ++d) {
    mn[d] = wave_min_uniform(mn[d]);
    mx[d] = wave_max_uniform(mx[d]);
  }
  if (lane_id() == 0) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      tbox[static_cast<int64_t>(t) * 2 * D + d] = mn[d];
      tbox[static_cast<int64_t>(t) * 2 * D + D + d] = mx[d];
    }
  }
}

__device__ __forceinline__ void zero_queues(int32_t* __restrict__ ctl) {
  if (threadIdx.x >= kQueueDensity && threadIdx.x < kQueueWords) ctl[threadIdx.x] = 0;
}

// The setup alone, where the queries keep their order.
template <int D, class T>
__global__ __launch_bounds__(kBlock) void k_tile_setup(const TileSetup setup,
                                                       const int32_t* __restrict__ toff, int n_tiles,
                                                       const T* __restrict__ sx, int64_t cs,
                                                       T* __restrict__ tbox,
                                                       int32_t* __restrict__ ctl) {
  if (blockIdx.x == 0) zero_queues(ctl);
  const int t = blockIdx.x * kWaves + threadIdx.x / kWave;
  if (t < n_tiles) tile_setup<D>(setup, t, n_tiles, toff[t], toff[t + 1], sx, cs, tbox);
}

// The query order of per <= W tiles per workgroup of W waves (8 for a lone event, whose
// dense tiles are the largest, else 4: one event of 2^20 points 81 us at 4 and 54 us at 8, the
// 4096-event batch 744 us and 990 us). A tile of at most one wave's
// points keeps its order (one wave each). The others are taken one after the other
// by the whole workgroup, a counting sort in LDS by the Hilbert index: the dense
// tiles, thousands of points where most tiles hold a few dozen, are what one wave
// per tile waited for (4096-event batch: 1043 -> 789 us; one event of 2^20 points
// in 2-D: 248 -> 89 us; of 100,000: 87 -> 28 us). Points of equal index are placed by LDS atomics, in no
// order among themselves: no result depends on the query order or on the order
// within the nearest-higher layout.
template <int D, int W, bool Fine, class T>
__global__ __launch_bounds__(W * kWave) void k_query_order(
    const RunParamsT<T> rp, const TileSetup setup, T* __restrict__ tbox, int32_t* __restrict__ ctl,
    const T* __restrict__ geo, const int32_t* __restrict__ toff, int n_tiles, int per,
    const T* __restrict__ sx, int64_t cs, int32_t* __restrict__ qfine, T* __restrict__ hx, int64_t hs, int32_t* __restrict__ hidx, T* __restrict__ hbox) {
  constexpr int kBins = QueryCells<D, Fine>::kBins;
  constexpr int kOrderBlock = W * kWave;
  constexpr int kHeld = 4;  // rounds whose indices stay in registers
  constexpr int kPer = (kBins + kOrderBlock - 1) / kOrderBlock;  // bins per thread in the scan
  __shared__ int32_t cnt[kBins];
  const int w = threadIdx.x / kWave;
  const int lane = lane_id();
  {
    const int t = blockIdx.x * per + w;
    const bool mine = w < per && t < n_tiles;
    const int b = mine ? toff[t] : 0, e = mine ? toff[t + 1] : 0;
    if (blockIdx.x == 0) zero_queues(ctl);
    if (mine) tile_setup<D>(setup, t, n_tiles, b, e, sx, cs, tbox);
    if (mine && e - b <= kWave) {  // one item: the query order is irrelevant
      if (b + lane < e) qfine[b + lane] = b + lane;
      if (hx) write_nh_layout<D>(t, b, e - b, nullptr, 0, 1, setup.nan_widens, sx, cs, hx, hs, hidx, hbox);
    }
  }
  for (int k = 0; k < per; ++k) {
    const int t = blockIdx.x * per + k;
    if (t >= n_tiles) break;
    const int b = toff[t], e = toff[t + 1];
    if (e - b <= kWave) continue;
    const int ev_i = tile_event(setup.events, setup.n_events, t);
    const EventDesc ev = setup.events[ev_i];
    const GeoT<T> g = event_geo(geo, rp, ev_i, ev.nper);
    int tb[D];
    {
      int r = t - ev.t_base;
#pragma unroll
      for (int d = D - 1; d >= 0; --d) {
        tb[d] = r % ev.nper;
        r /= ev.nper;
      }
    }
    for (int k2 = threadIdx.x; k2 < kBins; k2 += kOrderBlock) cnt[k2] = 0;
    __syncthreads();
    auto key_of = [&](int s) {
      T xi[D];
#pragma unroll
      for (int d = 0; d < D; ++d) xi[d] = sx[d * cs + s];
      return query_cell<D, Fine>(g, xi, tb);
    };
    uint32_t held[kHeld];
#pragma unroll
    for (int r = 0; r < kHeld; ++r) {
      const int s = b + r * kOrderBlock + static_cast<int>(threadIdx.x);
      held[r] = s < e ? key_of(s) : 0u;
      if (s < e) atomicAdd(&cnt[held[r]], 1);
    }
#pragma unroll 4
    for (int s = b + kHeld * kOrderBlock + static_cast<int>(threadIdx.x); s < e; s += kOrderBlock)
      atomicAdd(&cnt[key_of(s)], 1);
    __syncthreads();
    int total;
    const int bin0 = static_cast<int>(threadIdx.x) * kPer;
    int c[kPer], sum = 0;
#pragma unroll
    for (int k2 = 0; k2 < kPer; ++k2) {
      c[k2] = bin0 + k2 < kBins ? cnt[bin0 + k2] : 0;
      sum += c[k2];
    }
    int run = b + block_excl_scan<kOrderBlock>(sum, &total);
#pragma unroll
    for (int k2 = 0; k2 < kPer; ++k2) {
      if (bin0 + k2 < kBins) cnt[bin0 + k2] = run;
      run += c[k2];
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kHeld; ++r) {
      const int s = b + r * kOrderBlock + static_cast<int>(threadIdx.x);
      if (s < e) qfine[atomicAdd(&cnt[held[r]], 1)] = s;
    }
#pragma unroll 4
    for (int s = b + kHeld * kOrderBlock + static_cast<int>(threadIdx.x); s < e; s += kOrderBlock)
      qfine[atomicAdd(&cnt[key_of(s)], 1)] = s;
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");  // qfine of the tile
    __syncthreads();
    if (hx) write_nh_layout<D>(t, b, e - b, qfine, w, W, setup.nan_widens, sx, cs, hx, hs, hidx, hbox);
  }
}

// ---------------------------------------------------------------------------
// Kernel values (ConvolutionalKernel.hpp:21-57) for a candidate within the radius.
// K_GAUSS2 is the gaussian whose 2*sigma*sigma is a power of two: there division
// by it and multiplication by its reciprocal are the same correctly rounded
// operation on the same exact value, so the cheaper one is used (in float, the
// power of two is folded into the exp's constants instead, ExpScaled). The _UNIT
// forms are those of amplitude 1, whose product A * e is e itself (denormals are
// kept, so even a subnormal e is unchanged).
// ---------------------------------------------------------------------------
enum { K_GAUSS2 = 3, K_EXP_UNIT = 4, K_GAUSS2_UNIT = 5 };

// exp of an argument the host has shown to lie in [LO, HI] for every candidate
// within the radius (rp.exp_in_range, passed as InRange) skips the range
// handling; both forms give the same value there.
template <bool InRange>
__device__ __forceinline__ float kernel_exp(float x, const RunParamsT<float>&) {
  return InRange ? expf_cw_core<true>(x) : expf_cw(x);
}
template <bool InRange>
__device__ __forceinline__ double kernel_exp(double x, const RunParamsT<double>&) {
  return InRange ? expd_cw_core(x) : expd_cw(x);
}

// c0: rp.es.c[0] (float gaussian with a folded scale), possibly in a vector register.
template <int M, int K, bool InRange, bool Normal, class T>
__device__ __forceinline__ T kernel_value(T v, const RunParamsT<T>& rp, T c0) {
  if constexpr (K == K_FLAT) {
    return rp.kp0;
  } else if constexpr (K == K_EXP || K == K_EXP_UNIT) {
    const T e = kernel_exp<InRange>(-rp.kp0 * finish_distance<M, Normal>(v), rp);
    return K == K_EXP_UNIT ? e : rp.kp1 * e;
  } else if constexpr (K == K_GAUSS) {
    const T dd = finish_distance<M, Normal>(v);
    return rp.kp1 * kernel_exp<InRange>(-dd * dd / rp.gauss_den, rp);
  } else if constexpr (sizeof(T) == 4) {
    // exp((-dd*dd) * 2^-s) with 2^-s = 1 / gauss_den folded into rp.es.
    const T dd = finish_distance<M, Normal>(v);
    const T y = -dd * dd;
    const T e = InRange ? expf_cw_core_scaled<true>(y, rp.es, c0) : expf_cw_scaled(y, rp.es, c0);
    return K == K_GAUSS2_UNIT ? e : rp.kp1 * e;
  } else {
    const T dd = finish_distance<M, Normal>(v);
    const T e = kernel_exp<InRange>((-dd * dd) * rp.gauss_inv_den, rp);
    return K == K_GAUSS2_UNIT ? e : rp.kp1 * e;
  }
}

// Ordering key stored with each density: float packs (rho, tag) into 64 bits;
// double keeps rho's order alone and compares tags separately.
__device__ __forceinline__ uint64_t density_key(float rho, uint32_t tag) {
  return rho_tag_key(rho, tag, false);
}
__device__ __forceinline__ uint64_t density_key(double rho, uint32_t) {
  return rho_key_f64(rho, false);
}

// Loads U consecutive wave-uniform column values (a block of candidates) with
// one wide scalar load and holds them in scalar registers at this point: left to
// itself the compiler may sink each value's load into the candidate's branch,
// where every use then waits on its own load.
template <int U, class T>
__device__ __forceinline__ void load_block(const T* __restrict__ p, T (&out)[U]) {
  typedef T Vec __attribute__((ext_vector_type(U), aligned(sizeof(T))));
  Vec v = *reinterpret_cast<const Vec*>(p);
  asm volatile("" : "+s"(v));
#pragma unroll
  for (int k = 0; k < U; ++k) out[k] = v[k];
}

// A lower bound, over every query point in [qlo, qhi] and every candidate inside
// the box [bl, bh], of the value metric_value computes (the same operations on
// the per-dimension gaps, which never exceed the pairs' own differences after
// rounding). With qlo = qhi = x it bounds one query point. Weighted metrics
// need weights >= 0 (checked on the host).
template <int D, int M, class T>
__device__ __forceinline__ T metric_lb(const T (&qlo)[D], const T (&qhi)[D], const T (&bl)[D],
                                       const T (&bh)[D], const RunParamsT<T>& rp) {
  T g[D];
#pragma unroll
  for (int d = 0; d < D; ++d) g[d] = fmax_t(fmax_t(bl[d] - qhi[d], qlo[d] - bh[d]), T(0));
  if constexpr (M == M_EUCLID) {
    T s;
#pragma unroll
    for (int d = D - 1; d >= 0; --d) s = (d == D - 1) ? g[d] * g[d] : g[d] * g[d] + s;
    return s;
  } else if constexpr (M == M_WEUCLID) {
    T s = T(0);
#pragma unroll
    for (int d = D - 1; d >= 0; --d) s = rp.mparam[d] * g[d] * g[d] + s;
    return s;
  } else if constexpr (M == M_PERIODIC || M == M_PERIODIC_LAST) {
    // a = |dx| lies in [g, G]. With period P > 0, min(a, P - a) >= min(g, P - G)
    // when P - G >= 0 (else 0 bounds its square). With P <= 0 (an unwrapped
    // dimension), min(a, P - a) = P - a and |P - a| >= a >= g.
    T s;
#pragma unroll
    for (int d = D - 1; d >= 0; --d) {
      if (M == M_PERIODIC_LAST && d < D - 1) {
        s = g[d] * g[d] + s;
        continue;
      }
      const T P = rp.mparam[d];
      const T G = fmax_t(qhi[d] - bl[d], bh[d] - qlo[d]);
      const T pg = P - G;
      const T m = (P <= T(0)) ? g[d] : ((pg >= T(0)) ? fmin_t(g[d], pg) : T(0));
      s = (d == D - 1) ? m * m : m * m + s;
    }
    return s;
  } else if constexpr (M == M_MANHATTAN) {
    T s;
#pragma unroll
    for (int d = D - 1; d >= 0; --d) s = (d == D - 1) ? g[d] : g[d] + s;
    return s;
  } else if constexpr (M == M_CHEBYSHEV) {
    T m = T(0);
#pragma unroll
    for (int d = 0; d < D; ++d) m = (m < g[d]) ? g[d] : m;
    return m;
  } else {  // M_WCHEBYSHEV
    T m = T(0);
#pragma unroll
    for (int d = 0; d < D; ++d) {
      const T a = rp.mparam[d] * g[d];
      m = (m < a) ? a : m;
    }
    return m;
  }
}

// 1 where v * scale <= limit by at least one, 0 where it is not less (and for a NaN
// v): the fma's output clamped to [0, 1]. With limit = scale * t, t the next value
// above a threshold and scale a power of two that makes t's unit in the last place
// at least one, it is 1 exactly where v is within the threshold.
__device__ __forceinline__ float within(float v, float limit, float scale) {
  float in;
  asm("v_fma_f32 %0, -%1, %2, %3 clamp" : "=v"(in) : "v"(v), "s"(scale), "v"(limit));
  return in;
}
__device__ __forceinline__ double within(double v, double limit, double scale) {
  double in;
  asm("v_fma_f64 %0, -%1, %2, %3 clamp" : "=v"(in) : "v"(v), "s"(scale), "v"(limit));
  return in;
}
__device__ __forceinline__ float fma_t(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double fma_t(double a, double b, double c) { return __builtin_fma(a, b, c); }

// Lane i's value in every lane (i wave-uniform).
__device__ __forceinline__ float read_lane(float v, int i) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), i));
}
__device__ __forceinline__ double read_lane(double v, int i) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane(static_cast<int>(b), i);
  const int hi = __builtin_amdgcn_readlane(static_cast<int>(b >> 32), i);
  return __longlong_as_double((static_cast<long long>(hi) << 32) |
                              static_cast<long long>(static_cast<uint32_t>(lo)));
}
__device__ __forceinline__ uint64_t read_lane(uint64_t v, int i) {
  const uint32_t lo = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v), i));
  const uint32_t hi =
      static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v >> 32), i));
  return (static_cast<uint64_t>(hi) << 32) | lo;
}

// ---------------------------------------------------------------------------
// The candidates a wave of queries has to look at: the tiles of the union of the
// lanes' search boxes in the reference's order (dimension 0 outermost), listed 64
// at a time, one per lane, so that their offsets and boxes arrive together.
// ---------------------------------------------------------------------------
template <int D>
__device__ __forceinline__ BoxUnion<D> box_union(const int (&lo)[D], const int (&hi)[D]) {
  BoxUnion<D> u;
#pragma unroll
  for (int d = 0; d < D; ++d) {
    u.lo[d] = wave_min_uniform(lo[d]);
    const int h = wave_max_uniform(hi[d]);
    u.ext[d] = u.lo[d] > h ? 0 : h - u.lo[d] + 1;
  }
  first_tile_run(u);
  return u;
}

template <int D>
struct TileGroup {
  bool listed;    // this lane has a tile
  int t, j0, j1;  // the tile and its candidates
  int b[D];       // its bins (past nper on a wrapped dimension)
};
template <int D>
__device__ __forceinline__ void list_tiles(const BoxUnion<D>& u, int base, int nper,
                                           const int32_t* wrapped, int t_base,
                                           const int32_t* __restrict__ toff, TileGroup<D>* g) {
  const int idx = base + lane_id();
  int q = idx, t = 0, scale = 1;
#pragma unroll
  for (int d = D - 1; d >= 0; --d) {
    const int r = d == 0 ? q : q % u.ext[d];
    q = d == 0 ? 0 : q / u.ext[d];
    g->b[d] = u.lo[d] + r;
    t += scale * (wrapped[d] ? g->b[d] % nper : g->b[d]);
    scale *= nper;
  }
  g->t = t_base + t;
  g->j0 = g->j1 = 0;
  g->listed = idx < u.tiles;
  if (g->listed) {
    g->j0 = toff[g->t];
    g->j1 = toff[g->t + 1];
  }
}
// Does each lane's own box hold the tile of lane i?
template <int D>
__device__ __forceinline__ bool box_holds(const TileGroup<D>& g, int i, const int (&lo)[D],
                                          const int (&hi)[D]) {
  bool in = true;
#pragma unroll
  for (int d = 0; d < D; ++d) {
    const int b = __builtin_amdgcn_readlane(g.b[d], i);
    in = in && lo[d] <= b && b <= hi[d];
  }
  return in;
}

// Box of a wave's query points, and their largest sigmas (wave-uniform, in scalar
// registers). A query with a NaN coordinate widens it where it can be near any
// candidate (box_low); under the other metrics it is near none and left out.
template <int D, class T>
struct QueryBox {
  T lo[D], hi[D], s[D];
};
template <int D, int M, class T>
__device__ __forceinline__ QueryBox<D, T> query_box(const T (&x)[D], const T (&s)[D], bool active) {
  QueryBox<D, T> q;
#pragma unroll
  for (int d = 0; d < D; ++d) {
    T lo = x[d], hi = x[d];
    if constexpr (M == M_CHEBYSHEV || M == M_WCHEBYSHEV) {
      lo = box_low(lo);
      hi = box_high(hi);
    }
    q.lo[d] = wave_min_uniform(active ? lo : std::numeric_limits<T>::infinity());
    q.hi[d] = wave_max_uniform(active ? hi : -std::numeric_limits<T>::infinity());
    q.s[d] = M == M_MAHALANOBIS ? wave_max_uniform(active ? __builtin_fabs(s[d]) : T(0)) : T(0);
  }
  return q;
}
// A lower bound of the metric between any query of the box and a candidate at x (with
// sigma sx, Mahalanobis): the metric's own operations on the gaps and, Mahalanobis, on
// the largest sigma, each monotone after rounding. A candidate's NaN excludes nothing.
template <int D, int M, class T>
__device__ __forceinline__ bool out_of_reach(const QueryBox<D, T>& q, const T (&x)[D],
                                             const T (&sx)[D], const RunParamsT<T>& rp, T thr) {
  if constexpr (M == M_MAHALANOBIS) {
    T s = T(0);
#pragma unroll
    for (int d = D - 1; d >= 0; --d) {
      const T g = fmax_t(fmax_t(x[d] - q.hi[d], q.lo[d] - x[d]), T(0));
      s = g * g / (q.s[d] * q.s[d] + sx[d] * sx[d]) + s;
    }
    return s > thr;
  } else {
    return metric_lb<D, M>(q.lo, q.hi, x, x, rp) > thr;
  }
}

// Does the lane's tile hold candidates, and can a query of the box reach its box?
template <int D, int M, class T>
__device__ __forceinline__ bool tile_in_reach(const TileGroup<D>& g, const QueryBox<D, T>& q,
                                              const T* __restrict__ tbox, const RunParamsT<T>& rp,
                                              T thr) {
  bool reach = g.j0 < g.j1;
  if constexpr (M != M_MAHALANOBIS) {
    if (tbox && g.listed) {  // beside the offsets, not after them
      T bl[D], bh[D];
#pragma unroll
      for (int d = 0; d < D; ++d) {
        bl[d] = tbox[static_cast<int64_t>(g.t) * 2 * D + d];
        bh[d] = tbox[static_cast<int64_t>(g.t) * 2 * D + D + d];
      }
      reach = reach && !(metric_lb<D, M>(q.lo, q.hi, bl, bh, rp) > thr);
    }
  }
  return reach;
}

// Compile-time loop modes of the density stage: kernel exp arguments known to be
// in range, and square roots known to need no tiny-input branch (flat kernel: the
// sums by within()).
template <bool InRange, bool Normal>
struct ModeC {
  static constexpr bool kInRange = InRange;
  static constexpr bool kNormal = Normal;
};

// Candidates are walked in blocks of U so that their wave-uniform data arrives
// in a few wide scalar loads (measured on MI355X).
template <int D>
struct Unroll {
  static constexpr int U = D <= 3 ? 8 : 4;
};

// ---------------------------------------------------------------------------
// (b) Local density: rho_i = sum over visited j of ((float)(d <= dc) * K) * w_j
// (ClusteringKernels.hpp:53-69). Candidates beyond dc add +0 and are skipped;
// the additions keep the candidate order.
// ---------------------------------------------------------------------------
template <int D, int M, int K, bool Persistent, class T>
__global__ __launch_bounds__(kMaxNeighbourBlock) void k_density(
    const RunParamsT<T> rp, const EventDesc* __restrict__ events, const T* __restrict__ geo,
    const int32_t* __restrict__ toff, const Item* __restrict__ items,
    int32_t* __restrict__ n_items, const T* __restrict__ sx, int64_t cs,
    const T* __restrict__ sw, const T* __restrict__ sfw, const T* __restrict__ ssig,
    const uint32_t* __restrict__ stag, const int32_t* __restrict__ qperm,
    T* __restrict__ srho, uint64_t* __restrict__ skey, const T* __restrict__ tbox,
    uint64_t* __restrict__ hkey, uint64_t* __restrict__ hbkey) {
  constexpr int U = Unroll<D>::U;
  auto process = [&](const int item) {
    const Item it = items[item];
    const EventDesc ev = events[it.event];
    const GeoT<T> g = event_geo(geo, rp, it.event, ev.nper);
    const int q = it.begin + lane_id();
    const bool active = q < it.end;
    const int s = active ? (qperm ? qperm[q] : q) : -1;  // sorted position of this lane's point

    T xi[D], si[D];
  #pragma unroll
    for (int d = 0; d < D; ++d) {
      xi[d] = active ? sx[d * cs + s] : T(0);
      si[d] = (active && rp.has_sigma) ? ssig[d * cs + s] : T(0);
    }
    int lo[D], hi[D];
    search_box<D>(g, xi, si, rp.dc, lo, hi);
    if (!active) {
  #pragma unroll
      for (int d = 0; d < D; ++d) {
        lo[d] = INT32_MAX;
        hi[d] = INT32_MIN;
      }
    }
    const T thr_in = MetricTraits<M>::kSqrt ? rp.dc_sq_max : rp.dc;
    T rho = T(0);
    // The diagonal term K(i,i) * w_i = w_i; the flat kernel's off-diagonal weights
    // come pre-multiplied (fw = f * w).
    const T wself = active ? sw[s] : T(0);
    const T* __restrict__ wcol = (K == K_FLAT) ? sfw : sw;
    // The folded gaussian's leading coefficient, held in a vector register for the
    // whole walk (an fma takes one scalar operand; the next coefficient is one).
    T c0 = T(0);
    if constexpr (sizeof(T) == 4) {
      c0 = rp.es.c[0];
      asm volatile("" : "+v"(c0));
    }

    // term(j) = K(d_ij) * w_j, with K = 1 on the diagonal (self only in its own tile).
    // wj is the candidate's column value, loaded with its block of candidates.
    // own_c: std::true_type for the point's own tile, where the diagonal term lies;
    // mode_c: ModeC<in range, normal> (see below).
    auto add = [&](T v, int j, T wj, T thr, auto own_c, auto mode_c) {
      constexpr bool own = decltype(own_c)::value;
      constexpr bool inr = decltype(mode_c)::kInRange;
      constexpr bool nrm = decltype(mode_c)::kNormal;
      if constexpr (K == K_FLAT) {
        const T wt = (own && j == s) ? wself : wj;
        if constexpr (nrm) {
          // rho + 1 * w rounds as rho + w does, and rho + 0 * w is rho for a finite
          // w: two instructions where a compare, a select (both at half rate) and an
          // addition take three.
          rho = fma_t(within(v, thr, rp.in_scale), wt, rho);
        } else {
          // rho + 0 == rho here (rho is never -0), so selecting the unchanged sum is
          // the reference's addition of a zero term.
          const T next = rho + wt;
          rho = (v <= thr) ? next : rho;
        }
      } else if constexpr (K == K_EXP_UNIT || K == K_GAUSS2_UNIT) {
        // Amplitude 1: the diagonal's distance is 0 and exp(-0) is exactly 1, the
        // reference's K(i, i), so the diagonal needs no case of its own.
        if (v <= thr) rho += kernel_value<M, K, inr, nrm>(v, rp, c0) * wj;
      } else {
        if (v <= thr) {
          const T kv = (own && j == s) ? T(1) : kernel_value<M, K, inr, nrm>(v, rp, c0);
          rho += kv * wj;
        }
      }
    };
    // The diagonal needs a case of its own (not with amplitude 1, see add).
    constexpr bool kDiagonal = K != K_EXP_UNIT && K != K_GAUSS2_UNIT;
    auto walk = [&](int j0, int j1, T thr, auto own_c, auto mode_c) {
      int j = j0;
      for (; j + U <= j1; j += U) {
        T v[U], w[U];
  #pragma unroll
        for (int k = 0; k < U; ++k) v[k] = metric_value<D, M>(xi, si, sx, cs, j + k, ssig, rp);
        load_block<U>(wcol + j, w);
        if (decltype(own_c)::value &&
            ballot(static_cast<unsigned>(s - j) < static_cast<unsigned>(U)) != 0ull) {
  #pragma unroll
          for (int k = 0; k < U; ++k) add(v[k], j + k, w[k], thr, std::true_type{}, mode_c);
        } else {
  #pragma unroll
          for (int k = 0; k < U; ++k) add(v[k], j + k, w[k], thr, std::false_type{}, mode_c);
        }
      }
      for (; j < j1; ++j)
        add(metric_value<D, M>(xi, si, sx, cs, j, ssig, rp), j, wcol[j], thr, own_c, mode_c);
    };
    // A tile's candidates, 64 at a time, one per lane: those that no query of the wave
    // can reach (a lower bound of the metric above the radius: the reference adds
    // their terms as +0) are left out by one ballot. Where few are left, their
    // coordinates come from the lanes; where many are, the block is walked whole,
    // through the scalar cache, which costs a candidate four instructions less. The
    // line between them, measured at 1/8 to 13/16: the 4096-event batch is flat from
    // 1/4 to 1/2 (22.5-22.7 ms; 23.5 at 2/3), 2^20 points in 2-D and 3-D best from 3/8
    // to 1/2 (742, 733 us; 482, 473 us).
    const bool cull = rp.cull != 0;
    const QueryBox<D, T> qb = query_box<D, M>(xi, si, active);
    auto walk_tile = [&](int j0, int j1, T thr, auto mode_c) {
      T nx[D], ns[D];
      auto fetch = [&](int j) {
        const int c = j + lane_id();
  #pragma unroll
        for (int d = 0; d < D; ++d) {
          nx[d] = c < j1 ? sx[d * cs + c] : T(0);
          ns[d] = (M == M_MAHALANOBIS && c < j1) ? ssig[d * cs + c] : T(0);
        }
      };
      fetch(j0);
      for (int j = j0; j < j1; j += kWave) {
        T cx[D], cg[D];
  #pragma unroll
        for (int d = 0; d < D; ++d) {
          cx[d] = nx[d];
          cg[d] = ns[d];
        }
        if (j + kWave < j1) fetch(j + kWave);
        const int cnt = min(kWave, j1 - j);
        uint64_t left = ballot(lane_id() < cnt &&
                               !(cull && out_of_reach<D, M>(qb, cx, cg, rp, thr_in)));
        const int n = __popcll(left);
        if (n == 0) continue;
        const T cw = lane_id() < cnt ? wcol[j + lane_id()] : T(0);
        auto each = [&](auto self_c) {
          if (8 * n >= 3 * cnt) {
            walk(j, j + cnt, thr, self_c, mode_c);
            return;
          }
          while (left) {
            const int i = __builtin_ctzll(left);
            left &= left - 1ull;
            T xj[D], sj[D];
  #pragma unroll
            for (int d = 0; d < D; ++d) {
              xj[d] = read_lane(cx[d], i);
              sj[d] = M == M_MAHALANOBIS ? read_lane(cg[d], i) : T(0);
            }
            add(metric_pair<D, M>(xi, si, xj, sj, rp), j + i, read_lane(cw, i), thr, self_c,
                mode_c);
          }
        };
        // Only the blocks that hold a lane's own point test for it.
        if (kDiagonal && ballot(static_cast<unsigned>(s - j) < static_cast<unsigned>(cnt)) != 0ull)
          each(std::true_type{});
        else
          each(std::false_type{});
      }
    };
    const BoxUnion<D> boxes = box_union(lo, hi);
    auto run = [&](auto mode_c) {
      BoxUnion<D> u = boxes;
      do for (int base = 0; base < u.tiles; base += kWave) {
        TileGroup<D> g;
        list_tiles(u, base, ev.nper, rp.wrapped, ev.t_base, toff, &g);
        uint64_t held = ballot(tile_in_reach<D, M>(g, qb, tbox, rp, thr_in));
        while (held) {
          const int i = __builtin_ctzll(held);
          held &= held - 1ull;
          const bool in = box_holds(g, i, lo, hi);
          if (ballot(in) == 0ull) continue;
          const int j0 = __builtin_amdgcn_readlane(g.j0, i), j1 = __builtin_amdgcn_readlane(g.j1, i);
          const T thr = (K == K_FLAT && decltype(mode_c)::kNormal)
                            ? (in ? rp.in_limit : -rp.in_limit)
                            : (in ? thr_in : T(-1));
          walk_tile(j0, j1, thr, mode_c);
        }
      } while (next_tile_run(u));
    };
    // Both decisions are made once, outside the candidate loop:
    //  - in range: launch-wide, every exp argument within the radius is in range;
    //  - normal: Euclidean in float, and no lane of the wave has a coordinate of
    //    magnitude below 2^-24. Then every pair with v > 0 has some |dx| >= 2^-48
    //    (floats of magnitude >= 2^-24 are multiples of 2^-47, and the largest float
    //    below 2^-24 is 2^-24 - 2^-48), so v >= 2^-96 and the square root needs no
    //    tiny-input branch.
    // The flat kernel has one decision of another kind: sums through within(), taken
    // again with selects where a weight was not finite (0 * inf is NaN; finite
    // weights get here only when their sum overflows). 2^20 points in 2-D: 986 us
    // with selects, 801 us.
    if constexpr (K == K_FLAT) {
      bool again = true;
      if (rp.in_scale != T(0)) {
        run(ModeC<true, true>{});
        again = ballot(!(__builtin_fabs(rho) <= std::numeric_limits<T>::max())) != 0ull;
      }
      if (again) {
        rho = T(0);
        run(ModeC<true, false>{});
      }
    } else {
      bool tiny = false;
  #pragma unroll
      for (int d = 0; d < D; ++d) tiny = tiny || (__builtin_fabs(xi[d]) < T(0x1p-24));
      const bool normal = (M == M_EUCLID) && sizeof(T) == 4 && ballot(active && tiny) == 0ull;
      if (rp.exp_in_range && normal)
        run(ModeC<true, true>{});
      else if (rp.exp_in_range)
        run(ModeC<true, false>{});
      else
        run(ModeC<false, false>{});
    }
    if (hkey) {
      // The nearest-higher block layout takes the keys here: the lanes are the
      // tile's points in Hilbert order (qfine) from a multiple of 64, so
      // lane k's point fills layout slot k of the tile and each row of 16 lanes
      // is one block, whose largest key a row reduction gives. Lanes past the
      // tile's points write the padding's key 0 up to the last block.
      static_assert(kWave % kNhBlock == 0, "a block is a group of lanes of one wave");
      const int tb = toff[it.tile];
      const int k = q - tb;
      const int span = (toff[it.tile + 1] - tb + kNhBlock - 1) / kNhBlock * kNhBlock;
      const uint64_t key = active ? density_key(rho, stag[s]) : 0ull;
      const uint64_t m = row_max_u64<kNhBlock>(key);
      if (k < span) {
        const int64_t p = nh_first_block(tb, it.tile) * kNhBlock + k;
        hkey[p] = key;
        if ((k % kNhBlock) == 0) hbkey[p / kNhBlock] = m;
      }
      if (active) srho[s] = rho;
    } else if (active) {
      srho[s] = rho;
      skey[s] = density_key(rho, stag[s]);
    }
  };
  if constexpr (Persistent) {
    ItemCursor cursor(n_items, kQueueDensity, rp);
    for (int item = cursor.pull(); item >= 0; item = cursor.pull()) process(item);
  } else {
    const int item = xcd_block(blockIdx.x, gridDim.x, rp.xcd_chunk_log2) * (blockDim.x / kWave) +
                     threadIdx.x / kWave;
    if (item < *n_items) process(item);
  }
}

// ---------------------------------------------------------------------------
// (c) Nearest-higher (ClusteringKernels.hpp:164-206, 247-289). The search box uses
// dm; the acceptance radius is seed_dc for points at or above rhoc*u, else dm.
// A candidate is "higher" when its (rho, tag) key exceeds the point's. Only
// candidates at or below the current best distance can change the result; the
// running threshold below over-approximates that bound, and every candidate that
// passes it goes through the reference's exact comparison.
// ---------------------------------------------------------------------------
template <int M>
__device__ __forceinline__ float prune_threshold(float eff_thr, float delta) {
  if constexpr (MetricTraits<M>::kSqrt) {
    // sqrt_rn(t) <= delta implies t <= delta^2 (1 + 2^-22); delta*delta*(1 + 2^-20)
    // rounded bounds that from above for delta >= 2^-60 (no underflow).
    if (!(delta >= 0x1p-60f)) return eff_thr;
    const float b = (delta * delta) * 0x1.00001p+0f;
    return b < eff_thr ? b : eff_thr;
  } else {
    return delta < eff_thr ? delta : eff_thr;
  }
}
template <int M>
__device__ __forceinline__ double prune_threshold(double eff_thr, double delta) {
  if constexpr (MetricTraits<M>::kSqrt) {
    // Double: t <= delta^2 (1 + 2^-51.9) follows; delta*delta*(1 + 2^-48) rounded
    // bounds it from above for delta >= 2^-500.
    if (!(delta >= 0x1p-500)) return eff_thr;
    const double b = (delta * delta) * 0x1.000000000001p+0;
    return b < eff_thr ? b : eff_thr;
  } else {
    return delta < eff_thr ? delta : eff_thr;
  }
}

// "j is higher than i" (ClusteringKernels.hpp:180-182) from the stored keys. Float
// keys hold (rho, tag); double keys hold rho's order only, so equal densities
// compare the tags here (rho > 0 is the key above that of +0).
__device__ __forceinline__ bool key_higher(uint64_t kj, uint32_t, uint64_t ki, uint32_t, float) {
  return kj > ki;
}
__device__ __forceinline__ bool key_higher(uint64_t kj, uint32_t tj, uint64_t ki, uint32_t ti,
                                           double) {
  return (kj > ki) | ((kj == ki) & (kj > 0x8000000000000000ull) & (tj > ti));
}
__device__ __forceinline__ uint64_t query_key(float rho, uint32_t tag) {
  return rho_tag_key(rho, tag, true);
}
__device__ __forceinline__ uint64_t query_key(double rho, uint32_t) {
  return rho_key_f64(rho, true);
}

// A lower bound of the wave's smallest ordering key. (LDS permutes here and in
// wave_min_f: the DPP form costs more vector instructions, and this scan is short of
// them; measured on MI355X.)
// The smallest high word with a zero low word: never above the smallest key, so
// "a block key above it" keeps every block that could hold a higher candidate.
__device__ __forceinline__ uint64_t wave_min_key_bound(uint64_t v) {
  uint32_t h = static_cast<uint32_t>(v >> 32);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const uint32_t o = static_cast<uint32_t>(__shfl_xor(static_cast<int>(h), off, 64));
    h = o < h ? o : h;
  }
  return static_cast<uint64_t>(h) << 32;
}

// May a block whose largest key is bk hold a candidate higher than the query?
// Float keys decide it exactly; double keys leave equal densities to the tags.
__device__ __forceinline__ bool block_may_be_higher(uint64_t bk, uint64_t ki, float) {
  return bk > ki;
}
__device__ __forceinline__ bool block_may_be_higher(uint64_t bk, uint64_t ki, double) {
  return bk >= ki;
}
__device__ __forceinline__ bool key_maybe_higher(uint64_t kj, uint64_t ki, float) {
  return kj > ki;
}
__device__ __forceinline__ bool key_maybe_higher(uint64_t kj, uint64_t ki, double) {
  return (kj > ki) | ((kj == ki) & (kj > 0x8000000000000000ull));
}

template <int D, int M, class T>
__global__ __launch_bounds__(kMaxNeighbourBlock) void k_nearest_higher(
    const RunParamsT<T> rp, const EventDesc* __restrict__ events, const T* __restrict__ geo,
    const int32_t* __restrict__ toff, const Item* __restrict__ items,
    const int32_t* __restrict__ n_items, const T* __restrict__ sx, int64_t cs,
    const T* __restrict__ ssig, const T* __restrict__ su,
    const uint32_t* __restrict__ stag, const T* __restrict__ srho,
    const uint64_t* __restrict__ skey, const int32_t* __restrict__ qperm,
    int32_t* __restrict__ snh, T* __restrict__ sdelta) {
  constexpr bool kF64 = sizeof(T) == 8;
  constexpr int U = Unroll<D>::U;
  const int item = xcd_block(blockIdx.x, gridDim.x, rp.xcd_chunk_log2) * (blockDim.x / kWave) +
                   threadIdx.x / kWave;
  if (item >= *n_items) return;
  const Item it = items[item];
  const EventDesc ev = events[it.event];
  const GeoT<T> g = event_geo(geo, rp, it.event, ev.nper);
  const int q = it.begin + lane_id();
  const bool active = q < it.end;
  const int s = active ? (qperm ? qperm[q] : q) : -1;  // sorted position of this lane's point

  T xi[D], si[D];
#pragma unroll
  for (int d = 0; d < D; ++d) {
    xi[d] = active ? sx[d * cs + s] : T(0);
    si[d] = (active && rp.has_sigma) ? ssig[d * cs + s] : T(0);
  }
  const T rho_i = active ? srho[s] : T(0);
  const uint32_t tag_i = active ? stag[s] : 0u;
  const uint64_t key_i = active ? query_key(rho_i, tag_i) : ~0ull;
  const T ui = (active && rp.has_u) ? su[s] : T(1);
  const T eff_min = rp.rhoc * ui;
  const bool use_seed = rho_i >= eff_min;
  const T eff = use_seed ? rp.seed_dc : rp.dm;
  const T eff_thr =
      MetricTraits<M>::kSqrt ? (use_seed ? rp.seed_sq_max : rp.dm_sq_max) : eff;

  int lo[D], hi[D];
  search_box<D>(g, xi, si, rp.dm, lo, hi);
  if (!active) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      lo[d] = INT32_MAX;
      hi[d] = INT32_MIN;
    }
  }
  T delta = std::numeric_limits<T>::max();
  int nh = -1;
  T rho_nh = T(0);
  uint32_t tag_nh = 0u;
  T bound = eff_thr;  // prune_threshold(eff_thr, delta)

  // The reference's acceptance test, in candidate order. Its radius test, dist <=
  // eff, holds for every candidate that reaches it (callers pass only v <= bound
  // <= eff_thr, the largest value whose distance is <= eff), so it is left out.
  auto consider = [&](T v, T rj, uint32_t tj, int j) {
    const T dist = finish_distance<M>(v);
    if ((dist < delta) ||
        ((dist == delta) && (nh >= 0) && ((rj > rho_nh) || ((rj == rho_nh) && (tj > tag_nh))))) {
      delta = dist;
      nh = j;
      rho_nh = rj;
      tag_nh = tj;
      bound = prune_threshold<M>(eff_thr, delta);
    }
  };

  // A candidate's density and tag, loaded where its key does not hold them.
  auto accept = [&](T v, uint64_t kj, uint64_t key_in, int j) {
    if (!(key_maybe_higher(kj, key_in, T(0)) && v <= bound)) return;
    if constexpr (kF64) {
      const uint32_t tj = stag[j];
      if (key_higher(kj, tj, key_in, tag_i, T(0))) consider(v, srho[j], tj, j);
    } else {
      const float rj = key_rho(kj);
      consider(v, rj, rj > 0.0f ? static_cast<uint32_t>(kj) : stag[j], j);
    }
  };

  // As in the density stage, a tile's candidates 64 at a time, one per lane: those
  // out of every lane's reach (its bound, here) or not above the wave's smallest key
  // are left out by one ballot; then from the lanes, or through the scalar cache.
  const bool cull = rp.cull != 0;
  const QueryBox<D, T> qb = query_box<D, M>(xi, si, active);
  const uint64_t kmin = wave_min_key_bound(key_i);
  BoxUnion<D> u = box_union(lo, hi);
  do for (int base = 0; base < u.tiles; base += kWave) {
    TileGroup<D> g;
    list_tiles(u, base, ev.nper, rp.wrapped, ev.t_base, toff, &g);
    uint64_t held = ballot(g.j0 < g.j1);
    while (held) {
      const int t = __builtin_ctzll(held);
      held &= held - 1ull;
      const bool in = box_holds(g, t, lo, hi);
      if (ballot(in) == 0ull) continue;
      const int j0 = __builtin_amdgcn_readlane(g.j0, t), j1 = __builtin_amdgcn_readlane(g.j1, t);
      const uint64_t key_in = in ? key_i : ~0ull;
      for (int j = j0; j < j1; j += kWave) {
        const int cnt = min(kWave, j1 - j);
        const bool valid = lane_id() < cnt;
        T cx[D], cg[D];
#pragma unroll
        for (int d = 0; d < D; ++d) {
          cx[d] = valid ? sx[d * cs + j + lane_id()] : T(0);
          cg[d] = (M == M_MAHALANOBIS && valid) ? ssig[d * cs + j + lane_id()] : T(0);
        }
        const uint64_t ck = valid ? skey[j + lane_id()] : 0ull;
        const T bmax = wave_max_f(in ? bound : -std::numeric_limits<T>::infinity());
        uint64_t left = ballot(valid && block_may_be_higher(ck, kmin, T(0)) &&
                               !(cull && out_of_reach<D, M>(qb, cx, cg, rp, bmax)));
        if (left == 0ull) continue;
        if (8 * __popcll(left) < 3 * cnt) {
          while (left) {
            const int i = __builtin_ctzll(left);
            left &= left - 1ull;
            T xj[D], sj[D];
#pragma unroll
            for (int d = 0; d < D; ++d) {
              xj[d] = read_lane(cx[d], i);
              sj[d] = M == M_MAHALANOBIS ? read_lane(cg[d], i) : T(0);
            }
            accept(metric_pair<D, M>(xi, si, xj, sj, rp), read_lane(ck, i), key_in, j + i);
          }
          continue;
        }
        int k = j;
        const int ke = j + cnt;
        for (; k + U <= ke; k += U) {
          // m: the smallest distance among the block's higher candidates (vector
          // selects and minima instead of per-candidate scalar mask logic).
          T v[U];
          T m = std::numeric_limits<T>::infinity();
#pragma unroll
          for (int c = 0; c < U; ++c) {
            v[c] = metric_value<D, M>(xi, si, sx, cs, k + c, ssig, rp);
            const bool h = key_maybe_higher(skey[k + c], key_in, T(0));
            m = fmin_t(m, h ? v[c] : std::numeric_limits<T>::infinity());
          }
          // Most blocks hold no candidate for any lane: one wave-wide test skips them.
          if (ballot(m <= bound) != 0ull) {
#pragma unroll
            for (int c = 0; c < U; ++c) accept(v[c], skey[k + c], key_in, k + c);
          }
        }
        for (; k < ke; ++k)
          accept(metric_value<D, M>(xi, si, sx, cs, k, ssig, rp), skey[k], key_in, k);
      }
    }
  } while (next_tile_run(u));
  if (active) {
    snh[s] = nh;
    sdelta[s] = delta;
  }
}

// ---------------------------------------------------------------------------
// (c') Nearest-higher over Hilbert-ordered candidate blocks. The accepted
// candidate of the reference's scan is the one of smallest distance, equal
// distances going to the larger (rho, tag); with unique tags (the default ones:
// the input index) no two candidates tie on all three, so the result does not
// depend on the order in which candidates are visited. Each tile's candidates
// are laid out in Hilbert order in blocks of kNhBlock with the block's bounding
// box and largest key; a wave skips a block when for each lane either no
// candidate of the block is higher or the box lies beyond the lane's current
// bound. A skipped block holds no candidate that the scan would accept (the box
// bound never exceeds a candidate's computed distance value: rounding is
// monotone), so the results are those of the plain scan.
// ---------------------------------------------------------------------------

// Candidates per register block of the layout scan (a divisor of kNhBlock).
template <int D>
constexpr int nh_sub_block() {
  return D <= 3 ? 8 : 4;
}

// Eight waves per SIMD in 1-D and 2-D: the scan waits on chains of scalar loads,
// so resident waves matter more than registers (measured on MI355X on the
// 4096-event 2-D batch: 12.3 ms with the compiler's own choice, 11.0 ms with
// this bound, 10.2 ms with it and register blocks of 8 candidates instead of
// 16). From 3-D on the bound would spill to scratch; there the compiler chooses
// (equal time on the 2^20-point 3-D event).
template <int D, int M, bool Persistent, class T>
__global__ __launch_bounds__(kMaxNeighbourBlock)
__attribute__((amdgpu_waves_per_eu(D <= 2 ? 8 : 1))) void k_nh_blocks(
    const RunParamsT<T> rp, const EventDesc* __restrict__ events, const T* __restrict__ geo,
    const int32_t* __restrict__ toff, const Item* __restrict__ items,
    int32_t* __restrict__ n_items, const T* __restrict__ sx, int64_t cs,
    const T* __restrict__ ssig, const T* __restrict__ su, const uint32_t* __restrict__ stag,
    const T* __restrict__ srho, const int32_t* __restrict__ qperm, const T* __restrict__ hx,
    int64_t hs,
    const uint64_t* __restrict__ hkey, const int32_t* __restrict__ hidx,
    const T* __restrict__ hbox, const uint64_t* __restrict__ hbkey, int32_t* __restrict__ snh,
    T* __restrict__ sdelta) {
  constexpr int V = nh_sub_block<D>();
  auto process = [&](const int item) {
    const Item it = items[item];
    const EventDesc ev = events[it.event];
    const GeoT<T> g = event_geo(geo, rp, it.event, ev.nper);
    const int q = it.begin + lane_id();
    const bool active = q < it.end;
    const int s = active ? (qperm ? qperm[q] : q) : -1;  // sorted position of this lane's point

    T xi[D], si[D];
  #pragma unroll
    for (int d = 0; d < D; ++d) {
      xi[d] = active ? sx[d * cs + s] : T(0);
      si[d] = (active && rp.has_sigma) ? ssig[d * cs + s] : T(0);
    }
    const T rho_i = active ? srho[s] : T(0);
    const uint32_t tag_i = active ? stag[s] : 0u;
    const uint64_t key_i = active ? query_key(rho_i, tag_i) : ~0ull;
    const T ui = (active && rp.has_u) ? su[s] : T(1);
    const T eff_min = rp.rhoc * ui;
    const bool use_seed = rho_i >= eff_min;
    const T eff = use_seed ? rp.seed_dc : rp.dm;
    const T eff_thr =
        MetricTraits<M>::kSqrt ? (use_seed ? rp.seed_sq_max : rp.dm_sq_max) : eff;

    int lo[D], hi[D];
    search_box<D>(g, xi, si, rp.dm, lo, hi);
    if (!active) {
  #pragma unroll
      for (int d = 0; d < D; ++d) {
        lo[d] = INT32_MAX;
        hi[d] = INT32_MIN;
      }
    }
    T delta = std::numeric_limits<T>::max();
    int64_t nh_slot = -1;  // layout slot of the nearest-higher found so far
    T rho_nh = T(0);
    uint32_t tag_nh = 0u;
    T bound = eff_thr;  // prune_threshold(eff_thr, delta)

    // The reference's acceptance test (ClusteringKernels.hpp:180-195). Its radius
    // test, dist <= eff, holds for every candidate that reaches it: callers pass
    // only v <= bound <= eff_thr, the largest value whose distance is <= eff.
    auto consider = [&](T v, T rj, uint32_t tj, int64_t slot) {
      const T dist = finish_distance<M>(v);
      if ((dist < delta) ||
          ((dist == delta) && (nh_slot >= 0) &&
           ((rj > rho_nh) || ((rj == rho_nh) && (tj > tag_nh))))) {
        delta = dist;
        nh_slot = slot;
        rho_nh = rj;
        tag_nh = tj;
        bound = prune_threshold<M>(eff_thr, delta);
      }
    };

    // One block's candidates, V at a time.
    auto scan_block = [&](int64_t p0, bool in) {
      for (int k0 = 0; k0 < kNhBlock; k0 += V) {
        const int64_t p = p0 + k0;
        T v[V];
        T m = std::numeric_limits<T>::infinity();
  #pragma unroll
        for (int k = 0; k < V; ++k) {
          T xj[D], sj[D];
  #pragma unroll
          for (int d = 0; d < D; ++d) {
            xj[d] = hx[d * hs + p + k];
            sj[d] = T(0);
          }
          v[k] = metric_pair<D, M>(xi, si, xj, sj, rp);
          const bool h = in & key_maybe_higher(hkey[p + k], key_i, T(0));
          m = fmin_t(m, h ? v[k] : std::numeric_limits<T>::infinity());
        }
        if (ballot(m <= bound) != 0ull) {
  #pragma unroll
          for (int k = 0; k < V; ++k) {
            const uint64_t kj = hkey[p + k];
            if (in & key_maybe_higher(kj, key_i, T(0)) & (v[k] <= bound)) {
              if constexpr (sizeof(T) == 4) {
                // Float keys are exact and carry rho, and the tag when rho > 0: no
                // dependent loads on this path.
                const float rj = key_rho(kj);
                const uint32_t tj = rj > 0.0f ? static_cast<uint32_t>(kj) : stag[hidx[p + k]];
                consider(v[k], rj, tj, p + k);
              } else {
                const int j = hidx[p + k];
                const uint32_t tj = stag[j];
                if (key_higher(kj, tj, key_i, tag_i, T(0))) consider(v[k], srho[j], tj, p + k);
              }
            }
          }
        }
      }
    };

    // in: the lane's search box holds tile t. The boxes and keys of up to 64 blocks
    // arrive in one vector load (one block per lane); a wave-wide test against the
    // box, smallest key and largest bound of the lanes that hold the tile drops
    // most blocks at once, and each block left is tested per lane before its scan.
    // The tile's blocks are visited from block sb on, wrapping around: in the own
    // tile sb is the block that holds the wave's first point, whose neighbours
    // settle most bounds before the rest of the tile is tested. The result does
    // not depend on the order (the acceptance test is a strict total order).
    auto scan_tile = [&](int t, bool in, int sb) {
      const int b = toff[t];
      const int nblk = (toff[t + 1] - b + kNhBlock - 1) / kNhBlock;
      const int64_t blk0 = nh_first_block(b, t);
      T qlo[D], qhi[D];
  #pragma unroll
      for (int d = 0; d < D; ++d) {
        T lo = xi[d], hi = xi[d];
        if constexpr (M == M_CHEBYSHEV || M == M_WCHEBYSHEV) {
          lo = box_low(lo);
          hi = box_high(hi);
        }
        qlo[d] = wave_min_f(in ? lo : std::numeric_limits<T>::infinity());
        qhi[d] = wave_max_f(in ? hi : -std::numeric_limits<T>::infinity());
      }
      const uint64_t kmin = wave_min_key_bound(in ? key_i : ~0ull);
      for (int c0 = 0; c0 < nblk; c0 += kWave) {
        const T bmax = wave_max_f(in ? bound : -std::numeric_limits<T>::infinity());
        const int l = lane_id();
        const bool valid = c0 + l < nblk;
        int rl = c0 + (valid ? l : 0) + sb;
        rl -= rl >= nblk ? nblk : 0;
        const int64_t qb = blk0 + rl;
        T bl[D], bh[D];
  #pragma unroll
        for (int d = 0; d < D; ++d) {
          bl[d] = hbox[qb * 2 * D + d];
          bh[d] = hbox[qb * 2 * D + D + d];
        }
        const uint64_t bk = hbkey[qb];
        uint64_t cand = ballot(valid & block_may_be_higher(bk, kmin, T(0)) &
                               (metric_lb<D, M>(qlo, qhi, bl, bh, rp) <= bmax));
        while (cand) {
          const int i = __builtin_ctzll(cand);
          cand &= cand - 1ull;
          T sl[D], sh[D];
  #pragma unroll
          for (int d = 0; d < D; ++d) {
            sl[d] = read_lane(bl[d], i);
            sh[d] = read_lane(bh[d], i);
          }
          const bool need = in & block_may_be_higher(read_lane(bk, i), key_i, T(0)) &
                            (metric_lb<D, M>(xi, xi, sl, sh, rp) <= bound);
          int ri = c0 + i + sb;
          ri -= ri >= nblk ? nblk : 0;
          if (ballot(need) != 0ull) scan_block((blk0 + ri) * kNhBlock, in);
        }
      }
    };

    // The lanes' own tile first: the nearest candidates tighten the bounds early.
    // A lane scans it only if its box holds it: on a wrapped dimension a box wider
    // than half the data's extent can leave it out (the walk below reaches the
    // own tile at bin b or, wrapped, at b + nper).
    const int own = uniform(it.tile);  // wave-uniform: keeps the scan's loads scalar
    {
      bool in_own = active;
      int r = own - ev.t_base;
  #pragma unroll
      for (int d = D - 1; d >= 0; --d) {
        const int b = r % ev.nper;
        r /= ev.nper;
        in_own = in_own && (((lo[d] <= b) && (b <= hi[d])) ||
                            (rp.wrapped[d] && (lo[d] <= b + ev.nper) && (b + ev.nper <= hi[d])));
      }
      if (ballot(in_own) != 0ull) scan_tile(own, in_own, uniform(it.begin - toff[own]) / kNhBlock);
    }
    walk_tiles<D>(lo, hi, ev.nper, rp.wrapped, ev.t_base, [&](int t, bool in) {
      if (t != own) scan_tile(t, in, 0);
    });
    if (active) {
      snh[s] = nh_slot >= 0 ? hidx[nh_slot] : -1;
      sdelta[s] = delta;
    }
  };
  if constexpr (Persistent) {
    ItemCursor cursor(n_items, kQueueNh, rp);
    for (int item = cursor.pull(); item >= 0; item = cursor.pull()) process(item);
  } else {
    const int item = xcd_block(blockIdx.x, gridDim.x, rp.xcd_chunk_log2) * (blockDim.x / kWave) +
                     threadIdx.x / kWave;
    if (item < *n_items) process(item);
  }
}

// ---------------------------------------------------------------------------
// (d) Seed flags (ClusteringKernels.hpp:300-316) and the results in input order,
// one thread per sorted point. A seed sets its bit of bits[], in input order.
// snh is rewritten in place as the follower link of the label stage: -2 for a
// seed, -1 for a point without nearest-higher, else the sorted position of a point
// further up its chain. The thread follows up to kResultHops links for that; those
// it meets may be old or already rewritten, and all lie on its own chain, so the
// label stage's chase ends at the same point whatever order the threads run in.
// ---------------------------------------------------------------------------
constexpr int kResultHops = 3;
template <class T>
__global__ __launch_bounds__(kBlock) void k_results(
    const RunParamsT<T> rp, int n, const int32_t* __restrict__ perm, const T* __restrict__ srho,
    int32_t* snh, const T* __restrict__ sdelta, const T* __restrict__ su, T* __restrict__ rho,
    int32_t* __restrict__ nh, T* __restrict__ delta, int32_t* __restrict__ is_seed,
    uint32_t* __restrict__ bits) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n) return;
  const int i = perm[s];
  const T r = srho[s];
  const int h = snh[s];
  const T u = rp.has_u ? su[s] : T(1);
  const int seed = (h == -1) && (r >= rp.rhoc * u) ? 1 : 0;
  rho[i] = r;
  nh[i] = h >= 0 ? perm[h] : -1;
  if (delta) delta[i] = sdelta[s];
  is_seed[i] = seed;
  if (seed) {
    atomicOr(&bits[i >> 5], 1u << (i & 31));
    snh[s] = -2;
    return;
  }
  if (h < 0) return;
  int l = h;
  for (int k = 0; k < kResultHops; ++k) {
    const int next = snh[l];
    if (next < 0) break;
    l = next;
  }
  if (l != h) snh[s] = l;
}

// Seeds before every word of bits[] and their total: up to kRankWords words by one
// workgroup (rank_counts), more by k_seed_counts and the general scan.
static __global__ __launch_bounds__(kRankBlock) void k_seed_ranks(const uint32_t* __restrict__ bits,
                                                                  int words,
                                                                  int32_t* __restrict__ before,
                                                                  int32_t* __restrict__ total) {
  rank_counts(
      [&](int w, int (&c)[4]) {
        uint4 v = make_uint4(0u, 0u, 0u, 0u);
        if (w + 3 < words) {
          v = *reinterpret_cast<const uint4*>(bits + w);
        } else if (w < words) {
          v.x = bits[w];
          if (w + 1 < words) v.y = bits[w + 1];
          if (w + 2 < words) v.z = bits[w + 2];
        }
        c[0] = __popc(v.x);
        c[1] = __popc(v.y);
        c[2] = __popc(v.z);
        c[3] = __popc(v.w);
      },
      words, before, total);
}
static __global__ __launch_bounds__(kBlock) void k_seed_counts(const uint32_t* __restrict__ bits,
                                                               int words,
                                                               int32_t* __restrict__ count) {
  const int w = blockIdx.x * kBlock + threadIdx.x;
  if (w < words) count[w] = __popc(bits[w]);
}

// ---------------------------------------------------------------------------
// (d fused) With the per-event tile build, one workgroup per event does the seed
// stage of k_results, numbers the event's seeds in input order through a bit
// per point in LDS (one popcount scan over the bits: the rank of a seed among
// the event's seeds, stored in rank[i]), counts them (event_seeds[e]) and
// shortens the follower links by pointer jumping.
// The seeds of earlier events are added by the label stage from an exclusive
// scan of event_seeds. The seed flags and links are settled in sorted order;
// the results are then written in input order, each point's sorted values
// gathered through iperm, so that every store is coalesced. An event of at
// most kEvtLdsLinks points keeps its links in LDS as 16-bit event positions:
// the results pass reads them there, the jumping passes run there (more of
// them, as they cost no memory traffic) and the links go back to memory once.
// ---------------------------------------------------------------------------
constexpr int kLinkJumpPasses = 4;     // pointer-jumping passes in memory before the label chase
constexpr int kLdsJumpPasses = 6;      // in LDS: chains of up to 64 links end at their root
constexpr int kEvtLdsLinks = 1 << 15;  // events whose links fit LDS (16-bit positions)
constexpr int kEvtBitWords = kEvtMaxPoints / 32;
constexpr int kLdsBitWords = kEvtLdsLinks / 32;
// One LDS pool: the seed bits of any event, or the bits and links of a small one
// (two workgroups per CU, as the 16 waves of each allow).
constexpr int kSeedPoolWords =
    kEvtBitWords > kLdsBitWords + kEvtLdsLinks / 2 ? kEvtBitWords : kLdsBitWords + kEvtLdsLinks / 2;
static_assert(kEvtBitWords % kEvtBlock == 0, "bit words per thread");
static_assert(kEvtLdsLinks <= 32768, "links are 16-bit event positions");

template <class T>
__global__ __launch_bounds__(kEvtBlock) void k_event_seeds(
    const RunParamsT<T> rp, const EventDesc* __restrict__ events, const int32_t* __restrict__ order,
    const int32_t* __restrict__ perm, const int32_t* __restrict__ iperm,
    const T* __restrict__ srho, int32_t* __restrict__ snh, const T* __restrict__ sdelta,
    const T* __restrict__ su, T* __restrict__ rho, int32_t* __restrict__ nh, T* __restrict__ delta,
    int32_t* __restrict__ is_seed, int32_t* __restrict__ rank, int32_t* __restrict__ event_seeds,
    int32_t* __restrict__ cluster) {
  constexpr int kWordsPerThread = kEvtBitWords / kEvtBlock;
  __shared__ uint32_t pool[kSeedPoolWords];
  __shared__ int32_t wsum[kEvtWaves];
  uint32_t* bits = pool;
  int16_t* links = reinterpret_cast<int16_t*>(pool + kLdsBitWords);
  const int e = order[blockIdx.x];
  const EventDesc ev = events[e];
  const int b0 = ev.p_off, n = ev.n;
  const bool in_lds = n <= kEvtLdsLinks;
  const int n_words = in_lds ? kLdsBitWords : kEvtBitWords;  // bit words in use
  const int w = threadIdx.x / kWave;
  const int lane = lane_id();
  for (int k = threadIdx.x; k < n_words; k += kEvtBlock) bits[k] = 0u;
  __syncthreads();
  // Seed flags (ClusteringKernels.hpp:300-316) in sorted order: a seed's link
  // becomes -2, and its bit (input order) is set.
#pragma unroll 4
  for (int k = threadIdx.x; k < n; k += kEvtBlock) {
    const int s = b0 + k;
    const int h = snh[s];
    const T u = rp.has_u ? su[s] : T(1);
    const bool seed = (h == -1) && (srho[s] >= rp.rhoc * u);
    if (in_lds) links[k] = static_cast<int16_t>(seed ? -2 : (h >= 0 ? h - b0 : h));
    if (seed) {
      if (!in_lds) snh[s] = -2;
      const int i = perm[s] - b0;
      atomicOr(&bits[i >> 5], 1u << (i & 31));
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");  // the -2 links
  __syncthreads();
  // Results in input order.
#pragma unroll 4
  for (int k = threadIdx.x; k < n; k += kEvtBlock) {
    const int i = b0 + k;
    const int s = iperm[i];
    int h;
    if (in_lds) {
      h = links[s - b0];
      h = h >= 0 ? h + b0 : h;
    } else {
      h = snh[s];
    }
    rho[i] = srho[s];
    nh[i] = h >= 0 ? perm[h] : -1;
    if (delta) delta[i] = sdelta[s];
    is_seed[i] = h == -2 ? 1 : 0;
  }
  // Ranks in input order: each thread owns kWordsPerThread consecutive words
  // (words past the bits in use count nothing).
  const int w0 = threadIdx.x * kWordsPerThread;
  int mine = 0;
#pragma unroll
  for (int k = 0; k < kWordsPerThread; ++k) mine += w0 + k < n_words ? __popc(bits[w0 + k]) : 0;
  int incl = mine;
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const int y = __shfl_up(incl, off, 64);
    if (lane >= off) incl += y;
  }
  if (lane == kWave - 1) wsum[w] = incl;
  __syncthreads();
  int before = 0, total = 0;
  for (int k = 0; k < kEvtWaves; ++k) {
    before += k < w ? wsum[k] : 0;
    total += wsum[k];
  }
  int run = before + incl - mine;
#pragma unroll
  for (int k = 0; k < kWordsPerThread; ++k) {
    uint32_t word = w0 + k < n_words ? bits[w0 + k] : 0u;
    while (word) {
      const int bit = __builtin_ctz(word);
      word &= word - 1u;
      const int ii = (w0 + k) * 32 + bit;  // the seed's input position in the event
      if (in_lds) {
        // The event's seed list in rank order, and the seed's link: its rank as
        // a code (-3 - rank) that the jumping passes carry to its followers.
        rank[b0 + run] = b0 + ii;
        links[iperm[b0 + ii] - b0] = static_cast<int16_t>(-3 - run);
        ++run;
      } else {
        rank[b0 + ii] = run++;
      }
    }
  }
  if (threadIdx.x == 0) event_seeds[e] = total;
  // Pointer jumping on the event's links: a pass replaces a link by its target's link
  // when that target is itself a follower, which halves every chain (at least); any
  // interleaving of the updates leaves every link on its own chain.
  if (in_lds) {
    // A link is a position, a seed's code or -1 (the end of an outlier chain), and
    // every point shares the label of what its link names; replacing a position
    // by that point's link keeps this, in any interleaving. After the passes the
    // few chains longer than 2^kLdsJumpPasses are finished by a chase in LDS, and
    // each point's label within the event goes to cluster[] in input order (the
    // label stage adds the event's offset).
    for (int pass = 0; pass < kLdsJumpPasses; ++pass) {
      __syncthreads();
      for (int k = threadIdx.x; k < n; k += kEvtBlock) {
        const int l = links[k];
        if (l >= 0) links[k] = links[l];
      }
    }
    __syncthreads();
#pragma unroll 4
    for (int k = threadIdx.x; k < n; k += kEvtBlock) {
      const int i = b0 + k;
      int l = links[iperm[i] - b0];
      while (l >= 0) l = links[l];
      cluster[i] = l <= -3 ? -3 - l : -1;
    }
  } else {
    for (int pass = 0; pass < kLinkJumpPasses; ++pass) {
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
      __syncthreads();
      for (int k = threadIdx.x; k < n; k += kEvtBlock) {
        const int s = b0 + k;
        const int l = snh[s];
        if (l < 0) continue;
        const int l2 = snh[l];
        if (l2 >= 0) snh[s] = l2;
      }
    }
  }
}

// The same for a lone event of at most kLoneMaxPoints points, whose labels, seeds and
// total are final: no label stage follows. Everything that is read in another order
// than it was loaded goes through LDS (the kernel above: 16.6 us for 5,003 points, 5.3
// for 300; this one: 9.0 and 4.1).
template <class T>
__global__ __launch_bounds__(kEvtBlock) void k_lone_seeds(
    const RunParamsT<T> rp, const EventDesc ev, const int32_t* __restrict__ perm,
    const int32_t* __restrict__ iperm, const T* __restrict__ srho, const int32_t* __restrict__ snh,
    const T* __restrict__ sdelta, const T* __restrict__ su, T* __restrict__ rho,
    int32_t* __restrict__ nh, T* __restrict__ delta, int32_t* __restrict__ is_seed,
    int32_t* __restrict__ total, int32_t* __restrict__ seeds,
    int32_t* __restrict__ event_of_cluster, int32_t* __restrict__ cluster) {
  constexpr int R = kLoneRounds;
  constexpr int kWords = kLoneMaxPoints / 32;
  static_assert(kWords <= kEvtBlock, "one word per thread");
  __shared__ uint32_t bits[kWords];            // a bit per seed, in input order
  __shared__ int16_t links[kLoneMaxPoints];    // k_event_seeds' links and codes
  __shared__ uint16_t input[kLoneMaxPoints];   // sorted position -> input index
  __shared__ uint16_t sorted[kLoneMaxPoints];  // input index -> sorted position
  __shared__ T lrho[kLoneMaxPoints];
  __shared__ int32_t wsum[kEvtWaves];
  const int n = ev.n;
  const int w = threadIdx.x / kWave;
  const int lane = lane_id();
  const int rounds = (n + kEvtBlock - 1) / kEvtBlock;
  if (threadIdx.x < kWords) bits[threadIdx.x] = 0u;
  int h[R], p[R], q[R];
  T ro[R], u[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if (r >= rounds) break;
    const int k = min(static_cast<int>(threadIdx.x) + r * kEvtBlock, n - 1);
    h[r] = snh[k];
    p[r] = perm[k];
    q[r] = iperm[k];
    ro[r] = srho[k];
    u[r] = rp.has_u ? su[k] : T(1);
  }
  __syncthreads();
  // Seed flags (ClusteringKernels.hpp:300-316), in sorted order.
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int k = static_cast<int>(threadIdx.x) + r * kEvtBlock;
    if (k >= n) break;
    const bool seed = (h[r] == -1) && (ro[r] >= rp.rhoc * u[r]);
    links[k] = static_cast<int16_t>(seed ? -2 : h[r]);
    lrho[k] = ro[r];
    input[k] = static_cast<uint16_t>(p[r]);
    sorted[k] = static_cast<uint16_t>(q[r]);
    if (seed) atomicOr(&bits[p[r] >> 5], 1u << (p[r] & 31));
  }
  __syncthreads();
  // Results in input order.
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int k = static_cast<int>(threadIdx.x) + r * kEvtBlock;
    if (k >= n) break;
    const int l = links[q[r]];
    rho[k] = lrho[q[r]];
    nh[k] = l >= 0 ? input[l] : -1;
    is_seed[k] = l == -2 ? 1 : 0;
  }
  if (delta) {
    T v[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if (r >= rounds) break;
      v[r] = sdelta[q[r]];
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int k = static_cast<int>(threadIdx.x) + r * kEvtBlock;
      if (k >= n) break;
      delta[k] = v[r];
    }
  }
  // Ranks of the seeds in input order.
  uint32_t word = threadIdx.x < kWords ? bits[threadIdx.x] : 0u;
  const int mine = __popc(word);
  int incl = mine;
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const int y = __shfl_up(incl, off, 64);
    if (lane >= off) incl += y;
  }
  if (lane == kWave - 1) wsum[w] = incl;
  __syncthreads();  // and the results have read the links
  int run = incl - mine;
  for (int k = 0; k < w; ++k) run += wsum[k];
  if (threadIdx.x == kEvtBlock - 1) *total = run;  // no words: all seeds are before it
  while (word) {
    const int ii = static_cast<int>(threadIdx.x) * 32 + __builtin_ctz(word);
    word &= word - 1u;
    seeds[run] = ii;
    if (event_of_cluster) event_of_cluster[run] = ev.index;
    links[sorted[ii]] = static_cast<int16_t>(-3 - run);
    ++run;
  }
  // Pointer jumping, as in k_event_seeds, then the label of what each link names.
  for (int pass = 0; pass < kLdsJumpPasses; ++pass) {
    __syncthreads();
    for (int k = threadIdx.x; k < n; k += kEvtBlock) {
      const int l = links[k];
      if (l >= 0) links[k] = links[l];
    }
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int k = static_cast<int>(threadIdx.x) + r * kEvtBlock;
    if (k >= n) break;
    int l = links[q[r]];
    while (l >= 0) l = links[l];
    cluster[k] = l <= -3 ? -3 - l : -1;
  }
}

// ---------------------------------------------------------------------------
// (e) Labels: seeds take their rank in input order (the serial push_back order,
// ClusteringKernels.hpp:310, 318-327); followers chase nearest_higher to a seed
// or to a point without one (:329-343). The chase runs in tile-sorted space,
// where a chain stays among neighbouring tiles of one event. An event occupies
// the same range of positions in input and sorted order.
// ---------------------------------------------------------------------------
// After the fused seed stage, rank[i] of a seed i is its rank within its event, to
// which the seeds of the earlier events (event_offsets[e]) are added here. Chains
// are chased from sorted positions, so their first links are read in order and the
// label stores scatter within each event (chasing from input order instead
// stores in order but reads twice the bytes, for the same time on MI355X).
// An event the fused seed stage resolved in LDS (at most kEvtLdsLinks points)
// has its labels within the event in cluster[] already and its seed list in
// rank[p_off, p_off + event_seeds[e]): only the offset is added.
static __global__ __launch_bounds__(kBlock) void k_event_labels(
    const Chunk* __restrict__ chunks, const EventDesc* __restrict__ events,
    const int32_t* __restrict__ perm, const int32_t* __restrict__ link,
    const int32_t* __restrict__ rank, const int32_t* __restrict__ event_offsets,
    const int32_t* __restrict__ event_seeds, int32_t* __restrict__ cluster,
    int32_t* __restrict__ seeds, int32_t* __restrict__ event_of_cluster, int local_ids) {
  const Chunk ch = chunks[blockIdx.x];
  const EventDesc ev = events[ch.event];
  const int first = event_offsets[ch.event];
  if (ev.n <= kEvtLdsLinks) {
    const int count = event_seeds[ch.event];
    for (int p = ch.begin + threadIdx.x; p < ch.end; p += kBlock) {
      const int c = cluster[p];
      if (c >= 0 && !local_ids) cluster[p] = c + first;
      const int r = p - ev.p_off;
      if (r < count) {
        seeds[first + r] = rank[p];
        if (event_of_cluster) event_of_cluster[first + r] = ev.index;
      }
    }
    return;
  }
  const int sub = local_ids ? first : 0;
  for (int s = ch.begin + threadIdx.x; s < ch.end; s += kBlock) {
    int cur = s;
    int nx = link[cur];
    while (nx >= 0) {
      cur = nx;
      nx = link[cur];
    }
    const int i = perm[s];
    const int c = (nx == -2) ? rank[perm[cur]] + first : -1;
    cluster[i] = c >= 0 ? c - sub : -1;
    if (cur == s && nx == -2) {
      seeds[c] = i;
      if (event_of_cluster) event_of_cluster[c] = ev.index;
    }
  }
}

// The same after k_results: a seed's rank over the whole batch is the number of seed
// bits before its own. 2^parts_log2 workgroups share a chunk: as many as a full one has
// rounds, or one where most are far from full.
static __global__ __launch_bounds__(kBlock) void k_labels(
    const Chunk* __restrict__ chunks, const EventDesc* __restrict__ events,
    const int32_t* __restrict__ perm, const int32_t* __restrict__ link,
    const uint32_t* __restrict__ bits, const int32_t* __restrict__ before,
    int32_t* __restrict__ cluster, int32_t* __restrict__ seeds,
    int32_t* __restrict__ event_of_cluster, int local_ids, int parts_log2) {
  auto rank = [&](int i) {
    return before[i >> 5] + __popc(bits[i >> 5] & ((1u << (i & 31)) - 1u));
  };
  const Chunk ch = chunks[blockIdx.x >> parts_log2];
  const EventDesc ev = events[ch.event];
  const int part = static_cast<int>(blockIdx.x) & ((1 << parts_log2) - 1);
  for (int s = ch.begin + part * kBlock + static_cast<int>(threadIdx.x); s < ch.end;
       s += kBlock << parts_log2) {
    int cur = s;
    int nx = link[cur];
    while (nx >= 0) {
      cur = nx;
      nx = link[cur];
    }
    const int i = perm[s];
    const int c = (nx == -2) ? rank(perm[cur]) : -1;
    cluster[i] = c >= 0 ? c - (local_ids ? rank(ev.p_off) : 0) : -1;
    if (cur == s && nx == -2) {
      seeds[c] = i;
      if (event_of_cluster) event_of_cluster[c] = ev.index;
    }
  }
}

}  // namespace clue_dev

#include "clue_team.h"

namespace clue_dev {

// ---------------------------------------------------------------------------
// Dispatch over (D, metric, kernel).
// ---------------------------------------------------------------------------
// Compute units of the current device (cached per device).
inline int device_cus() {
  static int cus[64] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (cus[dev] == 0) {
    int v = 0;
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        v <= 0)
      v = 256;
    cus[dev] = v;
  }
  return cus[dev];
}

template <class T>
struct NeighbourLaunch {
  const RunParamsT<T>* rp;
  const BatchBuffersT<T>* bb;
  int64_t cs;
  unsigned grid;             // one wave per work item (the grid form)
  unsigned grid_persistent;  // rp.persistent waves per CU (kernels with persistent variants)
  unsigned block;  // threads per workgroup of the neighbour stages
  unsigned grid_team;  // one workgroup per work item (rp.team, clue_team.h)
  hipStream_t s;
};

// Persistent waves (the device work-item queues) are built for 1-3 dimensions,
// the ones the tuning table covers; other dimensions take the grid form.
template <int D>
constexpr bool kPersistentBuilt = D <= 3;

template <int D, int M, int K, class T>
static void launch_density_dmk(const NeighbourLaunch<T>& L) {
  const BatchBuffersT<T>& b = *L.bb;
  auto go = [&](auto kern, unsigned grid) {
    hipLaunchKernelGGL(kern, dim3(grid), dim3(L.block), 0, L.s, *L.rp, b.events, b.geo, b.toff,
                       b.items, b.n_items, b.sorted.x[0], L.cs, b.sorted.w, b.sorted.fw,
                       b.sorted.sigma[0], b.sorted.tag, b.qfine, b.srho, b.skey, b.tbox,
                       b.hkey, b.hbkey);
  };
  if constexpr (kPersistentBuilt<D>) {
    if (L.rp->persistent > 0) {
      go(k_density<D, M, K, true, T>, L.grid_persistent);
      return;
    }
  }
  go(k_density<D, M, K, false, T>, L.grid);
}

template <int D, int M, class T>
static void launch_density_dm(const NeighbourLaunch<T>& L) {
  if (L.rp->team) {
    const BatchBuffersT<T>& b = *L.bb;
    hipLaunchKernelGGL((k_density_team<D, M, T>), dim3(L.grid_team), dim3(kTeam * kWave), 0, L.s,
                       *L.rp, b.events, b.geo, b.toff, b.items, b.sorted.x[0], L.cs, b.sorted.w,
                       b.sorted.fw, b.sorted.sigma[0], b.sorted.tag, b.qfine, b.tbox,
                       b.srho, b.skey);
    return;
  }
  switch (L.rp->kernel) {
    case K_FLAT: launch_density_dmk<D, M, K_FLAT>(L); break;
    case K_EXP:
      if (L.rp->kp1 == T(1))
        launch_density_dmk<D, M, K_EXP_UNIT>(L);
      else
        launch_density_dmk<D, M, K_EXP>(L);
      break;
    default: {
      // Float folds the power of two into the exp's constants (|s| <= 8 only).
      const bool pow2 = sizeof(T) == 4 ? L.rp->gauss_fold != 0 : L.rp->gauss_pow2 != 0;
      if (pow2 && L.rp->kp1 == T(1))
        launch_density_dmk<D, M, K_GAUSS2_UNIT>(L);
      else if (pow2)
        launch_density_dmk<D, M, K_GAUSS2>(L);
      else
        launch_density_dmk<D, M, K_GAUSS>(L);
      break;
    }
  }
}

template <int D, int M, class T>
static void launch_nh_dm(const NeighbourLaunch<T>& L) {
  const BatchBuffersT<T>& b = *L.bb;
  if (L.rp->team) {
    hipLaunchKernelGGL((k_nearest_higher_team<D, M, T>), dim3(L.grid_team), dim3(kTeam * kWave), 0,
                       L.s, *L.rp, b.events, b.geo, b.toff, b.items, b.sorted.x[0], L.cs,
                       b.sorted.sigma[0], b.sorted.u, b.sorted.tag, b.srho, b.skey, b.qfine,
                       b.tbox, b.snh, b.sdelta);
    return;
  }
  hipLaunchKernelGGL((k_nearest_higher<D, M, T>), dim3(L.grid), dim3(L.block), 0, L.s, *L.rp,
                     b.events, b.geo, b.toff, b.items, b.n_items, b.sorted.x[0], L.cs,
                     b.sorted.sigma[0], b.sorted.u, b.sorted.tag, b.srho, b.skey, b.qfine,
                     b.snh, b.sdelta);
}

template <int D, int M, class T>
static void launch_nh_blocks_dm(const NeighbourLaunch<T>& L) {
  const BatchBuffersT<T>& b = *L.bb;
  auto go = [&](auto kern, unsigned grid) {
    hipLaunchKernelGGL(kern, dim3(grid), dim3(L.block), 0, L.s, *L.rp, b.events, b.geo, b.toff,
                       b.items, b.n_items, b.sorted.x[0], L.cs, b.sorted.sigma[0], b.sorted.u,
                       b.sorted.tag, b.srho, b.qfine, b.hx, b.h_stride, b.hkey, b.hidx,
                       b.hbox, b.hbkey, b.snh, b.sdelta);
  };
  if constexpr (kPersistentBuilt<D>) {
    if (L.rp->persistent > 0) {
      go(k_nh_blocks<D, M, true, T>, L.grid_persistent);
      return;
    }
  }
  go(k_nh_blocks<D, M, false, T>, L.grid);
}

// Nearest-higher over the block layout, which the query order and the density stage
// have written.
template <int D, class T>
static void launch_nh_blocks_d(const NeighbourLaunch<T>& L) {
  switch (L.rp->metric) {
    case M_EUCLID: launch_nh_blocks_dm<D, M_EUCLID>(L); break;
    case M_WEUCLID: launch_nh_blocks_dm<D, M_WEUCLID>(L); break;
    case M_PERIODIC: launch_nh_blocks_dm<D, M_PERIODIC>(L); break;
    case M_PERIODIC_LAST:
      if constexpr (D >= 2) launch_nh_blocks_dm<D, M_PERIODIC_LAST>(L);
      break;
    case M_MANHATTAN: launch_nh_blocks_dm<D, M_MANHATTAN>(L); break;
    case M_CHEBYSHEV: launch_nh_blocks_dm<D, M_CHEBYSHEV>(L); break;
    default: launch_nh_blocks_dm<D, M_WCHEBYSHEV>(L); break;
  }
}

// Defined here, instantiated per dimension in clue_neighbour.hip (one object per
// dimension, compiled in parallel); the pipeline's translation units only call it.
template <int D, class T>
void launch_neighbour_d(const NeighbourLaunch<T>& L, bool density) {
  if (!density && L.rp->nh_blocks && L.rp->metric != M_MAHALANOBIS) {
    launch_nh_blocks_d<D>(L);
    return;
  }
#define CLUE_METRIC_CASE(MID)               \
  case MID:                                 \
    if (density)                            \
      launch_density_dm<D, MID>(L);         \
    else                                    \
      launch_nh_dm<D, MID>(L);              \
    break;
  switch (L.rp->metric) {
    CLUE_METRIC_CASE(M_EUCLID)
    CLUE_METRIC_CASE(M_WEUCLID)
    CLUE_METRIC_CASE(M_PERIODIC)
    case M_PERIODIC_LAST:
      if constexpr (D >= 2) {
        if (density)
          launch_density_dm<D, M_PERIODIC_LAST>(L);
        else
          launch_nh_dm<D, M_PERIODIC_LAST>(L);
      }
      break;
    CLUE_METRIC_CASE(M_MANHATTAN)
    CLUE_METRIC_CASE(M_CHEBYSHEV)
    CLUE_METRIC_CASE(M_WCHEBYSHEV)
    default:
      if (density)
        launch_density_dm<D, M_MAHALANOBIS>(L);
      else
        launch_nh_dm<D, M_MAHALANOBIS>(L);
  }
#undef CLUE_METRIC_CASE
}

#define CLUE_NEIGHBOUR_EXTERN(D)                                                          \
  extern template void launch_neighbour_d<D, float>(const NeighbourLaunch<float>&, bool); \
  extern template void launch_neighbour_d<D, double>(const NeighbourLaunch<double>&, bool);
CLUE_NEIGHBOUR_EXTERN(1)
CLUE_NEIGHBOUR_EXTERN(2)
CLUE_NEIGHBOUR_EXTERN(3)
CLUE_NEIGHBOUR_EXTERN(4)
CLUE_NEIGHBOUR_EXTERN(5)
CLUE_NEIGHBOUR_EXTERN(6)
CLUE_NEIGHBOUR_EXTERN(7)
CLUE_NEIGHBOUR_EXTERN(8)
CLUE_NEIGHBOUR_EXTERN(9)
CLUE_NEIGHBOUR_EXTERN(10)
#undef CLUE_NEIGHBOUR_EXTERN

template <class T>
static TileSetup tile_setup_of(const NeighbourLaunch<T>& L) {
  const BatchBuffersT<T>& b = *L.bb;
  const bool chebyshev = L.rp->metric == M_CHEBYSHEV || L.rp->metric == M_WCHEBYSHEV;
  return {b.events, b.n_events, b.items, b.icount, b.max_items, chebyshev ? 1 : 0};
}

constexpr int kOrderTilesAlone = 2048;  // 8 workgroups of 8 waves per CU

template <int D, class T>
static void launch_query_order_d(const NeighbourLaunch<T>& L) {
  const BatchBuffersT<T>& b = *L.bb;
  const TileSetup setup = tile_setup_of(L);
  // Tiles per workgroup, whose sorts run one after the other. Few tiles leave CUs idle,
  // so each takes a workgroup of its own (5,003 points in 2-D: 13.4 us with eight
  // tiles, 7.2 with two, 5.7 with one; 16,384 points 13.2 -> 6.1, 20,011 in 6-D 12.2 ->
  // 8.4). A large lone event's dense tiles are too uneven for eight in a row (2^20
  // points in 2-D: 72 us, 58 with two, 65 with one); batches are not (the 4096-event
  // batch: 1.05 ms with four, 1.22 with two), nor tiles that mostly need no sort.
  const int64_t tiles = b.n_tiles_total;
  const bool uneven = b.n_events == 1 && b.n_total >= kWave * tiles;
  auto go = [&](auto kern, int waves) {
    const int per = tiles <= kOrderTilesAlone ? 1 : uneven ? 2 : waves;
    hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>((tiles + per - 1) / per)),
                       dim3(waves * kWave), 0, L.s, *L.rp, setup, b.tbox, b.n_items, b.geo, b.toff,
                       b.n_tiles_total, per, b.sorted.x[0], L.cs, b.qfine, b.hx, b.h_stride, b.hidx,
                       b.hbox);
  };
  const bool fine = !L.rp->team;
  if (b.n_events == 1)
    go(fine ? k_query_order<D, 8, true, T> : k_query_order<D, 8, false, T>, 8);
  else
    go(fine ? k_query_order<D, 4, true, T> : k_query_order<D, 4, false, T>, 4);
}

template <int D, class T>
static void launch_tile_setup_d(const NeighbourLaunch<T>& L) {
  const BatchBuffersT<T>& b = *L.bb;
  const unsigned grid = static_cast<unsigned>((b.n_tiles_total + kWaves - 1) / kWaves);
  const TileSetup setup = tile_setup_of(L);
  hipLaunchKernelGGL((k_tile_setup<D, T>), dim3(grid), dim3(kBlock), 0, L.s, setup, b.toff,
                     b.n_tiles_total, b.sorted.x[0], L.cs, b.tbox, b.n_items);
}

template <class T>
static void launch_tile_setup(const NeighbourLaunch<T>& L) {
  switch (L.rp->D) {
    case 1: launch_tile_setup_d<1>(L); break;
    case 2: launch_tile_setup_d<2>(L); break;
    case 3: launch_tile_setup_d<3>(L); break;
    case 4: launch_tile_setup_d<4>(L); break;
    case 5: launch_tile_setup_d<5>(L); break;
    case 6: launch_tile_setup_d<6>(L); break;
    case 7: launch_tile_setup_d<7>(L); break;
    case 8: launch_tile_setup_d<8>(L); break;
    case 9: launch_tile_setup_d<9>(L); break;
    default: launch_tile_setup_d<10>(L); break;
  }
}

// The query order of both neighbour stages, with the work items and tile boxes.
template <class T>
static void launch_query_order(const NeighbourLaunch<T>& L) {
  switch (L.rp->D) {
    case 1: launch_query_order_d<1>(L); break;
    case 2: launch_query_order_d<2>(L); break;
    case 3: launch_query_order_d<3>(L); break;
    case 4: launch_query_order_d<4>(L); break;
    case 5: launch_query_order_d<5>(L); break;
    case 6: launch_query_order_d<6>(L); break;
    case 7: launch_query_order_d<7>(L); break;
    case 8: launch_query_order_d<8>(L); break;
    case 9: launch_query_order_d<9>(L); break;
    default: launch_query_order_d<10>(L); break;
  }
}

template <class T>
static void launch_neighbour(const NeighbourLaunch<T>& L, bool density) {
  switch (L.rp->D) {
    case 1: launch_neighbour_d<1>(L, density); break;
    case 2: launch_neighbour_d<2>(L, density); break;
    case 3: launch_neighbour_d<3>(L, density); break;
    case 4: launch_neighbour_d<4>(L, density); break;
    case 5: launch_neighbour_d<5>(L, density); break;
    case 6: launch_neighbour_d<6>(L, density); break;
    case 7: launch_neighbour_d<7>(L, density); break;
    case 8: launch_neighbour_d<8>(L, density); break;
    case 9: launch_neighbour_d<9>(L, density); break;
    default: launch_neighbour_d<10>(L, density); break;
  }
}


template <class T>
void launch_pipeline(const RunParamsT<T>& rp, const PointArraysT<T>& in, const BatchBuffersT<T>& bb,
                     const ResultArraysT<T>& out, hipStream_t s, const StageHook* hook) {
  auto mark = [&](int stage) {
    if (hook && hook->mark) hook->mark(hook->self, stage, s);
  };
  const int D = rp.D;
  const int n = bb.n_total;
  CoordPtrs<T> cp{};
  for (int d = 0; d < D; ++d) cp.x[d] = in.x[d];

  // (a) tiles
  mark(kStageExtremes);
  if (bb.event_order) {
    // Every event fits one workgroup's tile counters: the fused per-event build.
    mark(kStageTiles);
    launch_event_tiles(rp, in, bb, s);
  } else {
  hipLaunchKernelGGL(k_extremes<T>, dim3(bb.n_chunks), dim3(kBlock), 0, s, cp, D, bb.lone,
                     bb.chunks, bb.events, bb.ext_group, bb.ext);
  mark(kStageTiles);
  const RadixPlan digits = radix_plan(bb.key_bits);
  const bool by_chunk = bb.sort_by_chunk != 0;
  hipLaunchKernelGGL((by_chunk ? k_tile_keys<T, true> : k_tile_keys<T, false>), dim3(bb.n_chunks),
                     dim3(by_chunk ? 1024 : 256), 0, s, cp, rp, bb.chunks, bb.events, bb.ext_group,
                     bb.ext, bb.geo, bb.keys0, digits.bits, bb.rs_hist);
  bool in_first = true;
  radix_sort_pairs(bb.keys0, bb.vals0, bb.keys1, bb.vals1, n, bb.key_bits, bb.rs_hist, by_chunk,
                   by_chunk ? bb.chunks : nullptr, bb.n_chunks, nullptr, 0, &in_first, s);
  const uint32_t* skeys = in_first ? bb.keys0 : bb.keys1;
  const int32_t* sperm = in_first ? bb.vals0 : bb.vals1;
  GatherArgs<T> ga;
  ga.in = in;
  ga.out = bb.sorted;
  ga.cs = 0;
  hipLaunchKernelGGL(k_gather<T>, dim3((n + kBlock - 1) / kBlock), dim3(kBlock), 0, s, ga, rp, skeys,
                     sperm, n, bb.n_tiles_total, bb.toff,
                     reinterpret_cast<uint32_t*>(bb.flag));
  }

  NeighbourLaunch<T> L;
  L.rp = &rp;
  L.bb = &bb;
  L.cs = bb.sorted_stride;
  const int waves = rp.block_waves;
  L.block = static_cast<unsigned>(waves * kWave);
  const int64_t blocks = (bb.max_items + waves - 1) / waves;
  L.grid = static_cast<unsigned>((blocks + kXcds - 1) / kXcds * kXcds);
  // Persistent waves: rp.persistent per CU, never more than the grid form's.
  const int64_t pblocks = std::min<int64_t>(
      blocks, (static_cast<int64_t>(device_cus()) * std::max(rp.persistent, 0) + waves - 1) / waves);
  L.grid_persistent = static_cast<unsigned>((pblocks + kXcds - 1) / kXcds * kXcds);
  L.grid_team =
      static_cast<unsigned>((static_cast<int64_t>(bb.max_items) + kXcds - 1) / kXcds * kXcds);
  L.s = s;
  if (bb.icount && bb.n_tiles_total <= kRankWords) {
    hipLaunchKernelGGL(k_item_ranks, dim3(1), dim3(kRankBlock), 0, s, bb.toff, bb.n_tiles_total,
                       bb.icount, bb.n_items);
  } else if (bb.icount) {
    hipLaunchKernelGGL(k_item_count, dim3((bb.n_tiles_total + kBlock - 1) / kBlock), dim3(kBlock),
                       0, s, bb.toff, bb.n_tiles_total, bb.icount);
    scan_exclusive(bb.icount, bb.icount, bb.n_tiles_total, bb.scan_tmp, bb.n_items, s);
  }
  if (bb.qfine)
    launch_query_order(L);  // with the work items and tile boxes
  else
    launch_tile_setup(L);

  // (b), (c)
  mark(kStageDensity);
  launch_neighbour(L, true);
  mark(kStageNearestHigher);
  launch_neighbour(L, false);

  // (d), (e)
  mark(kStageSeeds);
  if (bb.event_order && bb.lone.is) {
    hipLaunchKernelGGL(k_lone_seeds<T>, dim3(1), dim3(kEvtBlock), 0, s, rp, bb.lone.ev,
                       bb.sorted.perm, bb.iperm, bb.srho, bb.snh, bb.sdelta, bb.sorted.u, out.rho,
                       out.nh, out.delta, out.is_seed, bb.n_seeds, bb.seeds, out.event_of_cluster,
                       out.cluster);
    mark(kStageLabels);
  } else if (bb.event_order) {
    hipLaunchKernelGGL(k_event_seeds<T>, dim3(static_cast<unsigned>(bb.n_events)), dim3(kEvtBlock),
                       0, s, rp, bb.events, bb.event_order, bb.sorted.perm, bb.iperm, bb.srho, bb.snh,
                       bb.sdelta, bb.sorted.u, out.rho, out.nh, out.delta, out.is_seed, bb.rank,
                       bb.event_seeds, out.cluster);
    mark(kStageLabels);
    scan_exclusive(bb.event_seeds, bb.event_offsets, bb.n_events, bb.scan_tmp, bb.n_seeds, s);
    hipLaunchKernelGGL(k_event_labels, dim3(bb.n_chunks), dim3(kBlock), 0, s, bb.chunks, bb.events,
                       bb.sorted.perm, bb.snh, bb.rank, bb.event_offsets, bb.event_seeds,
                       out.cluster, bb.seeds, out.event_of_cluster, out.local_ids);
  } else {
    const int words = (n + 31) / 32;
    uint32_t* bits = reinterpret_cast<uint32_t*>(bb.flag);
    hipLaunchKernelGGL(k_results<T>, dim3((n + kBlock - 1) / kBlock), dim3(kBlock), 0, s, rp, n,
                       bb.sorted.perm, bb.srho, bb.snh, bb.sdelta, bb.sorted.u, out.rho, out.nh,
                       out.delta, out.is_seed, bits);
    if (words <= kRankWords) {
      hipLaunchKernelGGL(k_seed_ranks, dim3(1), dim3(kRankBlock), 0, s, bits, words, bb.rank,
                         bb.n_seeds);
    } else {
      hipLaunchKernelGGL(k_seed_counts, dim3((words + kBlock - 1) / kBlock), dim3(kBlock), 0, s,
                         bits, words, bb.rank);
      scan_exclusive(bb.rank, bb.rank, words, bb.scan_tmp, bb.n_seeds, s);
    }
    mark(kStageLabels);
    static_assert(kPointChunk == kBlock << 3, "eight rounds of a full chunk");
    const int parts_log2 = bb.sort_by_chunk ? 3 : 0;
    hipLaunchKernelGGL(k_labels, dim3(static_cast<unsigned>(bb.n_chunks) << parts_log2), dim3(kBlock),
                       0, s, bb.chunks, bb.events, bb.sorted.perm, bb.snh, bits, bb.rank, out.cluster,
                       bb.seeds, out.event_of_cluster, out.local_ids, parts_log2);
  }
  mark(kNumStages);
}

}  // namespace clue_dev
