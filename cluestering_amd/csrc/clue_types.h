// Plain structs shared by the host orchestration and the device stages.
#pragma once

#include <stdint.h>

namespace clue_dev {

constexpr int kMaxDim = 10;
// Candidates per block of the nearest-higher block layout (one bounding box and
// one largest key per block).
constexpr int kNhBlock = 16;

// Metric id of a periodic Euclidean metric whose only non-zero period is the last
// dimension's (a detector's phi): chosen by the host for the device stages alone.
constexpr int kMetricPeriodicLast = 7;

// Largest tile count of an event that the fused per-event tile build takes (its
// per-wave tile counters live in LDS); batches with a larger event take the
// radix-sort path.
constexpr int kEvtMaxTiles = 1024;
// Largest event the fused per-event stages take (one bit per point in LDS).
constexpr int kEvtMaxPoints = 1 << 17;
// Largest lone event of the fused stages.
constexpr int kLoneMaxPoints = 8192;

constexpr int kPointChunk = 2048;  // points per chunk of the per-point grids

// Workspace sizes of the scan and radix-sort primitives (clue_primitives.hip),
// here so that host-only code sizes workspaces exactly as the device path does.
constexpr int kScanTileElems = 4096;  // elements per block of the exclusive scan
constexpr int kRsTileKeys = 2048;     // keys per block of a radix pass
constexpr int kRsMaxBits = 10;        // of a radix digit
constexpr int kRsMaxBins = 1 << kRsMaxBits;
static_assert(kPointChunk == kRsTileKeys, "a chunk is a block of the radix sort");
inline int64_t scan_temp_elems(int64_t n) { return (n + kScanTileElems - 1) / kScanTileElems + 1; }
// Digits of a radix sort by key_bits bits: as few passes as kRsMaxBits allows, of equal
// widths.
struct RadixPlan {
  int bits;  // of a digit
  int passes;
};
inline RadixPlan radix_plan(int key_bits) {
  RadixPlan p;
  p.passes = key_bits <= 0 ? 1 : (key_bits + kRsMaxBits - 1) / kRsMaxBits;
  p.bits = key_bits <= 0 ? 1 : (key_bits + p.passes - 1) / p.passes;
  return p;
}
// Digit counts per block, then the digits' totals.
inline int64_t radix_hist_elems(int64_t blocks, int digit_bits) {
  return (blocks + 1) << digit_bits;
}

// The union of a wave's search boxes, in tiles: from lo on, ext of them per dimension. On
// wrapped dimensions it can span almost twice the tiles there are, 2^D times as many
// together. A launch has fewer than 2^26 tiles (2^32 threads at one wave each), so
// from six dimensions on that can be more than 32 bits count. Such a union is visited in
// runs, one per step of dimension 0 (in ten dimensions of 0 and 1), in the reference's
// order; any other is one run. (constexpr: host and device. Up to five dimensions there
// is nothing to keep between runs: the density stage has no scalar registers to spare
// there, 2^20 points in 2-D took 690 us without and 704 with them.)
constexpr int64_t kTileRunMax = INT32_MAX - 64;  // a wave counts a run's tiles by 64
template <int D>
struct BoxUnion {
  static constexpr int kOuter = D < 6 ? 0 : D < 10 ? 1 : 2;
  int lo[D], ext[D];
  int tiles;                          // of a run; 0: no active lane
  int last[kOuter > 0 ? kOuter : 1];  // lo of the outer dimensions in the last run
  int first1;                         // lo[1] in the first run (two outer dimensions)
};
// tiles and the first run of the union given by lo and ext.
template <int D>
constexpr void first_tile_run(BoxUnion<D>& u, int64_t most = kTileRunMax) {
  constexpr int K = BoxUnion<D>::kOuter;
  if constexpr (K == 0) {
    u.tiles = 1;
    for (int d = 0; d < D; ++d) u.tiles *= u.ext[d];
  } else {
    int64_t inner = 1;
    for (int d = D - 1; d >= K; --d) inner *= u.ext[d];
    int64_t all = inner;
    for (int d = 0; d < K; ++d) {
      all *= u.ext[d];
      u.last[d] = u.lo[d];
    }
    u.first1 = u.lo[K - 1];
    if (all > most) {
      for (int d = 0; d < K; ++d) {
        u.last[d] += u.ext[d] - 1;
        u.ext[d] = 1;
      }
      all = inner;
    }
    u.tiles = static_cast<int>(all);
  }
}
// Goes on to the next run; false after the last.
template <int D>
constexpr bool next_tile_run(BoxUnion<D>& u) {
  constexpr int K = BoxUnion<D>::kOuter;
  if constexpr (K == 0) {
    return false;
  } else {
    if (K == 2 && u.lo[K - 1] != u.last[K - 1]) {
      ++u.lo[K - 1];
      return true;
    }
    if (u.lo[0] == u.last[0]) return false;
    ++u.lo[0];
    if (K == 2) u.lo[K - 1] = u.first1;
    return true;
  }
}

// Constants of the float exp (Cody-Waite reduction x = k ln2 + r with a 15-bit
// ln2_hi, then the degree-6 minimax polynomial of e^r on [-ln2/2, ln2/2] whose
// constant and linear terms are 1), shared by the device code and the host code
// that folds power-of-two argument scales into them.
constexpr float kExpLog2e = 0x1.715476p+0f;
constexpr float kExpLn2Hi = 0x1.62e400p-1f;
constexpr float kExpLn2Lo = 0x1.7f7d1cp-20f;
constexpr float kExpPoly[5] = {0x1.6a244cp-10f, 0x1.1239d4p-7f, 0x1.5558f2p-5f, 0x1.555492p-3f,
                               0x1.fffffcp-2f};  // c6, c5, c4, c3, c2
constexpr float kExpCoreLo = -0x1.9fe368p+6f;  // the core needs no range handling on [lo, hi]
constexpr float kExpCoreHi = 0x1.62e42ep+6f;

// exp(y * 2^-s) evaluated without forming y * 2^-s: every step of the reduction
// and of the Horner polynomial is the float exp's own step scaled by a power of
// two (k = rint(y * (log2e 2^-s)); r' = 2^s r from ln2 2^s; the Horner partial
// sums carry 2^(-s i) through coefficients c_i 2^(-s i)), so with |s| <= 8 no
// step leaves the normal range and the bits equal exp(rn(y * 2^-s)) for every y.
struct ExpScaled {
  float log2e;   // log2e * 2^-s
  float ln2_hi;  // ln2_hi * 2^s
  float ln2_lo;  // ln2_lo * 2^s
  float c[6];    // c6 .. c1, c_i * 2^(-s i)
  float lo, hi;  // the core range, times 2^s
};

// One event of a batch. All offsets are host-computed from the event sizes.
struct EventDesc {
  int32_t p_off;   // first point of the event in the packed arrays
  int32_t n;       // points in the event
  int32_t nper;    // tiles per dimension (SetupTiles.hpp:30-34)
  int32_t ntiles;  // nper^D
  int32_t t_base;  // first global tile key of the event
  int32_t index;   // the caller's event index (empty events are not described)
  int32_t pad[2];
};

// A contiguous range of points of one event, the unit of the per-point grids.
struct Chunk {
  int32_t event;
  int32_t begin;  // global point index
  int32_t end;
  int32_t pad;
};

// The descriptor of a run's only event, as a kernel argument: the pipeline's first
// kernel writes the descriptors in memory from it (a launch, or two copies, fewer per
// call). A kernel before the pipeline takes its chunks from here too (lone_chunk).
struct LoneEvent {
  int32_t is;  // the run has one event, at offset 0
  EventDesc ev;
};

// A work item of the neighbour stages: up to 64 consecutive tile-sorted points of
// one tile (one lane each).
struct Item {
  int32_t tile;   // global tile key
  int32_t begin;  // sorted position of the first point
  int32_t end;
  int32_t event;
};

// Per-run scalar parameters as the device stages consume them; T is the point
// type (float, or double for Clusterer<Ndim, double>).
template <class T>
struct RunParamsT {
  int32_t D;
  int32_t kernel;
  int32_t metric;
  int32_t has_sigma;
  int32_t has_u;
  int32_t has_tags;
  int32_t n_events;
  int32_t n_total;
  int32_t max_items;       // work-item slots
  T dc;
  T rhoc;
  T dm;
  T seed_dc;
  T dc_sq_max;           // largest t with sqrt_rn(t) <= dc (sqrt metrics)
  T dm_sq_max;           // same for dm
  T seed_sq_max;         // same for seed_dc
  T in_scale;            // 2^k and 2^k times the value after the density radius' threshold, for
  T in_limit;            // the flat kernel's sums (0: selects instead)
  T kp0, kp1;            // kernel parameters (flat f | exp lambda, A | gauss sigma, A)
  T gauss_den;           // (2 * sigma) * sigma, as the reference evaluates it
  T gauss_inv_den;       // 1 / gauss_den when gauss_den is a power of two
  int32_t gauss_pow2;    // gauss_den is a power of two
  int32_t gauss_fold;    // float runs: gauss_den = 2^s with |s| <= 8, folded into es
  int32_t exp_in_range;  // every kernel exp argument within the radius is in the core range
  ExpScaled es;          // float runs: exp(y * 2^-s) with 2^s = gauss_den
  int32_t wrapped[kMaxDim];
  T mparam[kMaxDim];
  int32_t xcd_chunk_log2;  // neighbour stages: 2^k consecutive blocks per XCD turn; < 0: none
  int32_t block_waves;     // neighbour stages: waves per workgroup (1, 2, 4, 8 or 16)
  int32_t nh_blocks;       // nearest-higher over the Hilbert-ordered block layout
  int32_t cull;            // density: candidates bounded by the metric's lower bound (no weight below 0)
  int32_t team;            // neighbour stages: a team of waves per item (clue_team.h)
  int32_t persistent;      // neighbour stages: persistent waves per CU pulling items (0: none)
};
using RunParams = RunParamsT<float>;

}  // namespace clue_dev
