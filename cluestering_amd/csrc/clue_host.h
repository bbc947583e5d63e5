// Host-only sizing shared by the C ABI, the server and the CPU tests: the batch
// descriptor built from the event sizes, the launch tuning it selects, and the
// device bytes each workspace buffer needs. No HIP types here, so the same code
// builds with g++ under the address and undefined-behaviour sanitizers.
#pragma once

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <string>
#include <vector>

#include "clue_amd.h"
#include "clue_tuning_table.h"
#include "clue_types.h"

namespace clue_rt {

using clue_dev::Chunk;
using clue_dev::EventDesc;
using clue_dev::Item;
using clue_dev::radix_hist_elems;
using clue_dev::scan_temp_elems;

constexpr int kChunk = clue_dev::kPointChunk;
constexpr int kEvtSoloMaxPoints = clue_dev::kLoneMaxPoints;
constexpr int kDefaultPointsPerTile = 128;
// Launches up to this many points have their neighbour stages run by teams of waves
// (clue_team.h). Lone events on MI355X, one wave per item against a team of eight,
// whole calls: 16,000 points 258 -> 179 us (2-D) and 476 -> 301 us (3-D), 100,000
// points 662 -> 551 and 521 -> 449 us, 131,072 points 803 -> 678 and 533 -> 631 us.
// Batches of small events have short walks and fill the chip sooner: 36,558 points in
// 16 events 243 -> 192 us, 70,850 in 128 events 171 -> 185 us.
constexpr int kTeamMaxPoints = 110000;
constexpr int kTeamMaxPointsSmall = 49152;  // events of fewer than kTeamSmallEvent points
constexpr int kTeamSmallEvent = 4096;
// A team costs 5-13 ns of the chip whatever its item holds (512 threads to start, eight
// waves' worth of set-up), which only a long walk pays back: the item slots must hold
// kTeamItemPoints points on average. (Tiles of few points, by points_per_tile or by many
// dimensions: 100,000 points at 4 per tile 798 us in 2-D and 944 in 3-D by teams, 472 and
// 510 by waves; 50,000 in 8-D, 7 per slot, 758 and 582; 100,000 in 6-D, 18 per slot, 609
// and 718; 3,000 events of 16 285 and 212.) A lone event of few points and as few items
// still has CUs to spare: up to kTeamItemWork points times slots (8,000 points at one
// per tile 165 us by teams and 281 by waves, 16,384 at one 293 and 368, 50,000 at 16
// 348 and 353; 20,000 in 6-D at four, 3.2e8, 411 and 303).
constexpr int kTeamItemPoints = 16;
constexpr int64_t kTeamItemWork = 300000000;

// Constants of exp(y * 2^-s) (clue_dev::ExpScaled): each constant of the float
// exp scaled by a power of two, exact for |s| <= 8.
inline clue_dev::ExpScaled exp_scaled(int s) {
  clue_dev::ExpScaled e{};
  e.log2e = std::ldexp(clue_dev::kExpLog2e, -s);
  e.ln2_hi = std::ldexp(clue_dev::kExpLn2Hi, s);
  e.ln2_lo = std::ldexp(clue_dev::kExpLn2Lo, s);
  for (int i = 0; i < 5; ++i) e.c[i] = std::ldexp(clue_dev::kExpPoly[i], -s * (6 - i));
  e.c[5] = std::ldexp(1.0f, -s);
  e.lo = std::ldexp(clue_dev::kExpCoreLo, s);
  e.hi = std::ldexp(clue_dev::kExpCoreHi, s);
  return e;
}

// max_items: the launch's item slots.
inline bool team_launch(int64_t points, int64_t events, int64_t max_items) {
  const bool small = events > 1 && points / events < kTeamSmallEvent;
  if (points > (small ? kTeamMaxPointsSmall : kTeamMaxPoints)) return false;
  return points >= kTeamItemPoints * max_items || (events == 1 && points * max_items <= kTeamItemWork);
}

// Capacity a grow-only device buffer holds after a request of `bytes`: unchanged
// when it already fits, else the request plus a quarter and 256 bytes.
inline size_t grown_capacity(size_t cap, size_t bytes) {
  return bytes <= cap ? cap : bytes + bytes / 4 + 256;
}

// Workspace slots of one batch run.
enum Slot {
  S_EVENTS, S_CHUNKS, S_EXT, S_GEO, S_K0, S_V0, S_K1, S_V1, S_HIST, S_SCAN, S_TOFF, S_ICOUNT,
  S_NITEMS, S_ITEMS, S_SRHO, S_SKEY, S_SNH, S_SDELTA, S_FLAG, S_RANK, S_NSEEDS, S_SEEDS, S_SX,
  S_SW, S_SSIG, S_SU, S_STAG, S_SFW, S_PERM, S_RHO, S_NH, S_ISSEED, S_DELTA, S_HIN, S_HCL,
  S_QPERM, S_QPERM_NH, S_QFINE, S_HX, S_HKEY, S_HIDX, S_HBOX, S_HBKEY, S_EORDER, S_ESEEDS, S_EOFF, S_IPERM, S_SBOX, S_NUM
};

// Bits of the tile keys of a batch.
inline int tile_key_bits(int64_t tiles) {
  int bits = 0;
  while ((int64_t(1) << bits) < tiles) ++bits;
  return bits;
}

// Blocks of the tile sort: the events' chunks, whose first digits the key stage counts
// on the way; or, where small events make more than twice as many of them as the
// points fill, 2,048 consecutive points whatever their events (the keys are the
// batch's). A table of digit counts per chunk would then outgrow the points, and so
// would the workgroups. One event of 140,000 points in 2-D beside 100,000 of 10: 5,127 us
// and 414 MB of counts by chunks, 1,773 us and 1.1 MB by points; beside 20,000 of 256
// 2,981 and 2,235 us, 4,000 of 256 1,114 and 1,021, 2,000 of 600 1,092 and 1,063; beside
// 1,200 of 1,024, still by chunks, 1,295.
inline bool sort_by_chunk(int64_t points, int64_t chunks) {
  return chunks <= 2 * ((points + clue_dev::kRsTileKeys - 1) / clue_dev::kRsTileKeys);
}
inline int64_t sort_hist_elems(int64_t points, int64_t chunks, int64_t tiles) {
  const int64_t blocks =
      sort_by_chunk(points, chunks) ? chunks
                                    : (points + clue_dev::kRsTileKeys - 1) / clue_dev::kRsTileKeys;
  return radix_hist_elems(blocks, clue_dev::radix_plan(tile_key_bits(tiles)).bits);
}

// Host-side description of one batch (all derived from the event sizes).
struct BatchPlan {
  std::vector<EventDesc> events;
  std::vector<int32_t> event_order;  // fused per-event tile build: events largest first; empty: radix path
  std::vector<Chunk> chunks;
  int64_t n_total = 0;
  int64_t n_tiles_total = 0;
  int64_t max_items = 0;
  int key_bits = 0;
  bool team = false;  // neighbour stages by teams of waves
  int ext_group = 1;  // chunks per result of the extremes stage
  clue_tuning tuning{};
};

// Tiles per dimension of an event of n points (SetupTiles.hpp:30-34):
// ntiles = ceil(n / ppt), nper = min{k : k^D >= ntiles}; tiles = nper^D.
inline void event_tiles(int64_t n, int D, int ppt, int64_t* nper_out, int64_t* tiles_out) {
  const int64_t nt0 = (n + ppt - 1) / ppt;
  auto pw = [D](int64_t b) {
    int64_t r = 1;
    for (int k = 0; k < D; ++k) r *= b;
    return r;
  };
  int64_t nper = 1;
  while (pw(nper) < nt0) ++nper;
  *nper_out = nper;
  *tiles_out = pw(nper);
}

// Tuning of a batch: the built-in table's entry for its ndim and mean event size.
inline clue_tuning table_tuning(int ndim, int64_t n_total, int64_t n_events) {
  const int64_t mean = n_events > 0 ? n_total / n_events : n_total;
  clue_tuning out{};
  for (const TuningEntry& t : kTuningTable)
    if ((t.ndim == 0 || t.ndim == ndim) && mean <= t.max_mean_event) {
      out.group_queries = t.group_queries;
      out.xcd_chunk_log2 = t.xcd_chunk_log2;
      out.block_waves = t.block_waves;
      out.persistent = t.persistent;
      return out;
    }
  out.group_queries = 1;
  out.xcd_chunk_log2 = 4;
  out.block_waves = 4;
  return out;
}

// The tuning of a run that none is fixed for: the table's, or teams of waves.
inline clue_tuning chosen_tuning(int ndim, int64_t points, int64_t events, int64_t max_items) {
  clue_tuning t = table_tuning(ndim, points, events);
  t.team = team_launch(points, events, max_items) ? 1 : 0;
  if (t.team) t.group_queries = 1;  // small boxes around each team's points
  return t;
}

// Builds the batch descriptor: one EventDesc per non-empty event, its chunks,
// tile bases, work-item bound and radix key width. `fixed` (may be NULL) replaces
// the table's tuning. Returns CLUE_OK, or CLUE_ERR_CAPACITY with *err set when the
// batch exceeds 32-bit indexing.
inline clue_status plan_batch(int D, int points_per_tile, const uint32_t* sizes, int32_t n_events,
                              const clue_tuning* fixed, BatchPlan* bp, std::string* err) {
  const int ppt = points_per_tile > 0 ? points_per_tile : kDefaultPointsPerTile;
  bp->events.clear();
  bp->chunks.clear();
  int64_t off = 0, tiles = 0;
  for (int32_t e = 0; e < n_events; ++e) {
    const int64_t n = sizes[e];
    if (n == 0) continue;
    int64_t nper = 0, nt = 0;
    event_tiles(n, D, ppt, &nper, &nt);
    EventDesc ev{};
    ev.p_off = static_cast<int32_t>(off);
    ev.n = static_cast<int32_t>(n);
    ev.nper = static_cast<int32_t>(nper);
    ev.ntiles = static_cast<int32_t>(nt);
    ev.t_base = static_cast<int32_t>(tiles);
    ev.index = e;
    const int32_t eidx = static_cast<int32_t>(bp->events.size());
    bp->events.push_back(ev);
    for (int64_t b = 0; b < n; b += kChunk) {
      Chunk c{};
      c.event = eidx;
      c.begin = static_cast<int32_t>(off + b);
      c.end = static_cast<int32_t>(off + std::min<int64_t>(n, b + kChunk));
      bp->chunks.push_back(c);
    }
    off += n;
    tiles += nt;
    if (off > INT32_MAX / 2 || tiles > INT32_MAX / 2) {
      *err = "batch too large for 32-bit indexing";
      return CLUE_ERR_CAPACITY;
    }
  }
  bp->n_total = off;
  bp->n_tiles_total = tiles;
  // The fused per-event stages when every event's tiles and points fit their LDS,
  // except for one event alone above kEvtSoloMaxPoints: there the many-workgroup
  // stages win over one workgroup's serial passes (per-event calls on MI355X over
  // 512 events of 256-65,536 points: 3.3k -> 3.75k events/s, p99 1.19 -> 1.00 ms,
  // median 0.18 ms either way; a 16k-point event 0.31 -> 0.29 ms).
  bool local = !bp->events.empty() &&
               (bp->events.size() >= 2 || bp->events[0].n <= kEvtSoloMaxPoints);
  for (const EventDesc& ev : bp->events)
    local = local && ev.ntiles <= clue_dev::kEvtMaxTiles && ev.n <= clue_dev::kEvtMaxPoints;
  bp->event_order.clear();
  if (local) {
    for (int32_t k = 0; k < static_cast<int32_t>(bp->events.size()); ++k) bp->event_order.push_back(k);
    if (bp->event_order.size() > 1)
      std::stable_sort(bp->event_order.begin(), bp->event_order.end(),
                       [&](int32_t a, int32_t b) { return bp->events[a].n > bp->events[b].n; });
  }
  // At most 512 results per event: every workgroup of the key stage reads them all.
  int64_t largest = 0;
  for (const EventDesc& ev : bp->events) largest = std::max<int64_t>(largest, ev.n);
  bp->ext_group = static_cast<int>(std::max<int64_t>(1, (largest + 512 * kChunk - 1) / (512 * kChunk)));
  bp->max_items = (off + 63) / 64 + tiles;
  const int64_t n_described = static_cast<int64_t>(bp->events.size());
  bp->tuning = fixed ? *fixed : chosen_tuning(D, off, n_described, bp->max_items);
  // A fixed tuning allows teams; the launch must still be small enough for them.
  bp->team = bp->tuning.team && team_launch(off, n_described, bp->max_items);
  if (bp->team) bp->tuning.group_queries = 1;
  bp->key_bits = tile_key_bits(tiles);
  return CLUE_OK;
}

// What the workspace of one batch depends on.
struct WorkspaceShape {
  int D = 1;
  int value_bytes = 4;      // sizeof the point type
  int key_bytes = 4;        // sizeof the ordered-integer extremes (the point type's width)
  int64_t n = 0;            // points
  int64_t events = 0;       // non-empty events
  int64_t chunks = 0;
  int64_t tiles = 0;        // sum of nper^D
  int64_t max_items = 0;
  bool team = false;               // neighbour stages by teams of waves
  bool event_tiles = false;        // the fused per-event tile build (no radix-sort buffers)
  bool group_queries = false;
  bool separate_dm_order = false;  // a second query order for dm (no run asks for one)
  bool nh_blocks = false;          // nearest-higher over the Hilbert block layout
  bool flat_kernel = false;
  bool has_sigma = false;
  bool has_u = false;
  bool own_rho = false;            // results the caller does not provide live in the workspace
  bool own_nh = false;
  bool own_is_seed = false;
  bool sorted_boxes = false;       // density leaves out tiles by their bounding boxes
  bool density_morton = false;     // density takes the Hilbert order of qfine (every grouped run)
};

// Bytes of the tiles' bounding boxes, 0 where the stages do without. Small tables are
// always worth it; of the large ones those that hold fewer than 16 points per tile are
// left out: in many dimensions, or with very small tiles, they would take more memory
// than the columns of the points.
constexpr int64_t kTileBoxAlways = 4 << 20;
inline size_t tile_box_bytes(int64_t n, int64_t tiles, int D, int value_bytes) {
  const int64_t bytes = tiles * 2 * D * value_bytes;
  return bytes <= kTileBoxAlways || 16 * tiles <= n ? static_cast<size_t>(bytes) : 0;
}

// Bytes of every workspace slot for a batch of this shape (0: unused).
inline void workspace_requests(const WorkspaceShape& w, size_t (&bytes)[S_NUM]) {
  std::memset(bytes, 0, sizeof(bytes));
  const int64_t n = w.n, NT = w.tiles;
  const int64_t hist = sort_hist_elems(n, w.chunks, NT);
  const int64_t scan_elems =
      std::max({scan_temp_elems(n), scan_temp_elems(w.events), scan_temp_elems(NT)}) + 16;
  const int64_t stride = (n + 63) / 64 * 64;
  const int64_t h_blocks = w.nh_blocks ? (n + clue_dev::kNhBlock - 1) / clue_dev::kNhBlock + NT + 1 : 0;
  const int64_t h_slots = h_blocks * clue_dev::kNhBlock;
  const size_t T = static_cast<size_t>(w.value_bytes);
  const size_t D = static_cast<size_t>(w.D);
  bytes[S_EVENTS] = sizeof(EventDesc) * w.events;
  bytes[S_CHUNKS] = sizeof(Chunk) * w.chunks;
  bytes[S_EXT] = w.event_tiles ? 0 : static_cast<size_t>(w.key_bytes) * w.chunks * D * 2;
  bytes[S_GEO] = T * w.events * 3 * D;
  bytes[S_K0] = bytes[S_K1] = w.event_tiles ? 0 : sizeof(uint32_t) * n;
  bytes[S_V0] = bytes[S_V1] = w.event_tiles ? 0 : sizeof(int32_t) * n;
  bytes[S_HIST] = w.event_tiles ? 0 : sizeof(int32_t) * hist;
  bytes[S_EORDER] = w.event_tiles ? sizeof(int32_t) * w.events : 0;
  bytes[S_ESEEDS] = bytes[S_EOFF] = w.event_tiles ? sizeof(int32_t) * w.events : 0;
  bytes[S_IPERM] = w.event_tiles ? sizeof(int32_t) * n : 0;
  bytes[S_SCAN] = sizeof(int32_t) * scan_elems;
  bytes[S_TOFF] = sizeof(int32_t) * (NT + 1);
  bytes[S_ICOUNT] = w.team ? 0 : sizeof(int32_t) * NT;
  bytes[S_NITEMS] = sizeof(int32_t) * 32;  // item count, then the work-item queue counters
  bytes[S_ITEMS] = sizeof(Item) * w.max_items;
  bytes[S_QPERM] = (w.group_queries && !w.density_morton) ? sizeof(int32_t) * n : 0;
  bytes[S_QPERM_NH] = (w.group_queries && w.separate_dm_order) ? sizeof(int32_t) * n : 0;
  bytes[S_QFINE] = w.group_queries ? sizeof(int32_t) * n : 0;
  bytes[S_HX] = T * h_slots * D;
  bytes[S_HKEY] = sizeof(uint64_t) * h_slots;
  bytes[S_HIDX] = sizeof(int32_t) * h_slots;
  bytes[S_HBOX] = T * h_blocks * 2 * D;
  bytes[S_HBKEY] = sizeof(uint64_t) * h_blocks;
  bytes[S_SBOX] = w.sorted_boxes ? tile_box_bytes(n, NT, w.D, w.value_bytes) : 0;
  bytes[S_SRHO] = T * n;
  bytes[S_SKEY] = w.nh_blocks ? 0 : sizeof(uint64_t) * n;  // the block scan's keys: S_HKEY
  bytes[S_SFW] = w.flat_kernel ? T * n : 0;
  bytes[S_SNH] = sizeof(int32_t) * n;
  bytes[S_SDELTA] = T * n;
  bytes[S_FLAG] = w.event_tiles ? 0 : sizeof(uint32_t) * ((n + 31) / 32);
  bytes[S_RANK] = sizeof(int32_t) * n;
  bytes[S_NSEEDS] = sizeof(int32_t) * 4;
  bytes[S_SEEDS] = sizeof(int32_t) * n;
  bytes[S_SX] = T * stride * D;
  bytes[S_SW] = T * n;
  bytes[S_SSIG] = w.has_sigma ? T * stride * D : 0;
  bytes[S_SU] = w.has_u ? T * n : 0;
  bytes[S_STAG] = sizeof(uint32_t) * n;
  bytes[S_PERM] = sizeof(int32_t) * n;
  bytes[S_RHO] = w.own_rho ? T * n : 0;
  bytes[S_NH] = w.own_nh ? sizeof(int32_t) * n : 0;
  bytes[S_ISSEED] = w.own_is_seed ? sizeof(int32_t) * n : 0;
}

}  // namespace clue_rt
