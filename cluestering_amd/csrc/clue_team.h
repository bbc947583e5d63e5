// Density and nearest-higher by teams: a workgroup of kTeam waves works on one item
// (up to 64 points of one tile, one lane each, in every wave), for launches with too
// few items to fill the chip. One wave per item is a serial walk over its candidates
// there (a wave alone issues one vector instruction per 6-8 cycles, and waits for
// every load), and the launch lasts as long as its longest walk.
//
// The waves first look at the candidates of the reachable tiles, 64 at a time per
// wave, and list those that any of the item's queries can reach in LDS, in the
// reference's order. Then they share the list. A density's terms must be added in
// that order, but can be computed in any: wave w computes the terms of chunks w,
// w + kTeam, ... into registers, waits until the sums of the chunks before have been
// handed over through LDS, adds its terms and hands the sums on. The nearest-higher
// candidate is the extreme of a strict order: the waves search their shares alone
// and compare their results at the end.
//
// Included by clue_stages_impl.h.
#pragma once

namespace clue_dev {

// Waves per workgroup: 16 fill the chip too early (16,384 points in 2-D: density 25
// against 19 us), 4 leave small events waiting (1,000 points, whole call 94 against 85 us).
constexpr int kTeam = 8;
constexpr int kTeamBlock = 8;   // listed candidates evaluated together
// Blocks whose terms are added in one turn (four: 20.1 against 19.4 us).
constexpr int kChunkBlocks = 2;

// ---------------------------------------------------------------------------
// The sums on their way from wave to wave: per lane the value and the number of
// the chunk that may add to it next, in one 64-bit word (two for double), so that
// one LDS access hands over both.
// ---------------------------------------------------------------------------
template <class T>
struct SumRelay {
  uint64_t word[sizeof(T) / 4][kWave];
};

__device__ __forceinline__ void relay_store(uint64_t* p, uint32_t v, int turn) {
  __hip_atomic_store(p, (static_cast<uint64_t>(static_cast<uint32_t>(turn)) << 32) | v,
                     __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ uint64_t relay_load(uint64_t* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void relay_pass(SumRelay<float>& r, float sum, int turn) {
  relay_store(&r.word[0][lane_id()], __float_as_uint(sum), turn);
}
__device__ __forceinline__ void relay_pass(SumRelay<double>& r, double sum, int turn) {
  const uint64_t b = static_cast<uint64_t>(__double_as_longlong(sum));
  relay_store(&r.word[0][lane_id()], static_cast<uint32_t>(b), turn);
  relay_store(&r.word[1][lane_id()], static_cast<uint32_t>(b >> 32), turn);
}
// Waits for the turn. Chunks are taken in increasing order by every wave, so the
// wave that holds the lowest unfinished chunk never waits, and every wait ends.
__device__ __forceinline__ float relay_take(SumRelay<float>& r, int turn) {
  uint64_t a = relay_load(&r.word[0][lane_id()]);
  while (ballot(static_cast<int>(a >> 32) != turn) != 0ull) {
    __builtin_amdgcn_s_sleep(1);
    a = relay_load(&r.word[0][lane_id()]);
  }
  return __uint_as_float(static_cast<uint32_t>(a));
}
__device__ __forceinline__ double relay_take(SumRelay<double>& r, int turn) {
  uint64_t a, b;
  while (true) {
    a = relay_load(&r.word[0][lane_id()]);
    b = relay_load(&r.word[1][lane_id()]);
    if (ballot(static_cast<int>(a >> 32) != turn || static_cast<int>(b >> 32) != turn) == 0ull) break;
    __builtin_amdgcn_s_sleep(1);
  }
  return __longlong_as_double(
      static_cast<long long>((b << 32) | static_cast<uint64_t>(static_cast<uint32_t>(a))));
}

// ---------------------------------------------------------------------------
// A lane's query point.
// ---------------------------------------------------------------------------
template <int D, class T>
struct TeamQuery {
  bool active;
  int pos;  // sorted position; -1: no point in this lane
  T x[D], s[D];

  __device__ __forceinline__ void load(const Item& it, const int32_t* __restrict__ qperm,
                                       const T* __restrict__ sx, int64_t cs,
                                       const T* __restrict__ ssig, const RunParamsT<T>& rp) {
    const int q = it.begin + lane_id();
    active = q < it.end;
    pos = active ? (qperm ? qperm[q] : q) : -1;
#pragma unroll
    for (int d = 0; d < D; ++d) {
      x[d] = active ? sx[d * cs + pos] : T(0);
      s[d] = (active && rp.has_sigma) ? ssig[d * cs + pos] : T(0);
    }
  }
  __device__ __forceinline__ void box(const GeoT<T>& g, T R, int (&lo)[D], int (&hi)[D]) const {
    search_box<D>(g, x, s, R, lo, hi);
    if (!active) {
#pragma unroll
      for (int d = 0; d < D; ++d) {
        lo[d] = INT32_MAX;
        hi[d] = INT32_MIN;
      }
    }
  }
};

// With the best candidate found so far (k_nh_blocks: the same test and bound).
template <int D, int M, class T>
struct HigherQuery : TeamQuery<D, T> {
  uint64_t key;
  uint32_t tag, tag_nh;
  T eff_thr, bound, delta, rho_nh;
  int nh;

  __device__ __forceinline__ void load(const Item& it, const int32_t* __restrict__ qperm,
                                       const T* __restrict__ sx, int64_t cs,
                                       const T* __restrict__ ssig, const T* __restrict__ su,
                                       const uint32_t* __restrict__ stag,
                                       const T* __restrict__ srho, const RunParamsT<T>& rp) {
    TeamQuery<D, T>::load(it, qperm, sx, cs, ssig, rp);
    const T rho = this->active ? srho[this->pos] : T(0);
    tag = this->active ? stag[this->pos] : 0u;
    key = this->active ? query_key(rho, tag) : ~0ull;
    const T u = (this->active && rp.has_u) ? su[this->pos] : T(1);
    const bool use_seed = rho >= rp.rhoc * u;
    eff_thr = MetricTraits<M>::kSqrt ? (use_seed ? rp.seed_sq_max : rp.dm_sq_max)
                                     : (use_seed ? rp.seed_dc : rp.dm);
    delta = std::numeric_limits<T>::max();
    nh = -1;
    rho_nh = T(0);
    tag_nh = 0u;
    bound = eff_thr;
  }
  // earlier: decides between candidates that agree in all three.
  __device__ __forceinline__ bool beats(T dist, T r, uint32_t t, bool earlier) const {
    return (dist < delta) ||
           ((dist == delta) && (nh >= 0) &&
            ((r > rho_nh) || ((r == rho_nh) && ((t > tag_nh) || ((t == tag_nh) && earlier)))));
  }
  __device__ __forceinline__ void take(T dist, T r, uint32_t t, int j) {
    delta = dist;
    nh = j;
    rho_nh = r;
    tag_nh = t;
    bound = prune_threshold<M>(eff_thr, delta);
  }
  // A higher candidate with v <= bound.
  __device__ __forceinline__ bool consider(T v, T r, uint32_t t, int j) {
    const T dist = finish_distance<M>(v);
    if (!beats(dist, r, t, false)) return false;
    take(dist, r, t, j);
    return true;
  }
};

// ---------------------------------------------------------------------------
// The list of candidates in LDS. Payload: the weight (density) or the key
// (nearest-higher). kLooks: 64-candidate looks per wave between two barriers; the
// list is worked off once it holds a chunk for every wave, so it has room for one
// round more than that.
// ---------------------------------------------------------------------------
template <int D, int M, class T, class P>
struct TeamList {
  static constexpr int kSigmas = M == M_MAHALANOBIS ? D : 0;
  static constexpr int kEntry = (D + kSigmas) * sizeof(T) + sizeof(P) + 8;
  static constexpr int kLooks = kEntry <= 48 ? 2 : 1;
  static constexpr int kFull = kTeam * 32;
  static constexpr int kRoom = kFull + kTeam * kLooks * kWave;
  T x[D][kRoom];
  T s[kSigmas > 0 ? kSigmas : 1][kSigmas > 0 ? kRoom : 1];
  P payload[kRoom];
  int32_t j[kRoom];     // sorted position
  int32_t slot[kRoom];  // lane of its tile in the group
  int32_t count[kTeam];
};

// A group of tiles (one per lane) with its looks numbered in the reference's order.
template <int D>
struct TeamGroup : TileGroup<D> {
  uint64_t held;  // lanes whose tile is looked at
  int first;      // looks of the tiles before this lane's
  int looks;      // of the whole group
  uint64_t in;    // bit i: this lane's own box holds the tile of lane i

  __device__ __forceinline__ void number(bool hold) {
    held = ballot(hold);
    const int n = hold ? (this->j1 - this->j0 + kWave - 1) / kWave : 0;
    const int incl = wave_incl_scan(n);
    first = incl - n;
    looks = __builtin_amdgcn_readlane(incl, kWave - 1);
  }
  __device__ __forceinline__ void boxes(const int (&lo)[D], const int (&hi)[D]) {
    in = 0;
    for (uint64_t h = held; h; h &= h - 1ull) {
      const int i = __builtin_ctzll(h);
      in |= static_cast<uint64_t>(box_holds(*this, i, lo, hi) ? 1 : 0) << i;
    }
  }
};

// One round: every wave looks at kLooks times 64 candidates, look c0 on, and appends
// those that keep() wants to the list, in order. Returns the list's new length (the
// same in every wave; the list is readable on return).
template <int D, int M, class T, class P, class Keep>
__device__ __forceinline__ int list_round(const TeamGroup<D>& g, int c0, int n,
                                          const T* __restrict__ sx, int64_t cs,
                                          const T* __restrict__ ssig, const P* __restrict__ col,
                                          TeamList<D, M, T, P>& list, Keep keep) {
  constexpr int L = TeamList<D, M, T, P>::kLooks;
  const int wave = uniform(threadIdx.x / kWave);
  const int lane = lane_id();
  T x[L][D], s[L][D];
  P p[L];
  int j[L], slot[L];
  uint64_t want[L];
  int mine = 0;
#pragma unroll
  for (int a = 0; a < L; ++a) {
    const int c = c0 + wave * L + a;
    j[a] = -1;
    slot[a] = 0;
    if (c < g.looks) {
      const int i = 63 - __builtin_clzll(ballot(g.first <= c) & g.held);
      const int k = __builtin_amdgcn_readlane(g.j0, i) +
                    (c - __builtin_amdgcn_readlane(g.first, i)) * kWave + lane;
      slot[a] = i;
      if (k < __builtin_amdgcn_readlane(g.j1, i)) j[a] = k;
    }
    const bool real = j[a] >= 0;
#pragma unroll
    for (int d = 0; d < D; ++d) {
      x[a][d] = real ? sx[d * cs + j[a]] : T(0);
      s[a][d] = (M == M_MAHALANOBIS && real) ? ssig[d * cs + j[a]] : T(0);
    }
    p[a] = real ? col[j[a]] : P(0);
  }
#pragma unroll
  for (int a = 0; a < L; ++a) {
    want[a] = ballot(j[a] >= 0 && keep(x[a], s[a], p[a]));
    mine += __popcll(want[a]);
  }
  if (lane == 0) list.count[wave] = mine;
  __syncthreads();
  int at = n, total = n;
#pragma unroll
  for (int w = 0; w < kTeam; ++w) {
    const int c = list.count[w];
    at += w < wave ? c : 0;
    total += c;
  }
#pragma unroll
  for (int a = 0; a < L; ++a) {
    if ((want[a] >> lane) & 1ull) {
      const int e = at + __popcll(want[a] & lanemask_lt());
#pragma unroll
      for (int d = 0; d < D; ++d) {
        list.x[d][e] = x[a][d];
        if constexpr (M == M_MAHALANOBIS) list.s[d][e] = s[a][d];
      }
      list.payload[e] = p[a];
      list.j[e] = j[a];
      list.slot[e] = slot[a];
    }
    at += __popcll(want[a]);
  }
  __syncthreads();
  return uniform(total);
}

// Distances of the block of listed candidates at p; NaN, within no radius, past the
// list's n entries. Every lane reads the same words of LDS.
template <int D, int M, class T, class P>
__device__ __forceinline__ void block_distances(const TeamQuery<D, T>& me,
                                                const TeamList<D, M, T, P>& list, int p, int n,
                                                const RunParamsT<T>& rp, T (&v)[kTeamBlock]) {
#pragma unroll
  for (int c = 0; c < kTeamBlock; ++c) {
    T xj[D], sj[D];
#pragma unroll
    for (int d = 0; d < D; ++d) {
      xj[d] = list.x[d][p + c];
      sj[d] = T(0);
      if constexpr (M == M_MAHALANOBIS) sj[d] = list.s[d][p + c];
    }
    v[c] = metric_pair<D, M>(me.x, me.s, xj, sj, rp);
  }
  if (p + kTeamBlock > n) {
#pragma unroll
    for (int c = 0; c < kTeamBlock; ++c)
      v[c] = p + c < n ? v[c] : std::numeric_limits<T>::quiet_NaN();
  }
}

// exp of a block's arguments: the steps of expf_cw and expf_cw_scaled, with the
// constants of rp.es (those of s = 0 where no scale is folded), and of expd_cw.
__device__ __forceinline__ void block_exp(float (&y)[kTeamBlock], const RunParamsT<float>& rp) {
#pragma unroll
  for (int k = 0; k < kTeamBlock; ++k) {
    const float x = rp.exp_in_range ? y[k] : __builtin_fminf(__builtin_fmaxf(y[k], rp.es.lo), rp.es.hi);
    float e = expf_cw_core_scaled<false>(x, rp.es, rp.es.c[0]);
    if (!rp.exp_in_range) {
      e = (y[k] > rp.es.hi) ? __builtin_inff() : e;
      e = (y[k] < rp.es.lo) ? 0.0f : e;
      e = (y[k] != y[k]) ? y[k] : e;
    }
    y[k] = e;
  }
}
__device__ __forceinline__ void block_exp(double (&y)[kTeamBlock], const RunParamsT<double>& rp) {
  if (rp.exp_in_range) {
#pragma unroll
    for (int k = 0; k < kTeamBlock; ++k) y[k] = expd_cw_core(y[k]);
  } else {
#pragma unroll
    for (int k = 0; k < kTeamBlock; ++k) y[k] = expd_cw(y[k]);
  }
}

// The terms K(d) w of a block, 0 beyond the radius. The kernel is a runtime choice
// and its code is laid out once for all (a copy per kernel and loop mode measured the
// same, at ten times the code).
template <int M, class T>
__device__ __forceinline__ void block_terms(const T (&v)[kTeamBlock], const T (&w)[kTeamBlock],
                                            const T (&thr)[kTeamBlock], bool normal,
                                            const RunParamsT<T>& rp, T (&t)[kTeamBlock]) {
  if (rp.kernel == K_FLAT) {
#pragma unroll
    for (int k = 0; k < kTeamBlock; ++k) t[k] = v[k] <= thr[k] ? w[k] : T(0);
    return;
  }
  T y[kTeamBlock];
  if constexpr (MetricTraits<M>::kSqrt && sizeof(T) == 4) {
    bool odd = false;  // inputs the short square root does not take
#pragma unroll
    for (int k = 0; k < kTeamBlock; ++k) {
      y[k] = sqrt_rn_normal(v[k]);
      odd = odd || (v[k] <= thr[k] && v[k] != 0.0f && !(v[k] >= 0x1p-96f && v[k] <= 0x1.fffffep+127f));
    }
    if (!normal && ballot(odd) != 0ull) {
#pragma unroll
      for (int k = 0; k < kTeamBlock; ++k) y[k] = sqrt_rn(v[k]);
    }
  } else {
#pragma unroll
    for (int k = 0; k < kTeamBlock; ++k) y[k] = finish_distance<M>(v[k]);
  }
  if (rp.kernel == K_EXP) {
#pragma unroll
    for (int k = 0; k < kTeamBlock; ++k) y[k] = -rp.kp0 * y[k];
  } else {
#pragma unroll
    for (int k = 0; k < kTeamBlock; ++k) y[k] = -y[k] * y[k];
    if (sizeof(T) == 4 ? !rp.gauss_fold : !rp.gauss_pow2) {
#pragma unroll
      for (int k = 0; k < kTeamBlock; ++k) y[k] = y[k] / rp.gauss_den;
    } else if (sizeof(T) == 8) {
#pragma unroll
      for (int k = 0; k < kTeamBlock; ++k) y[k] = y[k] * rp.gauss_inv_den;
    }
  }
  block_exp(y, rp);
#pragma unroll
  for (int k = 0; k < kTeamBlock; ++k) t[k] = v[k] <= thr[k] ? rp.kp1 * y[k] * w[k] : T(0);
}

template <int D, int M, class T>
__global__ __launch_bounds__(kTeam * kWave) void k_density_team(
    const RunParamsT<T> rp, const EventDesc* __restrict__ events, const T* __restrict__ geo,
    const int32_t* __restrict__ toff, const Item* __restrict__ items,
    const T* __restrict__ sx, int64_t cs,
    const T* __restrict__ sw, const T* __restrict__ sfw, const T* __restrict__ ssig,
    const uint32_t* __restrict__ stag, const int32_t* __restrict__ qperm,
    const T* __restrict__ tbox, T* __restrict__ srho, uint64_t* __restrict__ skey) {
  constexpr int B = kTeamBlock, G = kChunkBlocks;
  using List = TeamList<D, M, T, T>;
  __shared__ SumRelay<T> relay;
  __shared__ List list;
  const int item = xcd_block(blockIdx.x, gridDim.x, rp.xcd_chunk_log2);
  if (item >= rp.max_items) return;
  const Item it = items[item];
  if (it.begin >= it.end) return;  // an empty slot
  const int wave = uniform(threadIdx.x / kWave);
  if (wave == 0) relay_pass(relay, T(0), 0);
  __syncthreads();
  // A lone event's descriptors are loaded beside the item, not after it.
  const int e = rp.n_events == 1 ? 0 : it.event;
  const EventDesc ev = events[e];
  const GeoT<T> geom = event_geo(geo, rp, e, ev.nper);
  const int own = uniform(it.tile);
  TeamQuery<D, T> me;
  me.load(it, qperm, sx, cs, ssig, rp);
  const T wself = me.active ? sw[me.pos] : T(0);
  int lo[D], hi[D];
  me.box(geom, rp.dc, lo, hi);
  const T thr_in = MetricTraits<M>::kSqrt ? rp.dc_sq_max : rp.dc;
  const T* __restrict__ wcol = rp.kernel == K_FLAT ? sfw : sw;
  // k_density's shorter square root: no coordinate of the item below 2^-24.
  bool tiny = M != M_EUCLID;
#pragma unroll
  for (int d = 0; d < D; ++d) tiny = tiny || __builtin_fabs(me.x[d]) < T(0x1p-24);
  const bool normal = ballot(me.active && tiny) == 0ull && thr_in <= std::numeric_limits<T>::max();
  const bool cull = rp.cull != 0;
  const QueryBox<D, T> qb = query_box<D, M>(me.x, me.s, me.active);
  auto keep = [&](const T (&x)[D], const T (&s)[D], T) {
    return !(cull && out_of_reach<D, M>(qb, x, s, rp, thr_in));
  };

  BoxUnion<D> u = box_union(lo, hi);
  int turn = 0;  // chunks of the lists before the current one
  do for (int base = 0; base < u.tiles; base += kWave) {
    TeamGroup<D> g;
    list_tiles(u, base, ev.nper, rp.wrapped, ev.t_base, toff, &g);
    g.number(tile_in_reach<D, M>(g, qb, tbox, rp, thr_in));
    g.boxes(lo, hi);
    // The own tile's lane; on a wrapped dimension it can be listed twice, but no lane's
    // box holds both.
    const uint64_t owns = ballot(g.t == own) & g.held;
    int n = 0;
    for (int c = 0; c < g.looks; c += kTeam * List::kLooks) {
      n = list_round<D, M, T, T>(g, c, n, sx, cs, ssig, wcol, list, keep);
      if (n < List::kFull && c + kTeam * List::kLooks < g.looks) continue;
      const int chunks = (n + G * B - 1) / (G * B);
      for (int k = (wave - turn) & (kTeam - 1); k < chunks; k += kTeam) {
        T t[G][B];
        unsigned any = 0;  // bit q: block q has terms
#pragma unroll 1
        for (int q = 0; q < G; ++q) {
          // The blocks move down one place each time, so that one copy of the code
          // fills them all.
#pragma unroll
          for (int r = 0; r + 1 < G; ++r)
#pragma unroll
            for (int c2 = 0; c2 < B; ++c2) t[r][c2] = t[r + 1][c2];
          any >>= 1;
          const int p = (k * G + q) * B;
          if (p >= n) continue;
          const int last = min(p + B, n) - 1;
          const int s0 = uniform(list.slot[p]), s1 = uniform(list.slot[last]);
          T v[B], w[B], thr[B];
          block_distances(me, list, p, n, rp, v);
#pragma unroll
          for (int c2 = 0; c2 < B; ++c2) {
            w[c2] = list.payload[p + c2];
            thr[c2] = ((g.in >> s0) & 1ull) ? thr_in : T(-1);
          }
          if (s0 != s1) {
#pragma unroll
            for (int c2 = 0; c2 < B; ++c2)
              thr[c2] = ((g.in >> list.slot[min(p + c2, last)]) & 1ull) ? thr_in : T(-1);
          }
          block_terms<M>(v, w, thr, normal, rp, t[G - 1]);
          // K(i, i) = 1: the point's own term is its weight.
          if ((((owns >> s0) << s0) & (~0ull >> (63 - s1))) &&
              (s0 != s1 || ballot(me.pos >= list.j[p] && me.pos <= list.j[last]) != 0ull)) {
#pragma unroll
            for (int c2 = 0; c2 < B; ++c2)
              if (list.j[p + c2] == me.pos && v[c2] <= thr[c2]) t[G - 1][c2] = wself;
          }
          any |= 1u << (G - 1);
        }
        // The turn: short and on every wave's way, so it goes first on its SIMD.
        T rho = relay_take(relay, turn + k);
        __builtin_amdgcn_s_setprio(3);
#pragma unroll
        for (int q = 0; q < G; ++q) {
          if ((any >> q) & 1u) {
#pragma unroll
            for (int c2 = 0; c2 < B; ++c2) rho += t[q][c2];
          }
        }
        relay_pass(relay, rho, turn + k + 1);
        __builtin_amdgcn_s_setprio(0);
      }
      turn += chunks;
      n = 0;
      __syncthreads();  // the list is free again
    }
  } while (next_tile_run(u));
  if (wave != 0) return;
  const T rho = relay_take(relay, turn);
  if (me.active) {
    srho[me.pos] = rho;
    skey[me.pos] = density_key(rho, stag[me.pos]);
  }
}

// ---------------------------------------------------------------------------
// Nearest-higher. Candidates that agree in distance, density and tag (user tags only)
// go to the first in the reference's order, so their place in it is compared last.
// With the default tags the own tile comes first: its points settle most bounds
// before the other tiles are looked at.
// ---------------------------------------------------------------------------
template <int D, int M, class T>
__global__ __launch_bounds__(kTeam * kWave) void k_nearest_higher_team(
    const RunParamsT<T> rp, const EventDesc* __restrict__ events, const T* __restrict__ geo,
    const int32_t* __restrict__ toff, const Item* __restrict__ items,
    const T* __restrict__ sx, int64_t cs,
    const T* __restrict__ ssig, const T* __restrict__ su, const uint32_t* __restrict__ stag,
    const T* __restrict__ srho, const uint64_t* __restrict__ skey,
    const int32_t* __restrict__ qperm, const T* __restrict__ tbox, int32_t* __restrict__ snh,
    T* __restrict__ sdelta) {
  using U = typename FloatBits<T>::UInt;
  using List = TeamList<D, M, T, uint64_t>;
  constexpr int B = kTeamBlock;
  __shared__ List list;
  __shared__ U bounds[kWave];  // the bits of non-negative bounds order as the bounds do
  __shared__ T best_delta[kTeam][kWave], best_rho[kTeam][kWave];
  __shared__ uint32_t best_tag[kTeam][kWave];
  __shared__ int32_t best_nh[kTeam][kWave], best_order[kTeam][kWave];
  const int item = xcd_block(blockIdx.x, gridDim.x, rp.xcd_chunk_log2);
  if (item >= rp.max_items) return;
  const Item it = items[item];
  if (it.begin >= it.end) return;  // an empty slot
  const int wave = uniform(threadIdx.x / kWave);
  const int lane = lane_id();
  // A lone event's descriptors are loaded beside the item, not after it.
  const int e = rp.n_events == 1 ? 0 : it.event;
  const EventDesc ev = events[e];
  const GeoT<T> geom = event_geo(geo, rp, e, ev.nper);
  const int own = uniform(it.tile);
  HigherQuery<D, M, T> me;
  me.load(it, qperm, sx, cs, ssig, su, stag, srho, rp);
  int lo[D], hi[D];
  me.box(geom, rp.dm, lo, hi);
  if (wave == 0) bounds[lane] = std::numeric_limits<U>::max();
  __syncthreads();
  const bool cull = rp.cull != 0;
  const QueryBox<D, T> qb = query_box<D, M>(me.x, me.s, me.active);
  const uint64_t kmin = wave_min_key_bound(me.key);
  T bmax = wave_max_f(me.active ? me.bound : -std::numeric_limits<T>::infinity());
  auto keep = [&](const T (&x)[D], const T (&s)[D], uint64_t key) {
    return block_may_be_higher(key, kmin, T(0)) &&
           !(cull && out_of_reach<D, M>(qb, x, s, rp, bmax));
  };
  int order = 0;     // of the best candidate
  int listed = 0;    // candidates of the lists before the current one
  auto search = [&](const TeamGroup<D>& g) {
    int n = 0;
    for (int c = 0; c < g.looks; c += kTeam * List::kLooks) {
      n = list_round<D, M, T, uint64_t>(g, c, n, sx, cs, ssig, skey, list, keep);
      if (n < List::kFull && c + kTeam * List::kLooks < g.looks) continue;
      for (int p = wave * B; p < n; p += kTeam * B) {
        const int last = min(p + B, n) - 1;
        const int s0 = uniform(list.slot[p]), s1 = uniform(list.slot[last]);
        T v[B];
        uint64_t key[B], key_in[B];
        block_distances(me, list, p, n, rp, v);
#pragma unroll
        for (int k = 0; k < B; ++k) {
          key[k] = list.payload[p + k];
          key_in[k] = ((g.in >> s0) & 1ull) ? me.key : ~0ull;
        }
        if (s0 != s1) {
#pragma unroll
          for (int k = 0; k < B; ++k)
            key_in[k] = ((g.in >> list.slot[min(p + k, last)]) & 1ull) ? me.key : ~0ull;
        }
        T m = std::numeric_limits<T>::infinity();
#pragma unroll
        for (int k = 0; k < B; ++k)
          m = fmin_t(m, key_maybe_higher(key[k], key_in[k], T(0))
                            ? v[k] : std::numeric_limits<T>::infinity());
        if (ballot(m <= me.bound) != 0ull) {
#pragma unroll
          for (int k = 0; k < B; ++k) {
            if (key_maybe_higher(key[k], key_in[k], T(0)) && v[k] <= me.bound) {
              const int j = list.j[p + k];
              bool took = false;
              if constexpr (sizeof(T) == 4) {
                const float rj = key_rho(key[k]);
                took = me.consider(v[k], rj, rj > 0.0f ? static_cast<uint32_t>(key[k]) : stag[j], j);
              } else {
                const uint32_t tj = stag[j];
                if (key_higher(key[k], tj, key_in[k], me.tag, T(0)))
                  took = me.consider(v[k], srho[j], tj, j);
              }
              if (took) order = listed + p + k;
            }
          }
        }
      }
      listed += n;
      n = 0;
      // The waves' bounds together: what is left out by them cannot win.
      U bits;
      __builtin_memcpy(&bits, &me.bound, sizeof(bits));
      atomicMin(&bounds[lane], bits);
      __syncthreads();  // and the list is free again
      bits = bounds[lane];
      __builtin_memcpy(&me.eff_thr, &bits, sizeof(bits));
      me.bound = me.eff_thr;
      bmax = wave_max_f(me.active ? me.bound : -std::numeric_limits<T>::infinity());
    }
  };

  TeamGroup<D> g;
  const bool own_first = !rp.has_tags;
  if (own_first) {
    bool in_own = me.active;
    int r = own - ev.t_base;
#pragma unroll
    for (int d = D - 1; d >= 0; --d) {
      const int b = r % ev.nper;
      r /= ev.nper;
      g.b[d] = b;
      in_own = in_own && (((lo[d] <= b) && (b <= hi[d])) ||
                          (rp.wrapped[d] && (lo[d] <= b + ev.nper) && (b + ev.nper <= hi[d])));
    }
    g.t = own;
    g.j0 = toff[own];
    g.j1 = toff[own + 1];
    g.number(lane == 0);
    g.in = in_own ? 1ull : 0ull;
    search(g);
  }
  BoxUnion<D> u = box_union(lo, hi);
  do for (int base = 0; base < u.tiles; base += kWave) {
    list_tiles(u, base, ev.nper, rp.wrapped, ev.t_base, toff, &g);
    g.number(!(own_first && g.t == own) && tile_in_reach<D, M>(g, qb, tbox, rp, bmax));
    g.boxes(lo, hi);
    search(g);
  } while (next_tile_run(u));

  if (wave != 0) {
    best_delta[wave][lane] = me.delta;
    best_rho[wave][lane] = me.rho_nh;
    best_tag[wave][lane] = me.tag_nh;
    best_nh[wave][lane] = me.nh;
    best_order[wave][lane] = order;
  }
  __syncthreads();
  if (wave != 0) return;
  for (int w = 1; w < kTeam; ++w) {
    const int nh = best_nh[w][lane], o = best_order[w][lane];
    if (nh < 0) continue;
    const bool better =
        me.nh < 0 || me.beats(best_delta[w][lane], best_rho[w][lane], best_tag[w][lane], o < order);
    if (better) {
      me.take(best_delta[w][lane], best_rho[w][lane], best_tag[w][lane], nh);
      order = o;
    }
  }
  if (me.active) {
    snh[me.pos] = me.nh;
    sdelta[me.pos] = me.delta;
  }
}

}  // namespace clue_dev
