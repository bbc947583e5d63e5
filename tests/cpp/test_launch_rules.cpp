// The rules by which the host sizes and shapes a launch, on the CPU (built with g++
// under the address and undefined-behaviour sanitizers).
#include <cstdio>
#include <cstring>
#include <vector>

#include "clue_host.h"

static int g_fail = 0, g_pass = 0;
#define CHECK(cond)                                              \
  do {                                                           \
    if (cond) {                                                  \
      ++g_pass;                                                  \
    } else {                                                     \
      ++g_fail;                                                  \
      std::printf("FAIL %s:%d: %s\n", __FILE__, __LINE__, #cond); \
    }                                                            \
  } while (0)

using namespace clue_rt;

// One event too large for the fused stages beside many small ones: the sort's digit
// counts grow with the points, however many events they come in.
static void test_sort_histogram() {
  for (int D = 1; D <= 10; ++D)
    for (uint32_t small : {1u, 10u, 64u, 256u, 700u, 2049u})
      for (int count : {0, 1, 100, 5000, 100000}) {
        std::vector<uint32_t> sizes(static_cast<size_t>(count) + 1, small);
        sizes[0] = 140000;
        BatchPlan bp;
        std::string err;
        CHECK(plan_batch(D, 0, sizes.data(), count + 1, nullptr, &bp, &err) == CLUE_OK);
        CHECK(bp.event_order.empty());  // the radix path
        WorkspaceShape w;
        w.D = D;
        w.n = bp.n_total;
        w.events = static_cast<int64_t>(bp.events.size());
        w.chunks = static_cast<int64_t>(bp.chunks.size());
        w.tiles = bp.n_tiles_total;
        w.max_items = bp.max_items;
        size_t b[S_NUM];
        workspace_requests(w, b);
        CHECK(b[S_HIST] <= 4 * static_cast<size_t>(bp.n_total) + (64 << 10));
        // Room for the counts of every block of the sort and the totals.
        const int64_t blocks = sort_by_chunk(w.n, w.chunks) ? w.chunks : (w.n + 2047) / 2048;
        const int bits = clue_dev::radix_plan(bp.key_bits).bits;
        CHECK(b[S_HIST] >= sizeof(int32_t) * static_cast<size_t>((blocks + 1) << bits));
      }
  // A lone event's chunks are full: they are the blocks.
  for (int64_t n : {1, 2047, 2048, 2049, 140000, 1 << 20})
    CHECK(sort_by_chunk(n, (n + 2047) / 2048));
}

static bool team(int D, int per_tile, uint32_t n, int count = 1) {
  std::vector<uint32_t> sizes(static_cast<size_t>(count), n);
  BatchPlan bp;
  std::string err;
  CHECK(plan_batch(D, per_tile, sizes.data(), count, nullptr, &bp, &err) == CLUE_OK);
  return bp.team;
}

// Teams of waves where an item's walk is long; one wave per item where the items are many
// and hold few points.
static void test_team_rule() {
  for (int D = 1; D <= 7; ++D)
    for (uint32_t n : {1u, 300u, 5003u, 20011u, 30000u, 65536u}) CHECK(team(D, 0, n));
  CHECK(team(2, 0, 110000) && !team(2, 0, 110001));
  CHECK(team(2, 1, 3000) && team(2, 1, 8000) && team(2, 16, 50000));
  CHECK(!team(2, 1, 50000) && !team(2, 1, 100000) && !team(2, 4, 100000) && !team(3, 4, 100000));
  CHECK(!team(6, 4, 20000) && !team(6, 8, 100000) && !team(8, 0, 50000));
  CHECK(team(2, 0, 1000, 48) && team(2, 0, 400, 100) && team(3, 0, 4100, 26));
  CHECK(!team(2, 0, 16, 3000) && !team(2, 0, 1, 40000) && !team(2, 0, 1000, 50));
}

// The tuning a batch is given, fixed, gives the same launch.
static void test_chosen_tuning_keeps_the_launch() {
  for (int D = 1; D <= 10; ++D)
    for (uint32_t n : {1u, 300u, 5003u, 50000u, 110000u, 131072u, 1u << 20})
      for (int count : {1, 2, 50})
        for (int ppt : {0, 1, 16}) {
          if (int64_t(n) * count > (1 << 21)) continue;
          std::vector<uint32_t> sizes(static_cast<size_t>(count), n);
          BatchPlan a, b;
          std::string err;
          CHECK(plan_batch(D, ppt, sizes.data(), count, nullptr, &a, &err) == CLUE_OK);
          const clue_tuning t = a.tuning;
          CHECK(plan_batch(D, ppt, sizes.data(), count, &t, &b, &err) == CLUE_OK);
          CHECK(a.team == (t.team != 0) && b.team == a.team);
          CHECK(std::memcmp(&b.tuning, &t, sizeof(t)) == 0);
        }
}

// Every tile of a union once, dimension 0 outermost, in one run or (a small limit) several.
template <int D>
static void check_tile_order(const int (&first)[D], const int (&extents)[D], int64_t most) {
  clue_dev::BoxUnion<D> u{};
  int want[D] = {};
  int64_t count = 0, all = 1;
  for (int d = 0; d < D; ++d) {
    u.lo[d] = first[d];
    u.ext[d] = extents[d];
    all *= extents[d];
  }
  bool same = true, more = true;
  clue_dev::first_tile_run(u, most);
  do {
    for (int idx = 0; idx < u.tiles; ++idx, ++count) {
      int q = idx;
      same = same && more;
      for (int d = D - 1; d >= 0; --d) {
        same = same && u.lo[d] + (d == 0 ? q : q % u.ext[d]) == first[d] + want[d];
        q /= u.ext[d];
      }
      int d = D - 1;
      for (; d >= 0 && ++want[d] == extents[d]; --d) want[d] = 0;
      more = d >= 0;
    }
  } while (clue_dev::next_tile_run(u));
  CHECK(same && count == all);
}

// The widest union of nper tiles per dimension in D, all wrapped: counted in full.
template <int D>
static void check_widest(int nper, int64_t tiles) {
  clue_dev::BoxUnion<D> u{};
  for (int d = 0; d < D; ++d) u.ext[d] = 2 * nper - 1;
  clue_dev::first_tile_run(u);
  int64_t count = 0;
  bool fits = true;
  do {
    fits = fits && u.tiles > 0 && u.tiles <= clue_dev::kTileRunMax;
    count += u.tiles;
  } while (clue_dev::next_tile_run(u));
  CHECK(fits && count == tiles);
}

static void test_tile_runs() {
  for (int64_t most : {int64_t(1), int64_t(5), int64_t(300), clue_dev::kTileRunMax}) {
    check_tile_order<1>({4}, {7}, most);
    check_tile_order<3>({1, 2, 3}, {5, 1, 6}, most);
    check_tile_order<6>({1, 2, 3, 4, 5, 6}, {3, 1, 2, 4, 2, 3}, most);
    check_tile_order<9>({0, 0, 1, 0, 0, 2, 0, 0, 3}, {2, 3, 1, 2, 2, 2, 1, 3, 2}, most);
    check_tile_order<10>({5, 6, 0, 0, 0, 0, 0, 0, 0, 7}, {2, 3, 1, 2, 2, 2, 1, 3, 2, 2}, most);
  }
  // The most tiles per dimension of fewer than 2^26: 8191^2 up to 6^10.
  check_widest<2>(8191, 268337161);
  check_widest<5>(36, 1804229351);
  check_widest<6>(20, 3518743761);
  check_widest<7>(13, 6103515625);
  check_widest<8>(9, 6975757441);
  check_widest<9>(7, 10604499373);
  check_widest<10>(6, 25937424601);
  clue_dev::BoxUnion<10> none{};  // no active lane
  clue_dev::first_tile_run(none);
  CHECK(none.tiles == 0 && !clue_dev::next_tile_run(none));
}

int main() {
  test_tile_runs();
  test_team_rule();
  test_chosen_tuning_keeps_the_launch();
  test_sort_histogram();
  std::printf("%d passed, %d failed\n", g_pass, g_fail);
  return g_fail == 0 ? 0 : 1;
}
