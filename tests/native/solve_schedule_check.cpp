// Checks the launch schedules of the wide solves on the host: every
// (block row, member, column tile) exactly once and no workgroup besides, in
// sweep order, nothing written past the schedule's arrays.  Prints "ok".
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "solve_schedule.hpp"

using namespace pgp;

#define CHECK(c)                                               \
  do {                                                         \
    if (!(c)) {                                                \
      std::printf("line %d, case %s: %s\n", __LINE__, name, #c); \
      std::exit(1);                                            \
    }                                                          \
  } while (0)

struct Guarded {
  SolveSched ss;
  int32_t guard[64];
};

static int last_le(const int32_t* pre, int n, int v) {  // the last i < n with pre[i] <= v
  int i = n - 1;
  while (pre[i] > v) --i;
  return i;
}

// members of nb[m] block rows (not increasing) and mt[m] column tiles
static void each_once(const char* name, const std::vector<int>& nb, const std::vector<int>& mt) {
  const int members = (int)nb.size();
  long long units = 0;
  for (int m0 = 0, n = 0; m0 < members; m0 += n) {
    Guarded g;
    std::memset(&g, 0x5a, sizeof g);
    n = fill_tiles(g.ss, members - m0, [&](int m) { return mt[m0 + m]; });
    CHECK(n >= 1 && n == g.ss.members && m0 + n <= members);
    std::vector<std::vector<int>> seen(n);
    for (int m = 0; m < n; ++m) seen[m].assign((size_t)nb[m0 + m] * mt[m0 + m], 0);
    int next = 0;
    for (int row0 = 0; row0 < nb[m0]; row0 += ROWS_MAX) {
      const int tot = fill_rows(g.ss, row0, [&](int m) { return nb[m0 + m]; });
      units += tot;
      CHECK(g.ss.row0 == row0 && g.ss.count <= ROWS_MAX && g.ss.rows[g.ss.count] == tot);
      for (int r = 0; r < g.ss.count; ++r) CHECK(row0 + r == next++);
      for (int u = 0; u < tot; ++u) {
        const int r = last_le(g.ss.rows, g.ss.count, u), local = u - g.ss.rows[r];
        const int m = g.ss.nct > 0 ? local / g.ss.nct : last_le(g.ss.tiles, n, local);
        const int ct = local - (g.ss.nct > 0 ? m * g.ss.nct : g.ss.tiles[m]);
        CHECK(m < n && row0 + r < nb[m0 + m] && ct >= 0 && ct < mt[m0 + m]);
        ++seen[m][(size_t)(row0 + r) * mt[m0 + m] + ct];
      }
    }
    CHECK(next == nb[m0]);
    for (int32_t v : g.guard) CHECK(v == 0x5a5a5a5a);
    for (auto& s : seen)
      for (int v : s) CHECK(v == 1);
  }
  long long want = 0;
  for (int m = 0; m < members; ++m) want += (long long)nb[m] * mt[m];
  CHECK(units == want);
}

int main() {
  each_once("one block row", {1}, {3});
  each_once("a full launch", {512}, {2});
  each_once("one row more", {513}, {2});
  each_once("three launches", {1100}, {1});
  each_once("members across launches", {1030, 700, 512, 511, 9}, {3, 3, 3, 3, 3});
  each_once("uneven tiles", {40, 40, 17, 16, 1}, {1, 79, 4, 16, 128});
  each_once("some without tiles", {40, 33, 17, 16, 1}, {0, 5, 0, 128, 0});
  each_once("uneven across launches", {1030, 700, 512, 511, 9}, {2, 1, 3, 1, 4});
  std::vector<int> nb, mt;
  for (int m = 0; m < 600; ++m) {
    nb.push_back(64 - m / 10);
    mt.push_back(1);
  }
  each_once("more members than an uneven launch, even", nb, mt);
  mt[3] = 79;
  mt[255] = 2;
  mt[256] = 3;
  mt[599] = 5;
  each_once("more members than an uneven launch", nb, mt);
  for (int m = 0; m < 300; ++m) mt[m] = 0;
  each_once("none with tiles in the first launch", nb, mt);
  std::puts("ok");
  return 0;
}
