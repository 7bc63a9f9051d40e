// Checks the launch schedules of the wide solves on the host: every
// (block row, member, column tile) exactly once, in sweep order, and nothing
// written past the schedule's arrays.  Prints "ok" and returns 0.
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
  RowSched rows;
  int32_t guard[64];
};

static void rows_once(const char* name, const std::vector<int>& nb, int nct) {
  std::vector<std::vector<int>> seen(nb.size());
  for (size_t m = 0; m < nb.size(); ++m) seen[m].assign((size_t)nb[m] * nct, 0);
  int next = 0;
  for (int row0 = 0; row0 < nb[0]; row0 += ROWS_MAX) {
    Guarded g;
    std::memset(&g, 0x5a, sizeof g);
    const int tot = fill_rows(g.rows, row0, nb[0], (int)nb.size(), [&](int m) { return nb[m]; }, nct);
    for (int32_t v : g.guard) CHECK(v == 0x5a5a5a5a);
    CHECK(g.rows.row0 == row0 && g.rows.count <= ROWS_MAX && g.rows.pre[g.rows.count] == tot);
    for (int r = 0; r < g.rows.count; ++r) {
      const int row = row0 + r;
      CHECK(row == next++);
      for (int u = g.rows.pre[r]; u < g.rows.pre[r + 1]; ++u) {
        const int m = (u - g.rows.pre[r]) / nct, ct = (u - g.rows.pre[r]) % nct;
        CHECK(m < (int)nb.size() && row < nb[m]);
        ++seen[m][(size_t)row * nct + ct];
      }
    }
  }
  CHECK(next == nb[0]);
  for (auto& s : seen)
    for (int v : s) CHECK(v == 1);
}

int main() {
  rows_once("one block row", {1}, 3);
  rows_once("a full launch", {512}, 2);
  rows_once("one row more", {513}, 2);
  rows_once("three launches", {1100}, 1);
  rows_once("members across launches", {1030, 700, 512, 511, 9}, 3);
  std::puts("ok");
  return 0;
}
