// Launch schedules of the wavefront solves with many right-hand sides, as
// plain host code.
#pragma once
#include <cstdint>

namespace pgp {

// A launch holds block rows [row0, row0 + count) of the sweep (every
// member's first, second, ... in sweep order); row0 + r's workgroups are
// rows[r] .. rows[r + 1], member after member, a member's workgroups its
// column tiles of the launch.  Longer sweeps take several launches: the rows
// before row0 are complete when a launch starts.  Passed by value as a kernel
// argument, of 4 KB at most.
constexpr int ROWS_MAX = 512;
constexpr int UNEVEN_MAX = 256;
struct SolveSched {
  int32_t row0, count;
  int32_t members;
  int32_t nct;  // column tiles of every member; 0: they differ
  int32_t rows[ROWS_MAX + 1];
  int32_t tiles[UNEVEN_MAX + 1];  // (nct = 0) column tiles of the members before m
};
static_assert(sizeof(SolveSched) <= 3584, "a kernel argument beside pointers");

// The tile part of the schedules of `members` members with tiles_of(m) column
// tiles each: all of them where the counts agree, else the first UNEVEN_MAX.
// Returns how many members it holds.
template <class Tiles>
inline int fill_tiles(SolveSched& ss, int members, Tiles tiles_of) {
  int m = 1;
  while (m < members && tiles_of(m) == tiles_of(0)) ++m;
  ss.nct = m == members ? tiles_of(0) : 0;
  ss.members = ss.nct > 0 || members < UNEVEN_MAX ? members : UNEVEN_MAX;
  if (ss.nct > 0) return members;
  ss.tiles[0] = 0;
  for (int i = 0; i < ss.members; ++i) ss.tiles[i + 1] = ss.tiles[i] + tiles_of(i);
  return ss.members;
}

// The launch from block row row0 on, of the members of ss with nb_of(m) block
// rows each (not increasing); returns its workgroups.
template <class Nb>
inline int fill_rows(SolveSched& ss, int row0, Nb nb_of) {
  const int left = nb_of(0) - row0;
  ss.row0 = row0;
  ss.count = left < ROWS_MAX ? left : ROWS_MAX;
  int tot = 0, n = ss.members;
  for (int r = 0; r < ss.count; ++r) {
    ss.rows[r] = tot;
    while (nb_of(n - 1) <= row0 + r) --n;
    tot += ss.nct > 0 ? n * ss.nct : ss.tiles[n];
  }
  ss.rows[ss.count] = tot;
  return tot;
}

}  // namespace pgp
