// Launch schedules of the wavefront solves with many right-hand sides, as
// plain host code.
#pragma once
#include <cstdint>

namespace pgp {

// A launch holds block rows [row0, row0 + count) of the sweep (every
// member's first, second, ... in sweep order); row0 + r's workgroups are
// pre[r] .. pre[r + 1].  Longer sweeps take several launches: the rows before
// row0 are complete when a launch starts.  Passed by value as a kernel
// argument.
constexpr int ROWS_MAX = 512;
struct RowSched {
  int32_t row0, count;
  int32_t pre[ROWS_MAX + 1];
};

// The launch from block row row0 on, of `members` members with nb_of(m) block
// rows (at most nb) and nct workgroups a row each; returns its workgroups.
template <class Nb>
inline int fill_rows(RowSched& rows, int row0, int nb, int members, Nb nb_of, int nct) {
  rows.row0 = row0;
  rows.count = nb - row0 < ROWS_MAX ? nb - row0 : ROWS_MAX;
  int tot = 0;
  for (int r = 0; r < rows.count; ++r) {
    rows.pre[r] = tot;
    for (int m = 0; m < members; ++m)
      if (nb_of(m) > row0 + r) tot += nct;
  }
  rows.pre[rows.count] = tot;
  return tot;
}

}  // namespace pgp
