// outer_schedule_check <op> <G> <block rows of each member, largest first>:
// prints, per super-step of G block columns of a batch, 1 if its outer update
// is launched in 128-tiles and 0 if in 64-tiles.
#include <cstdio>
#include <cstdlib>

#include "chol_schedule.hpp"

int main(int argc, char** argv) {
  const auto op = (pgp::OuterOp)std::atoi(argv[1]);
  const int G = std::atoi(argv[2]), count = argc - 3;
  auto nb_of = [&](int m) { return std::atoi(argv[3 + m]); };
  for (int s_end = G; s_end < nb_of(0); s_end += G) {
    const int rest = pgp::outer_ahead(op, count, nb_of, s_end, G);
    const int wd = rest < 0 ? 0 : G;
    std::printf("%d ", pgp::outer_takes_wide(op, count, nb_of, s_end, wd, rest) ? 1 : 0);
  }
  std::puts("");
  return 0;
}
