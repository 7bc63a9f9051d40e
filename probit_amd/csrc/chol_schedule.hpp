// Which tiles the outer updates of the Cholesky take and where they run, as
// plain host code (the counts, constexpr, on the device too).
#pragma once
#include <cstdint>

namespace pgp {

enum OuterOp { OUTER_FP64, OUTER_FP32, OUTER_BF16 };

// 64-tiles of the first wd block columns of a lower triangle of Tk.
constexpr int outer_tiles64(int Tk, int wd) {
  const int w = wd < Tk ? wd : Tk;
  return w * Tk - w * (w - 1) / 2;
}

// 128-tiles of a lower triangle of tb block rows
constexpr int tiles128(int tb) {
  const int t = (tb + 1) / 2;
  return tb > 0 ? t * (t + 1) / 2 : 0;
}

// 128-tiles of an outer update of a lower triangle of tb block rows, or (wd >
// 0) of its first wd block columns and, of the triangle right of them, all but
// the last `rest` tiles.
constexpr int outer_tiles128(int tb, int wd, int rest) {
  if (wd == 0) return tiles128(tb);
  const int a = tiles128(tb), t = tiles128(tb - wd);
  return a - t + (t > rest ? t - rest : 0);
}

// Whether an outer update of t128 128-tiles takes them, or the 64-tiles.  Two
// workgroups of 128-tiles fit a CU, and a CU given one more than its
// neighbours keeps the launch waiting for a whole tile (K = 512 FP64: 73 us
// for one, 133 for two), four times a 64-tile's.  Measured, 128- against
// 64-tiles: FP64 (K = 512) 210 tiles 79 / 93 us, 300 132 / 121, 406 133 / 164,
// 528 200 / 207, 1176 335 / 424; FP32 (K = 768) 210 64 / 69, 351 109 / 101,
// 528 160 / 148, 741 163 / 196; 78 tiles (of 24 block rows) 74 / 50 FP64.
// BF16 is bound by C's bytes and the operands', not by the tile's MFMAs: 210
// 15 / 23, 300 24 / 29, 528 34 / 47.
inline bool outer_wide(long long t128, bool bf16) {
  constexpr int CUS = 256;
  if (bf16) return t128 >= 3 * CUS / 4;
  return t128 >= 5 * CUS / 2 || (t128 >= 3 * CUS / 4 && t128 <= CUS);
}

// The same for the members m < count, of nb_of(m) block rows, after the
// super-step that ends at block row s_end (wd, rest as above): the 64-tiles
// hold whole block columns only.
template <class Nb>
inline bool outer_takes_wide(OuterOp op, int count, Nb nb_of, int s_end, int wd, int rest) {
  long long t128 = 0;
  for (int m = 0; m < count; ++m) {
    const int tb = nb_of(m) - s_end;
    t128 += outer_tiles128(tb, wd, rest);
    if (wd > 0 && tiles128(tb - wd) > rest) return true;
  }
  return wd % 2 == 0 && outer_wide(t128, op == OUTER_BF16);
}

constexpr int LOOKB = 64;  // members of a launch with outer tiles

// Outer tiles that a super-step's launch takes along, one workgroup a CU, in
// the CUs that its `chain` workgroups on the column chain and its `rows` rows
// below leave idle, and how many of them go before the rows (first).  The
// chain lasts `all` tiles' times (in tenths; FP64 100 us for 6 columns, 60 a
// tile of K = 384; FP32 175 for 12, 65 of K = 768; BF16 100 for 8, 13 of K =
// 512; both grow with G).  A row below takes about as long as the chain if it
// starts with it, waiting most of the time, and less once the chain has got
// ahead: few rows start with it, many after the first rounds of tiles.  Many
// FP32 rows, two a CU without outer tiles, take none (N = 16384, 244 rows: 334
// us with 240 tiles, 194 without and 51 for the tiles).
inline int look_tiles(OuterOp op, int chain, int rows, int& first) {
  const int all = op == OUTER_FP64 ? 20 : op == OUTER_BF16 ? 80 : 28;
  const int head = op == OUTER_BF16 ? 30 : 10;
  if (op == OUTER_FP32 && rows > 160) return first = 0;
  first = rows <= 96 || chain > 256 ? 0 : head * (256 - chain) / 10;
  return first + (all - (first > 0 ? head : 0)) * (256 - chain - rows) / 10;
}

// The outer update after the super-step that ends at block row s_end: how many
// of each member's last tiles go into the next super-step's launch (of G
// columns), -1: the whole update before it.
template <class Nb>
inline int outer_ahead(OuterOp op, int count, Nb nb_of, int s_end, int G) {
  int nb = 0, chain = 0, rows = 0;  // row blocks of the next super-step, and below it
  for (int m = 0; m < count; ++m) {
    const int left = nb_of(m) - s_end;
    nb = nb_of(m) > nb ? nb_of(m) : nb;
    chain += left < 0 ? 0 : left < G ? left : G;
    rows += left > G ? left - G : 0;
  }
  if (count > LOOKB || s_end + G >= nb || G % 2 != 0) return -1;
  int first;
  const int ahead = look_tiles(op, chain, rows, first) / count;
  return ahead > 0 ? ahead : -1;
}

}  // namespace pgp
