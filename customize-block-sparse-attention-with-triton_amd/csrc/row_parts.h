// Row blocks much longer than the others of their head, and the parts they are cut into (fwd_kernel, one wavefront per row
// block).  Plain C++ (constexpr functions are usable on the device too).
#pragma once
#include <cstdint>

namespace bsattn {

constexpr int LONG_ROW_MIN = 24;      // row blocks up to this many tiles are never cut
constexpr int LONG_PART_MIN = 8;      // shortest part

// Is a row block of len tiles a long one in a head of T tiles in nb row blocks: above 2.5 times the mean length?
constexpr bool is_long_row(int len, int T, int nb) { return len > LONG_ROW_MIN && 2 * (int64_t)nb * len > 5 * (int64_t)T; }

// Tiles of a part (the last ones of a row block may have one less), for `rows` long row blocks of `tiles` together.  A
// part has at least the mean length of the head's row blocks, and as many tiles as leave at most W parts of row blocks
// that are cut: with x tiles there are less than tiles / x + rows parts, and less than 2 tiles / x of row blocks longer than x.
constexpr int long_part_tiles(int tiles, int rows, int W, int mean) {
  const int most = W - rows > W / 2 ? W - rows : W / 2, fit = (tiles + most - 1) / most;
  return fit > mean ? (fit > LONG_PART_MIN ? fit : LONG_PART_MIN) : (mean > LONG_PART_MIN ? mean : LONG_PART_MIN);
}

constexpr int parts_of_row(int len, int part_tiles) { return (len + part_tiles - 1) / part_tiles; }
constexpr int part_begin(int len, int parts, int i) { return (int)((int64_t)len * i / parts); }

}  // namespace bsattn
