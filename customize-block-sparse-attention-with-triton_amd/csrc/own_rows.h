// Which heads of a launch on ranges of workgroups (fwd_kernel, COOP) go a row block to a workgroup instead, and which row block or part of
// one a workgroup then takes.  Plain C++ (constexpr functions are usable on the device too).
#pragma once

namespace bsattn {

constexpr int OWN_PART_TILES = 8;      // tiles of a part, at least

constexpr int OWN_ROWS_MOST = 512;     // row blocks of a head, at most

// What the host knows: W workgroups per head, the first `firsts` of them first on their compute unit.  most, least: tiles of a head (most = 0:
// none); the longest list has at most long_base tiles and 1 to 1.5 times the mean (long_per_tile: this factor by nb); where compute units have
// more than one row block (not alone), at most a quarter of the lists are longer than 2 tiles and 1.5 times the mean, or 14 and 0.7 times.
struct OwnLines { int most, least, long_base; float long_per_tile, per_tile; bool alone; };
constexpr OwnLines own_lines(int nb, int W, int firsts) {
  if (nb > W || nb > OWN_ROWS_MOST) return {0, 0, 0, 0.f, 0.f, false};
  const bool alone = nb <= firsts, whole = alone || 4 * nb >= 3 * W;      // no row block is left for parts, or no workgroups
  const int most = (alone ? 32 : !whole ? 56 : 20 * nb >= 17 * W ? 64 : 30) * nb;
  const int least = whole || 10 * nb >= 7 * W ? 0 : 17 * nb;
  // (two workgroups of whole row blocks on a compute unit: beside a long one the other has ended early)
  const bool two = whole && !alone;
  return {most, least, alone ? 20 : two ? 16 : 17, (alone ? 1.f : two ? 1.5f : 1.2f) / nb, 1.f / nb, alone};
}

// T: tiles of the head, middle: those of its first nb / 2 row blocks.
constexpr bool own_rows_by_tiles(const OwnLines& l, int T, int nb) { return T <= l.most && (T >= l.least || T <= 4 * nb); }
constexpr bool own_rows_by_middle(int T, int middle) { return 8 * middle > 3 * T; }
// lists longer than this: none, a quarter of them
constexpr int own_rows_longest(const OwnLines& l, int T) { return l.long_base + (int)(l.long_per_tile * T); }
constexpr int own_rows_even(const OwnLines& l, int T) {
  if (l.alone) return own_rows_longest(l, T);
  const float mean = l.per_tile * T;
  const int many = 2 + (int)(1.5f * mean), few = 14 + (int)(0.7f * mean);
  return many > few ? many : few;
}

// The row block of workgroup wg (>= nb: none), which of its parts, and how many these are at most.
struct OwnItem { int row, part, most; };
constexpr OwnItem own_item(int wg, int nb, int W, int firsts) {
  if (wg < firsts || nb <= firsts) return {wg, 0, 1};
  const int most = (W - firsts) / (nb - firsts), i = wg - firsts;
  return {firsts + i / most, i % most, most};
}
constexpr int own_parts(int len, int most) {
  return len < 2 * OWN_PART_TILES ? 1 : len / OWN_PART_TILES < most ? len / OWN_PART_TILES : most;
}

}  // namespace bsattn
