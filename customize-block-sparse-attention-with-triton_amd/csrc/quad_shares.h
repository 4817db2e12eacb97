// Into how many shares the list of a row block is cut (fwd_short_kernel; fwd_quad_kernel, fwd_wide_kernel), by its own length.  Plain C++ (constexpr functions are
// usable on the device too).
#pragma once
#include "place.h"

namespace bsattn {

// fwd_short_kernel: shares of a list of len tiles, `split` at most (2 to 4), of at least 2^shift tiles each, and where share c begins (c = shares: the
// list's end).  Without divisions, which stand in front of a workgroup's first access: launches of short lists take 0.1 to 0.3 us less without them
// (1 head N = 3400 keep 0.1 10.25 -> 9.95, a window of 0.1 8.60 -> 8.39, N = 2048 keep 0.1 8.94 -> 8.82; where lists are never shared 9.93, 8.25, 8.80).
constexpr int short_shares(int len, int split, int shift) {
  const int n = len >> shift;
  return n < 2 ? 1 : n < split ? n : split;
}
constexpr int short_share_begins(int len, int c, int shares) {      // len * c / shares, below 2^16
  const int n = len * c;
  return shares == 1 ? n : shares == 2 ? n / 2 : shares == 3 ? (int)((unsigned)n * 43691u >> 17) : n / 4;
}

constexpr int SHARE_SAMPLE = 4;       // lists looked at in the middle and at the end of a head
constexpr int SHARE_MIN_BLOCKS = 8;   // row blocks of a head whose lists may be cut, at least

// len: tiles of the list; mid, end: of SHARE_SAMPLE lists in the middle of the head and of its last ones; tail: shares that a list of
// the last, incomplete round of workgroups is cut into (tail_of; 1: it is in front of it); load: row blocks per resident workgroup, times
// 4096; most: shares that a list gets by its length.
// Where the lists grow along the head (causal masks), those above the mean are cut into shares of about the mean work of a resident
// workgroup, and so are lists of twice the mean in any head, in launches of one round (5 heads N = 8192 block-causal, D = 256, in 1.25
// rounds 217 -> 225 us).  least: tiles of a share, at least.  (Lists of like length in one round of workgroups stay whole: cutting
// some of them by chance of a random mask costs a hand-off and evens out nothing, 6 heads N = 4096 keep 0.3 36 -> 47 us.)
constexpr int quad_shares(int len, int mid, int end, int tail, int load, int most, int least) {
  int n = tail;
  const bool grows = 2 * end > 3 * mid;
  if (load <= 4096 && SHARE_SAMPLE * len > (grows ? mid : 2 * mid)) {
    const long long target = (long long)mid * load;                      // times SHARE_SAMPLE * 4096
    const long long work = (long long)len * SHARE_SAMPLE * 4096;
    const int even = target > 0 ? (int)((work + target / 2) / target < most ? (work + target / 2) / target : most) : most;
    n = n > even ? n : even;
  }
  const int fit = len / least;
  n = n < fit ? n : fit;
  return n > 1 ? n : 1;
}

// The lists of the last, incomplete round of workgroups: from which workgroup on they are, and into how many shares those of at least `len`
// tiles are cut.  As many as fit the round, XCD by XCD (170 lists in three shares each are 66 workgroups on some XCDs, with 64 places: D = 128
// 1 head N = 10880 dense 120 us, 99 by pairs).  Where two do not fit the only round that there is, so many that the rounds of shares take least,
// if a list saves FILL_GAIN tiles by it.  us, whole / cut: D = 128 4 heads N = 4352 dense (68 tiles, 23 saved) 80 / 75, keep 0.3 (20, 7) 35 / 42,
// 3 heads N = 5632 dense (88, 29) 101 / 88, 1 head N = 17920 token window of 4480 (70, 23) 77 / 82, of 8064 (126, 42) 124 / 117; D = 256
// 3 heads N = 6016 dense (94, 31) 173 / 153, 4 heads N = 4608 keep 0.3 (22, 7) 61 / 62.
constexpr int FILL_GAIN = 26;
struct TailShares { int from, shares, len; };
constexpr TailShares tail_of(int rows, int slots, int split) {
  const int left = rows % slots, per_xcd = (left + XCDS - 1) / XCDS, places = slots / XCDS > 1 ? slots / XCDS : 1;
  TailShares tail = {rows - left, 1, 0};
  if (left == 0) return tail;
  const int fit = places / per_xcd;
  if (fit > 1 || rows >= slots) { tail.shares = fit < 1 ? 1 : fit < split ? fit : split; return tail; }
  int rounds = 1;                      // the best so far: `rounds` of lists in `shares` shares
  for (int n = 2; n <= split; ++n) {
    const int r = (n * per_xcd + places - 1) / places;
    if (r * tail.shares < rounds * n) { rounds = r; tail.shares = n; }
  }
  if (tail.shares > rounds) tail.len = (FILL_GAIN * tail.shares + tail.shares - rounds - 1) / (tail.shares - rounds);
  return tail;
}

}  // namespace bsattn
