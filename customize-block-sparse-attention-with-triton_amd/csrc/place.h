// Which head, and which of its row blocks, column blocks or ranges, a workgroup takes.  Plain C++ (constexpr functions are
// usable on the device too).
//
// Workgroups go to the 8 XCDs round-robin by linear id, and each XCD has an L2 of its own, which one head's K and V (or Q and
// dO) fill.  So an XCD works on as few heads as the balance allows: with a multiple of 8 heads on whole heads, else on a
// stretch of heads / 8 of them.
#pragma once
#include <cstdint>

namespace bsattn {

constexpr int XCDS = 8;

struct Place { int head, item; };

// Division by a number the host knows, for the way from a workgroup's index to its work, in front of which nothing else can
// start: one multiplication in place of the 0.2 us of an integer division.  Exact for n up to the `most` it was made for;
// where that is too large for the reciprocal (mul = 0) an ordinary division.
struct Divisor {
  unsigned d = 1, mul = 0;      // mul: 2^32 / d, rounded up
  constexpr unsigned of(unsigned n) const {
    if (__builtin_expect(mul == 0 && d != 1, 0)) return n / d;       // (out of the way: code that is jumped over costs a fetch)
    return d == 1 ? n : (unsigned)(((uint64_t)n * mul) >> 32);
  }
};
constexpr Divisor divisor(unsigned d, uint64_t most) {      // (2^32 <= mul d < 2^32 + d: the error is below n / 2^32)
  return {d, d > 1 && most * d < (1ull << 32) ? (unsigned)(((1ull << 32) + d - 1) / d) : 0u};
}

// ---- one workgroup per (head, item), the items of all heads of a group first, in ascending order ----
// Linear ids that `heads` heads of a group take.  Heads that are not a multiple of 8 are dealt in eighths: unit 8 head + e
// has the items e, e + 8, ... of a head (so that every unit has early and late ones, which block-causal masks make short
// and long), and XCD x has the units heads x .. heads x + heads - 1.
constexpr int placed_in_group(int heads, int items) {
  return heads % XCDS == 0 ? heads * items : heads * XCDS * ((items + XCDS - 1) / XCDS);
}

constexpr Place place_in_group(int l, int heads, int items) {
  if (heads % XCDS == 0) { const int item = l / heads; return {l - item * heads, item}; }
  const int x = l % XCDS, i = l / XCDS, rank = i / heads, unit = heads * x + (i - rank * heads);
  (void)items;
  return {unit / XCDS, rank * XCDS + unit % XCDS};
}

// The same for all heads, taken in groups of `group` (a multiple of 8) and a last one of what is left.  The item is
// >= items for the ids that only fill a group up.
constexpr int placed(int heads, int group, int items) { return heads / group * group * items + placed_in_group(heads % group, items); }

constexpr Place place(int L, int heads, int group, int items) {
  const int grp = L / (group * items), whole = heads / group, first = (grp < whole ? grp : whole) * group;
  const Place p = place_in_group(L - first * items, grp < whole ? group : heads - first, items);
  return {first + p.head, p.item};
}

// The same for groups of 8 heads in a launch of `split` shares of all items (the share is the slowest index, so that a head stays
// on its XCDs).
struct PlaceOfEight {
  int heads, items, split, per_share;      // workgroups of a share
  Divisor per_group, left;                 // 8 items; heads % 8
  constexpr Place of(int L, int& share) const {
    for (share = 0; share + 1 < split && L >= per_share; ++share) L -= per_share;
    const int grp = heads < XCDS ? 0 : (int)per_group.of((unsigned)L), whole = heads / XCDS;
    if (__builtin_expect(grp < whole, 1)) { const int l = L - grp * XCDS * items; return {XCDS * grp + l % XCDS, l / XCDS}; }
    const int rest = heads % XCDS, l = L - whole * XCDS * items, x = l % XCDS, i = l / XCDS;
    const int rank = (int)left.of((unsigned)i), unit = rest * x + (i - rank * rest);
    return {whole * XCDS + unit / XCDS, rank * XCDS + unit % XCDS};
  }
};
constexpr PlaceOfEight place_of_eight(int heads, int items, int split) {
  const int n = placed(heads, XCDS, items);
  return {heads, items, split, n, divisor((unsigned)(XCDS * items), (uint64_t)n), divisor(heads % XCDS ? (unsigned)(heads % XCDS) : 1u, (uint64_t)n)};
}

// ---- W ranges per head, all resident at once ----
// The first `fast` linear ids are the first workgroups on their compute units: the heads share them as evenly as they go
// (head h gets fast / heads of them and one more if h < fast % heads), and a head's ranges 0, 1, ... are its fast ones.  Both
// kinds are dealt out to the XCDs in stretches, head after head.
constexpr int xcd_position(int L, int n) {       // the n ids of XCD 0, of XCD 1, ... one after the other
  const int x = L % XCDS, rest = n % XCDS;
  return x * (n / XCDS) + (x < rest ? x : rest) + L / XCDS;
}

// quot, rest: fast / heads, fast % heads
constexpr Place place_range(int L, int heads, int W, int fast, int quot, int rest) {
  const bool is_fast = L < fast;
  const int pos = is_fast ? xcd_position(L, fast) : xcd_position(L - fast, heads * W - fast);
  const int more = is_fast ? quot + 1 : W - quot - 1, less = is_fast ? quot : W - quot;     // ranges of a head h < rest, of another
  const bool early = pos < rest * more;
  const int per = early ? more : less, p = early ? pos : pos - rest * more, h = p / per;
  return {early ? h : rest + h, p - h * per + (is_fast ? 0 : early ? quot + 1 : quot)};
}

}  // namespace bsattn
