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

// A launch of whole row blocks, nb of each head and W workgroups per head for parts of long ones, which come behind the first `first_ids` ids: one of
// the latter (extra) or not, and which of its kind's `per` items of a head; item >= per: an id that only fills a group up.
// (No more than the row blocks' ids are first ones: an id behind them would be a row block of a head that is not there.)
constexpr int first_ids_of_rows(int resident, int heads, int group, int nb) {
  const int ids = placed(heads, group, nb);
  return resident < ids ? resident : ids;
}
struct PlaceOfRows { Place p; int per; bool extra; };
constexpr PlaceOfRows place_rows(int id, int heads, int group, int nb, int W, int first_ids) {
  const int extras = placed(heads, group, W);
  const bool extra = id >= first_ids && id < first_ids + extras;
  const int L = id < first_ids ? id : extra ? id - first_ids : id - extras, per = extra ? W : nb;
  return {place(L, heads, group, per), per, extra};
}

// A launch of `split` shares of all items (the share is the slowest index, so that a head stays on its XCDs): heads in groups of `group` (a
// multiple of 8), as above; then a last group of 8 `whole` heads and the `rest` in eighths, all of them at once: an XCD has `whole` heads and
// `rest` units, and takes eight items of each of the former and one of each of the latter in turn.
struct Groups { int group, whole, rest; };
struct PlaceOfEight {
  int split, per_share;                    // per_share: workgroups of a share
  int first, first_ids, group, items;      // heads in groups of `group`, their linear ids
  int whole, rest;
  Divisor per_group, in_group;             // group items; group
  Divisor per_rank, in_rank;               // 8 whole + rest; whole
  constexpr Place of(int L, int& share) const {
    for (share = 0; share + 1 < split && L >= per_share; ++share) L -= per_share;
    if (__builtin_expect(L < first_ids, 1)) {
      const int grp = (int)per_group.of((unsigned)L), l = L - grp * group * items, item = (int)in_group.of((unsigned)l);
      return {group * grp + l - item * group, item};
    }
    L -= first_ids;
    const int x = L % XCDS, i = L / XCDS, rank = (int)per_rank.of((unsigned)i), k = i - rank * (XCDS * whole + rest);
    if (k < XCDS * whole) {
      const int j = (int)in_rank.of((unsigned)k);
      return {first + XCDS * (k - j * whole) + x, rank * XCDS + j};
    }
    const int unit = rest * x + k - XCDS * whole;
    return {first + XCDS * whole + unit / XCDS, rank * XCDS + unit % XCDS};
  }
};
constexpr PlaceOfEight place_of_eight(int heads, int items, int split, Groups g) {
  const int first = heads - XCDS * g.whole - g.rest, ids = first * items, per_rank = XCDS * g.whole + g.rest;
  const int n = ids + XCDS * per_rank * ((items + XCDS - 1) / XCDS);
  auto by = [&](int d) { return divisor(d > 0 ? (unsigned)d : 1u, (uint64_t)n); };
  return {split, n, first, ids, g.group, items, g.whole, g.rest, by(g.group * items), by(g.group), by(per_rank), by(g.whole)};
}
constexpr PlaceOfEight place_of_eight(int heads, int items, int split) { return place_of_eight(heads, items, split, Groups{XCDS, 0, heads % XCDS}); }

// The groups for kernels whose workgroups walk a list each: as many heads per XCD at once as its L2 (4 MB) holds the K and V (or Q and dO) of and
// as divide the heads of an XCD, at most 8.  With one head per XCD a causal mask's last heads start their longest lists when the short ones of the
// heads before have ended, and these are all that is left in the end; with more than the L2 holds the sparse uniform masks get slower.
// us, bf16, a forward / its training step, 8 heads at a time and so; block-causal, causal keep 0.25, keep 0.2, dense:
//   D = 64    16 heads N = 4096    55 / 263 ->  54 / 232    27 / 103 ->  24 /  93    32 / 112 ->  31 / 110    91 /  362 ->  91 /  361
//             10 heads N = 4096    45 / 162 ->  36 / 138    21 /  72 ->  17 /  72    25 /  81 ->  24 /  79    70 /  262 ->  70 /  262
//   D = 128   32 heads N = 4096   180 / 712 -> 152 / 647    62 / 268 ->  58 / 263    76 / 321 ->  77 / 323   305 / 1222 -> 306 / 1225
//             64 heads N = 2048   102 / 412 ->  82 / 353    41 / 166 ->  37 / 152    47 / 200 ->  48 / 197   151 /  656 -> 151 /  657
//             24 heads N = 2048    56 / 190 ->  47 / 163    26 /  88 ->  21 /  81    28 / 104 ->  24 /  98    63 /  259 ->  64 /  260
//   D = 256   16 heads N = 2048    63 / 261 ->  56 / 248    30 / 122 ->  26 / 118    33 / 148 ->  29 / 141    77 /  360 ->  77 /  358
// 1.6 times as much where these are all heads (block-causal, causal keep 0.5, keep 0.25, 0.1):
//   D = 128   16 heads N = 6016 (3 MB)   176 / 737 -> 160 / 692    98 / 414 ->  90 / 387   103 / 425 -> 102 / 419    53 / 208 -> 52 / 209
//   D = 256   16 heads N = 3000          94 / 455 ->  88 / 452     57 / 275 ->  54 / 262    62 / 293 ->  61 / 276    39 / 171 -> 38 / 169
// With twice as much the causal launches gain and the sparse uniform ones lose:
//   D = 128   32 heads N = 8192 (4 MB)   560 / 2454 -> 557 / 2419  177 / 762 -> 167 / 741  251 / 1091 -> 267 / 1140 150 / 644 -> 154 / 651   (keep 0.25, causal and not)
//   D = 256   16 heads N = 4096          150 / 717 -> 150 / 705    88 / 424 ->  84 / 404    96 / 461 ->  97 / 452    58 / 274 -> 61 / 277
// Heads beyond a multiple of 8 go out with the last group, but three or more of them behind it where a head and they are more than 1.6 times
// what the L2 holds, or 1.4 times where there is no other group, which these do not touch (D = 128 and 256; the backward of D = 64 loses nothing by
// them).  Behind / with it, forward and step; keep 0.3, 0.1, block-causal, window of 0.3:
//   D = 128   12 heads N = 8192 (8 MB)   161 /  668 -> 163 /  671    68 / 272 ->  71 / 283   244 / 1090 -> 229 / 1008   137 / 562 -> 140 / 555   (not there)
//             15 heads N = 8000          181 /  785 -> 184 /  789    78 / 321 ->  82 / 342   267 / 1168 -> 264 / 1167   157 / 639 -> 158 / 642   (nor there)
//   D = 256   14 heads N = 6000 (12 MB)  211 /  975 -> 222 /  994   105 / 455 -> 109 / 462   297 / 1438 -> 286 / 1358   171 / 767 -> 174 / 779   (nor there)
//             12 heads N = 3000 (6 MB)    67 /  304 ->  66 /  304    35 / 151 ->  35 / 154    94 /  451 ->  89 /  409    54 / 225 ->  54 / 234   (nor there)
//             20 heads N = 3000            88 /  400 ->   89 /  398     50 /  213 ->   49 /  209    146 /  704 ->  131 /  571     79 /  338 ->   78 /  339
//             17 heads N = 5000 (10 MB)  183 /  875 -> 183 /  855    89 / 398 ->  91 / 398   314 / 1532 -> 251 / 1205   153 / 710 -> 151 / 688   (one head alone)
// (A choice by the lists, in the kernels, costs the backward's registers: 8 heads N = 4096 D = 128 dense 334 -> 345.)
constexpr Groups groups_of_heads(int heads, int64_t N, int D) {
  const int64_t bytes = 4 * N * D, fit = (4ll << 20) / bytes;
  const int per_xcd = heads / XCDS, rest = heads % XCDS, most = fit < 1 ? 1 : fit > 8 ? 8 : (int)fit;
  auto fits = [&](int n, int tenths) { return 10 * n * bytes <= (int64_t)tenths * (4 << 20); };      // tenths of the L2
  int n = per_xcd < most ? per_xcd : most;       // (like groups)
  if (rest == 0 && per_xcd <= 8 && fits(per_xcd, 16)) n = per_xcd;
  while (n > 1 && per_xcd % n != 0) --n;
  const bool behind = rest >= 3 && D > 64 && !fits(2, per_xcd > 1 ? 16 : 14);      // (n is 1 then)
  return {XCDS * (n > 1 ? n : 1), rest > 0 && !behind ? n : 0, rest};
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
