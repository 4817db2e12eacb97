// Checks csrc/place.h on the host: every (head, item) is taken by exactly one workgroup, fast ranges come first and are
// shared evenly, and an XCD works on as few heads as the balance allows.
#include <cstdio>
#include <vector>
#include "place.h"
using namespace bsattn;

static int bad(const char* what, int a, int b, int c) { std::printf("%s: %d %d %d\n", what, a, b, c); return 1; }

int main() {
  for (int heads = 1; heads <= 50; ++heads)
    for (int group = 8; group <= 24; group += 8)
      for (int items : {1, 2, 5, 7, 8, 9, 31, 64, 100}) {
        std::vector<int> seen(heads * items);
        std::vector<std::vector<int>> of_xcd(XCDS, std::vector<int>(heads));
        for (int L = 0; L < placed(heads, group, items); ++L) {
          const Place p = place(L, heads, group, items);
          if (group == XCDS) {
            const PlaceOfEight e = place_of_eight(heads, items, 3);
            for (int share = 0; share < 3; ++share) {
              int got = -1;
              const Place same = e.of(L + share * e.per_share, got);
              if (got != share || same.head != p.head || same.item != p.item) return bad("eight", heads, items, L);
            }
          }
          if (p.item >= items) continue;
          if (p.head < 0 || p.head >= heads || p.item < 0 || seen[p.head * items + p.item]++) return bad("group", heads, group, items);
          of_xcd[L % XCDS][p.head] = 1;
        }
        for (int s : seen) if (s != 1) return bad("not taken", heads, group, items);
        if (placed(heads, group, items) % XCDS != 0) return bad("length", heads, group, items);
        for (auto& x : of_xcd) {
          int n = 0;
          for (int h : x) n += h;
          if (n > heads / XCDS + 2) return bad("heads of an XCD", heads, group, items);
        }
      }
  // (the groups that the L2 holds: every item once, an XCD on as few heads as at once, the items of a group in ascending order)
  for (int heads = 1; heads <= 100; ++heads)
    for (int D : {64, 128, 256})
      for (int items : {1, 3, 8, 9, 16, 47, 64, 128, 274}) {
        const Groups g = groups_of_heads(heads, 64 * items, D);
        const PlaceOfEight e = place_of_eight(heads, items, 2, g);
        if (g.group % XCDS != 0 || g.rest != heads % XCDS || (heads - XCDS * g.whole - g.rest) % g.group != 0) return bad("groups", heads, items, D);
        for (int share = 0; share < 2; ++share) {
          std::vector<int> seen(heads * items);
          std::vector<std::vector<int>> last(XCDS, std::vector<int>(heads, -1));
          for (int L = 0; L < e.per_share; ++L) {
            int got = -1;
            const Place p = e.of(L + share * e.per_share, got);
            if (got != share) return bad("share", heads, items, D);
            if (p.item >= items) continue;
            if (p.head < 0 || p.head >= heads || p.item < 0 || seen[p.head * items + p.item]++) return bad("of a group", heads, items, D);
            if (last[L % XCDS][p.head] >= p.item) return bad("order", heads, items, D);
            last[L % XCDS][p.head] = p.item;
          }
          for (int n : seen) if (n != 1) return bad("not of a group", heads, items, D);
          if (e.per_share % XCDS != 0) return bad("ids", heads, items, D);
          for (auto& x : last) {
            int n = 0;
            for (int i : x) n += i >= 0;
            if (n > heads / XCDS + 2) return bad("heads on an XCD", heads, items, D);
          }
        }
      }
  for (unsigned d : {1u, 2u, 3u, 5u, 6u, 7u, 8u, 24u, 513u, 2192u, 65535u, 1u << 20})
    for (uint64_t most : {10ull, 1000ull, 65535ull, 1ull << 20, 1ull << 31}) {
      const Divisor v = divisor(d, most);
      const uint64_t at[] = {0, 1, d - 1, d, d + 1, most / 2, most - 1, most, most / d * d, most / d * d - 1};
      for (uint64_t n : at) if (n <= most && v.of((unsigned)n) != (unsigned)n / d) return bad("division", (int)d, (int)n, (int)most);
      for (uint64_t n = 0; n <= most && n < 100000; ++n) if (v.of((unsigned)n) != (unsigned)n / d) return bad("division", (int)d, (int)n, (int)most);
    }
  for (int heads = 1; heads <= 600; ++heads)
    for (int slots : {256, 512, 2048, 250})
      for (int cap : {1, 3, 100, 100000})
        for (int first : {0, 256, 250}) {
          int W = slots / heads < cap ? slots / heads : cap;
          if (W < 1) W = 1;
          const int fast = first < W * heads ? first : W * heads, quot = fast / heads, rest = fast % heads;
          std::vector<int> seen(heads * W);
          for (int L = 0; L < W * heads; ++L) {
            const Place p = place_range(L, heads, W, fast, quot, rest);
            if (p.head < 0 || p.head >= heads || p.item < 0 || p.item >= W || seen[p.head * W + p.item]++) return bad("range", heads, W, first);
            const int mine = quot + (p.head < rest ? 1 : 0);
            if ((L < fast) != (p.item < mine)) return bad("fast", heads, W, first);
          }
          for (int s : seen) if (s != 1) return bad("range not taken", heads, W, first);
        }
  std::puts("ok");
  return 0;
}
