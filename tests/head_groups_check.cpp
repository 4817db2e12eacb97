// Checks how many heads go out at once (csrc/place.h, groups_of_heads): what the L2 does not hold is not asked for at once but by one or two
// heads beyond a multiple of 8, and each (head, item) is one workgroup's.
#include <cstdio>
#include <initializer_list>
#include <vector>
#include "place.h"
using namespace bsattn;

int main() {
  const int L2 = 4 << 20;
  int behind = 0, with = 0;
  for (int heads = 1; heads <= 72; ++heads)
    for (int D : {64, 128, 256})
      for (int items : {1, 8, 15, 40, 47, 64, 94, 128, 150, 320}) {
        const long long bytes = 4ll * 64 * items * D;
        const Groups g = groups_of_heads(heads, 64 * items, D);
        const int per_xcd = g.group / XCDS, at_once = per_xcd > g.whole + 1 || g.rest == 0 || g.whole == 0 ? per_xcd : g.whole + 1;
        const int tenths = heads / XCDS > 1 || g.rest == 0 ? 16 : 14;      // of the L2
        const bool held = at_once == 1 || 10 * at_once * bytes <= (long long)tenths * L2;
        if (!held && D > 64 && (g.rest == 0 || g.rest >= 3)) { std::printf("%d heads of %lld bytes, D = %d: %d at once\n", heads, bytes, D, at_once); return 1; }
        (heads > XCDS && g.rest > 0 && g.whole == 0 ? behind : with)++;
        const PlaceOfEight e = place_of_eight(heads, items, 1, g);
        std::vector<int> seen(heads * items);
        for (int L = 0; L < e.per_share; ++L) {
          int share = 0;
          const Place p = e.of(L, share);
          if (p.item >= items) continue;
          if (p.head < 0 || p.head >= heads || p.item < 0 || seen[p.head * items + p.item]++) { std::printf("%d heads of %d items: id %d\n", heads, items, L); return 1; }
        }
        for (int n : seen) if (n != 1) { std::printf("%d heads of %d items: one not taken\n", heads, items); return 1; }
      }
  if (behind == 0 || with == 0) { std::printf("%d behind, %d not\n", behind, with); return 1; }
  std::printf("%d behind, %d not\nok\n", behind, with);
  return 0;
}
