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
