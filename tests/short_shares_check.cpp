// Checks into which shares fwd_short_kernel cuts a list (csrc/quad_shares.h): against the quotients themselves, for all lengths that it takes.
#include <cstdio>
#include <initializer_list>
#include "quad_shares.h"
using namespace bsattn;

int main() {
  for (int len = 0; len <= 1024; ++len)
    for (int split = 2; split <= 4; ++split)
      for (int shift : {0, 3}) {
        const int tiles = 1 << shift, shares = short_shares(len, split, shift);
        const int want = len >= split * tiles ? split : len < 2 * tiles ? 1 : len / tiles;
        if (shares != want) { std::printf("%d shares of %d tiles, %d at most of %d: %d\n", shares, len, split, tiles, want); return 1; }
        for (int c = 0; c <= shares; ++c)
          if (short_share_begins(len, c, shares) != len * c / shares) { std::printf("share %d of %d of %d tiles\n", c, shares, len); return 1; }
      }
  std::printf("\nok\n");
  return 0;
}
