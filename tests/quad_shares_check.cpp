// Host-side check of how the forward at D = 128 shares the lists of row blocks (csrc/quad_shares.h): a list has between one and `most`
// shares, none shorter than `least`, which tile it as the kernel cuts it; lists of like length in front of the last round stay whole,
// and the long ones of a head whose lists grow are cut.
#include <cstdio>
#include <random>
#include "quad_shares.h"
using namespace bsattn;

int main() {
  std::mt19937 g(1);
  for (int it = 0; it < 400000; ++it) {
    const int nb = SHARE_MIN_BLOCKS + (int)(g() % 500), len = (int)(g() % (nb + 1)), most = 1 + (int)(g() % 4), least = (const int[]){4, 8, 24}[g() % 3];
    const int mid = (int)(g() % (SHARE_SAMPLE * nb + 1)), end = (int)(g() % (SHARE_SAMPLE * nb + 1));
    const int rows = nb * (1 + (int)(g() % 64)), slots = g() % 2 ? 256 : 512, left = rows % slots;
    const int tail = g() % 2 ? 1 : left > 0 ? slots / left : 1, load = (int)((long long)rows * 4096 / slots);
    const int n = quad_shares(len, mid, end, tail, load, most, least);
    if (n < 1 || n > most || (n > 1 && len / n < least)) { printf("%d shares of %d tiles, at most %d\n", n, len, most); return 1; }
    int at = 0;
    for (int c = 0; c < n; ++c) {
      const int t0 = (int)((long long)len * c / n), t1 = (int)((long long)len * (c + 1) / n);
      if (t0 != at || t1 < t0) { printf("the shares do not tile the list\n"); return 1; }
      at = t1;
    }
    if (at != len) { printf("the shares do not tile the list\n"); return 1; }
    const int like = len * SHARE_SAMPLE;
    if (quad_shares(len, like, like, 1, load, most, least) != 1) { printf("a list among like ones is cut\n"); return 1; }
  }
  // dense block-causal, 2 heads of 94 row blocks on 256 places: the longest lists get two shares, those below the mean stay whole
  const int mid = SHARE_SAMPLE * 47, end = 91 + 92 + 93 + 94, load = 188 * 4096 / 256;
  if (quad_shares(94, mid, end, 1, load, 2, 8) != 2 || quad_shares(40, mid, end, 1, load, 2, 8) != 1) { printf("block-causal\n"); return 1; }
  printf("ok\n");
  return 0;
}
