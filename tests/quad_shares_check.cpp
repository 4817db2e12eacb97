// Host-side check of how the forward at D = 128 and 256 shares the lists of row blocks (csrc/quad_shares.h): a list has at least one share and
// at most what its launch has room for, none shorter than `least`, which tile it as the kernel cuts it; lists of like length in front of the
// last round stay whole, and so do all in launches of more than a round; the long ones of a head whose lists grow are cut, and those of
// more than twice the mean in any head; the shares of the last round fit it, or take less time than whole lists.
#include <cstdio>
#include <random>
#include "quad_shares.h"
using namespace bsattn;

int main() {
  std::mt19937 g(1);
  for (int it = 0; it < 400000; ++it) {
    const int nb = SHARE_MIN_BLOCKS + (int)(g() % 500), len = (int)(g() % (nb + 1)), most = 1 + (int)(g() % 4), least = (const int[]){3, 4, 6, 8, 24}[g() % 5];
    const int mid = (int)(g() % (SHARE_SAMPLE * nb + 1)), end = (int)(g() % (SHARE_SAMPLE * nb + 1));
    const int rows = nb * (1 + (int)(g() % 64)), slots = g() % 2 ? 256 : 512, split = most + (int)(g() % 3), load = (int)((long long)rows * 4096 / slots);
    const TailShares last = tail_of(rows, slots, split);
    const int tail = g() % 2 || len < last.len ? 1 : last.shares, room = tail > most ? tail : most;
    if (last.from > rows || rows - last.from >= slots || last.from % slots != 0 || last.shares < 1 || last.shares > split || last.len < 0) {
      printf("last round: %d rows %d slots: from %d, %d shares of %d tiles\n", rows, slots, last.from, last.shares, last.len);
      return 1;
    }
    // an XCD takes every eighth workgroup
    const int places = slots / XCDS, lists = (rows - last.from + XCDS - 1) / XCDS;
    if (last.shares > 1 && last.shares * lists > places) {
      const int rounds = (last.shares * lists + places - 1) / places;
      if (rows >= slots || rounds >= last.shares || last.len * (last.shares - rounds) < FILL_GAIN * last.shares) { printf("the shares of %d lists do not pay\n", rows); return 1; }
    } else if (last.len != 0) { printf("%d lists of the last round stay whole\n", rows); return 1; }
    const int n = quad_shares(len, mid, end, tail, load, most, least);
    if (n < 1 || n > room || (n > 1 && len / n < least)) { printf("%d shares of %d tiles, at most %d\n", n, len, room); return 1; }
    int at = 0;
    for (int c = 0; c < n; ++c) {
      const int t0 = (int)((long long)len * c / n), t1 = (int)((long long)len * (c + 1) / n);
      if (t0 != at || t1 < t0) { printf("the shares do not tile the list\n"); return 1; }
      at = t1;
    }
    if (at != len) { printf("the shares do not tile the list\n"); return 1; }
    const int like = len * SHARE_SAMPLE;
    if (quad_shares(len, like, like, 1, load, most, least) != 1) { printf("a list among like ones is cut\n"); return 1; }
    if (load > 4096 && quad_shares(len, mid, end, 1, load, most, least) != 1) { printf("a list in front of the last round is cut\n"); return 1; }
    // a head that does not grow: cut above twice the mean and not at it
    const int mean = len / 3;
    if (load >= 1024 && load <= 4096 && most > 1 && mean >= least && 2 * mean >= 2 * least &&
        (quad_shares(2 * mean, SHARE_SAMPLE * mean, SHARE_SAMPLE * mean, 1, load, most, least) != 1 ||
         quad_shares(2 * mean + 1, SHARE_SAMPLE * mean, SHARE_SAMPLE * mean, 1, load, most, least) < 2)) { printf("twice the mean\n"); return 1; }
  }
  // dense block-causal, 2 heads of 94 row blocks on 256 places: the longest lists get two shares, those below the mean stay whole
  const int mid = SHARE_SAMPLE * 47, end = 91 + 92 + 93 + 94, load = 188 * 4096 / 256;
  if (quad_shares(94, mid, end, 1, load, 2, 8) != 2 || quad_shares(40, mid, end, 1, load, 2, 8) != 1) { printf("block-causal\n"); return 1; }
  // 512 places: three shares of 168 lists fit, of 170 they do not on every XCD; 300 lists of at least 78 tiles take two rounds of thirds
  const TailShares a = tail_of(168, 512, 3), b = tail_of(170, 512, 3), c = tail_of(300, 512, 3), d = tail_of(300, 512, 2);
  if (a.shares != 3 || a.len != 0 || b.shares != 2 || c.shares != 3 || c.len != 78 || d.shares != 1) { printf("places of an XCD\n"); return 1; }
  printf("ok\n");
  return 0;
}
