// Host-side check of how the forward kernel cuts long row blocks (csrc/row_parts.h): for heads of many kinds the parts
// tile every long row block, none is empty, and those of row blocks that are cut fit the W slots of a head.
#include <cstdio>
#include <cstdint>
#include <random>
#include <vector>
#include "row_parts.h"
using namespace bsattn;

int main() {
  std::mt19937 g(1);
  int cut = 0, fullest = 0;
  for (int it = 0; it < 40000; ++it) {
    const int nb = (const int[]){1, 2, 26, 30, 64, 65, 128, 278, 500, 2048}[g() % 10];
    const int W = (const int[]){8, 9, 10, 21, 42, 85, 170, 682}[g() % 8], kind = (int)(g() % 5), share = (int)(g() % 45);
    std::vector<int> len(nb);
    for (int r = 0; r < nb; ++r)
      len[r] = kind == 0 ? (int)(g() % (nb + 1)) : kind == 1 ? (r < 4 ? nb : nb / 20) : kind == 2 ? ((int)(g() % 100) < share ? nb : (int)(g() % 3))
             : kind == 3 ? ((int)(g() % 100) < share ? 25 + (int)(g() % (nb > 25 ? nb - 24 : 1)) : 0) : (r == nb / 2 ? nb : 0);
    int64_t T = 0;
    for (int l : len) T += l;
    int tiles = 0, rows = 0;
    for (int l : len) if (is_long_row(l, (int)T, nb)) { tiles += l; ++rows; }
    if (rows == 0) continue;
    const int x = long_part_tiles(tiles, rows, W, (int)T / nb);
    int slots = 0;
    for (int l : len) {
      if (!is_long_row(l, (int)T, nb)) continue;
      const int n = parts_of_row(l, x);
      if (n < 1 || part_begin(l, n, 0) != 0 || part_begin(l, n, n) != l) { printf("parts do not tile a row block\n"); return 1; }
      for (int i = 0; i < n; ++i) {
        const int t = part_begin(l, n, i + 1) - part_begin(l, n, i);
        if (t < 1 || t > x) { printf("a part of %d tiles (%d)\n", t, x); return 1; }
      }
      if (n > 1) slots += n;
    }
    if (slots > W) { printf("%d parts for %d slots: nb %d, %d long row blocks of %d tiles\n", slots, W, nb, rows, tiles); return 1; }
    cut += slots > 0;
    if (slots == W) ++fullest;
  }
  printf("%d heads with row blocks that are cut, %d with every slot used\nok\n", cut, fullest);
  return cut > 1000 ? 0 : 1;
}
