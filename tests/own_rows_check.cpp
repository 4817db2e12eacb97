// Host-side check of which heads go a row block to a workgroup and how (csrc/own_rows.h): their row blocks are each taken once, in parts that
// tile them, no workgroup walks a list much longer than the mean, and heads whose lists are of like length are among them.
#include <algorithm>
#include <cstdio>
#include <numeric>
#include <random>
#include <vector>
#include "own_rows.h"
using namespace bsattn;

struct Launch { int heads, nb; };
static const int WORKGROUPS = 512, FIRSTS = 256;      // of 256 compute units

struct Head {
  int nb, W, firsts, T;
  std::vector<int> len;
  Head(Launch l, std::vector<int> lens) : nb(l.nb), W(WORKGROUPS / l.heads), firsts(FIRSTS / l.heads), T(std::accumulate(lens.begin(), lens.end(), 0)), len(std::move(lens)) {}
  bool taken() const {
    const OwnLines lines = own_lines(nb, W, firsts);
    const int middle = std::accumulate(len.begin(), len.begin() + nb / 2, 0);
    if (T == 0 || !own_rows_by_tiles(lines, T, nb) || !own_rows_by_middle(T, middle)) return false;
    int longest = 0, uneven = 0;
    for (int l : len) { longest = std::max(longest, l); uneven += l > own_rows_even(lines, T); }
    return longest <= own_rows_longest(lines, T) && 4 * uneven <= nb;
  }
  int longest_piece(bool& sound) const {      // of all workgroups' (each row block once and whole, or in parts that tile it)
    std::vector<int> seen(nb);
    int longest = 0;
    for (int wg = 0; wg < W; ++wg) {
      const OwnItem it = own_item(wg, nb, W, firsts);
      if (it.row >= nb) continue;
      const int l = len[it.row], parts = own_parts(l, it.most);
      if (it.part >= parts || l == 0) continue;
      const int a = l * it.part / parts, b = l * (it.part + 1) / parts;
      sound = sound && a == seen[it.row] && (parts == 1 || b - a >= OWN_PART_TILES) && wg - it.part >= 0 && wg - it.part + parts <= W;
      seen[it.row] = b;
      longest = std::max(longest, b - a);
    }
    for (int r = 0; r < nb; ++r) sound = sound && seen[r] == len[r];
    return longest;
  }
};

int main() {
  std::mt19937 g(1);
  auto random = [&](int nb, double keep) {
    std::vector<int> len(nb);
    for (int& l : len) l = std::max(1, (int)std::binomial_distribution<int>(nb, keep)(g));
    return len;
  };
  // every row block once, whatever the lists
  int heads = 0;
  for (int it = 0; it < 20000; ++it) {
    const Launch l = {1 + (int)(g() % 5), 1 + (int)(g() % 512)};
    const int kind = (int)(g() % 4);
    std::vector<int> len = random(l.nb, 0.002 * (1 + g() % 200));
    if (kind == 1) for (int i = 0; i < 3; ++i) len[g() % l.nb] = l.nb;
    if (kind == 2) for (int& x : len) if (g() % 3 == 0) x = 0;
    if (kind == 3) for (int r = 0; r < l.nb; ++r) len[r] = len[r] * (l.nb - r) / l.nb;
    const Head h(l, len);
    if (!h.taken()) continue;
    ++heads;
    bool sound = true;
    const int longest = h.longest_piece(sound);
    if (!sound) { printf("%d heads of %d row blocks: not every row block once\n", l.heads, l.nb); return 1; }
    if (longest > 20 + 1.5 * h.T / h.nb) { printf("%d heads of %d row blocks, mean %.1f: a workgroup walks %d tiles\n", l.heads, l.nb, (double)h.T / h.nb, longest); return 1; }
  }
  if (heads < 1000) { printf("only %d heads taken\n", heads); return 1; }
  // one or four row blocks kept whole in a sparse mask, a few lists of all row blocks and none beside them, much longer and short ones in turn: the ranges'
  for (const auto& [l, keep] : std::vector<std::pair<Launch, double>>{{{1, 274}, 0.1}, {{1, 188}, 0.1}, {{1, 256}, 0.03}, {{2, 141}, 0.1}, {{1, 500}, 0.05}, {{3, 157}, 0.1}, {{2, 251}, 0.05}})
    for (int whole : {1, 4}) {
      std::vector<int> len = random(l.nb, keep), one = len, few(l.nb, 0), every(l.nb, 1), turns(l.nb, 2);      // (of 56 tiles: 29 on the average)
      for (int r = 0; r < whole; ++r) len[r] = one[l.nb / 2 + r] = few[r * 7] = every[l.nb / 3] = l.nb;
      for (int r = 0; r < l.nb; r += 2) turns[r] = 56;
      for (const auto& x : {len, one, few, every, turns})
        if (Head(l, x).taken()) { printf("%d heads of %d row blocks, keep %.2f, %d whole: taken\n", l.heads, l.nb, keep, whole); return 1; }
    }
  // uniform masks: taken (a list that random masks hardly ever have is what the line leaves)
  int lost = 0, all = 0;
  for (const auto& [l, keep] : std::vector<std::pair<Launch, double>>{{{1, 274}, 0.1}, {{1, 157}, 0.02}, {{1, 157}, 0.1}, {{1, 256}, 0.1}, {{1, 500}, 0.05}, {{1, 500}, 0.1}, {{3, 157}, 0.1}, {{3, 157}, 0.3}, {{2, 251}, 0.1}, {{2, 141}, 0.2}})
    for (int it = 0; it < 100; ++it, ++all) lost += !Head(l, random(l.nb, keep)).taken();
  if (100 * lost > all) { printf("%d of %d uniform masks left to the ranges\n", lost, all); return 1; }
  printf("%d heads, %d of %d uniform masks left to the ranges\nok\n", heads, lost, all);
  return 0;
}
