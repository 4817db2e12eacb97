// Checks the ids of a launch of whole row blocks (csrc/place.h) on the host: every row block and every workgroup for parts of long ones is taken
// once and no head behind the last one is named, whether or not the row blocks are more than are resident at once.
#include <cstdio>
#include <vector>
#include "place.h"
using namespace bsattn;

int main() {
  for (int heads = 1; heads <= 40; ++heads)
    for (int group = 8; group <= 48; group += 8)
      for (int nb : {1, 7, 8, 33, 64, 130})
        for (int W : {0, 1, 8, 51})
          for (int resident : {8, 256, 2048}) {
            const int first = first_ids_of_rows(resident, heads, group, nb), ids = placed(heads, group, nb) + placed(heads, group, W);
            std::vector<int> seen(heads * (nb + W));
            int taken = 0;
            for (int id = 0; id < ids; ++id) {
              const PlaceOfRows at = place_rows(id, heads, group, nb, W, first);
              if (at.p.item >= at.per) continue;
              const int item = at.p.item + (at.extra ? nb : 0);
              if (at.p.head < 0 || at.p.head >= heads || at.per != (at.extra ? W : nb) || at.p.item < 0 || seen[at.p.head * (nb + W) + item]++ || (at.extra && id < first)) {
                std::printf("%d heads of %d row blocks, group %d, %d workgroups for parts, %d resident: id %d takes head %d item %d\n", heads, nb, group, W, resident, id, at.p.head, item);
                return 1;
              }
              ++taken;
            }
            if (taken != (int)seen.size()) { std::printf("%d heads of %d row blocks, group %d, %d workgroups for parts: %d taken\n", heads, nb, group, W, taken); return 1; }
          }
  std::printf("\nok\n");
  return 0;
}
