// The word of every slot whose list has 0 to 64 nodes (cuhnsw_amd/csrc/team_slots.h), on the host, for the first and last ids: prints how
// many are not taken for a list of their node and of that node only, and how many have the wrong number of eights of nodes.
#include <cstdio>

#include "team_slots.h"

using namespace cuhnsw_amd;

int main() {
  const uint32_t ids[] = {0u, 1u, 7u, 1183513u, 0x08000000u, 0x0FFFEFFFu};  // (fewer than 2^28 - 4 096 points have a visited filter)
  int lost = 0, wrong = 0;
  for (uint32_t id : ids)
    for (int n = 0; n <= 64; ++n) {
      const uint32_t word = slot_word(id, n);
      lost += !slot_holds_list(word) || slot_being_made(word) || !slot_is_of(word, id) ? 1 : 0;
      for (uint32_t other : ids) lost += other != id && slot_is_of(word, other) ? 1 : 0;
      wrong += 8 * slot_eights(word) < n || 8 * (slot_eights(word) - 1) >= (n > 0 ? n : 1) ? 1 : 0;
    }
  printf("%d %d\n", lost, wrong);
  return 0;
}
