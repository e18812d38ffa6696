// Every id's place in a visited filter (cuhnsw_amd/csrc/visited_filter.h), on the host: filter_places SETS N [STEP] walks the
// ids 0, STEP, 2 STEP .. of N and prints how many sets the filter has, how many ids fall outside of it, how many share set and
// tag with another, and how many have their set's empty tag.
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "visited_filter.h"

using namespace cuhnsw_amd;

int main(int argc, char** argv) {
  const int n = argc > 2 ? atoi(argv[2]) : 0, step = argc > 3 ? atoi(argv[3]) : 1;
  const FilterShape f = filter_shape(argc > 1 ? atoi(argv[1]) : 0, n);
  const size_t sets = (size_t)f.sets();
  std::vector<bool> taken(sets << 16);
  std::vector<uint32_t> empty(sets);
  for (size_t s = 0; s < sets; ++s) empty[s] = filter_empty_tag(f, (uint32_t)s);
  long long outside = 0, shared = 0, as_empty = 0;
  for (long long i = 0; i < n && sets > 0; i += step) {
    const uint32_t id = (uint32_t)i;
    const uint32_t place = f.more_bits() != 0 ? filter_place<true>(id) : filter_place<false>(id);
    const uint32_t set = f.more_bits() != 0 ? filter_set<true>(f, place) : filter_set<false>(f, place);
    if (set >= sets) {
      ++outside;
      continue;
    }
    const size_t at = ((size_t)set << 16) | (place & 0xFFFFu);
    shared += taken[at] ? 1 : 0;
    taken[at] = true;
    as_empty += (place & 0xFFFFu) == empty[set] ? 1 : 0;
  }
  printf("%zu %lld %lld %lld\n", sets, outside, shared, as_empty);
  return 0;
}
