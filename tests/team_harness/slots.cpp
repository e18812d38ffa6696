// A team's slot between two levels of a build (device_core.h, team_close and team_help; cuhnsw_amd/csrc/team_slots.h), on the host: one
// wavefront that searches and three that help, one step -- one access to LDS -- at a time, in every order there is.  Prints in how
// many states two helpers write the one list, and in how many a list of the level before is there on the next.
// slots RULE: 0 the header's, 1 every slot is stored to when a level ends.
#include <array>
#include <cstdio>
#include <cstdlib>
#include <set>
#include <vector>

#include "team_slots.h"

using namespace cuhnsw_amd;

constexpr int kHelpers = 3, kClaims = 2;
// word, level (odd: closed), search's step, word it read, then per helper: step, level it works for, claims made
typedef std::array<uint32_t, 4 + 3 * kHelpers> State;

int main(int argc, char** argv) {
  const bool every = argc > 1 && atoi(argv[1]) == 1;
  std::set<State> seen;
  std::vector<State> open;
  long long clashes = 0, stale = 0;
  auto go = [&](const State& s) {
    if (seen.insert(s).second) open.push_back(s);
  };
  State first{};
  first[0] = kNobody;
  go(first);
  while (!open.empty()) {
    const State s = open.back();
    open.pop_back();
    int writing = 0;
    for (int h = 0; h < kHelpers; ++h) writing += s[4 + 3 * h] == 3 ? 1 : 0;
    clashes += writing > 1 ? 1 : 0;
    stale += s[2] == 4 && slot_holds_list(s[0]) && ((s[0] >> 8) & 0xFFu) != s[1] ? 1 : 0;
    State n = s;
    switch (s[2]) {  // the search
      case 0: n[1] |= 1u; n[2] = 1; go(n); break;
      case 1: n[3] = s[0]; n[2] = 2; go(n); break;
      case 2:
        if (slot_being_made(s[3])) n[2] = 1;
        else {
          if (every || slot_holds_list(s[3])) n[0] = kNobody;
          n[2] = 3;
        }
        go(n);
        break;
      case 3: n[1] = 2; n[2] = 4; go(n); break;
    }
    for (int h = 0; h < kHelpers; ++h) {
      const int at = 4 + 3 * h;
      const uint32_t id = (uint32_t)h + 1u + (s[at + 1] << 8);  // (the level it was made for, to be recognised)
      n = s;
      switch (s[at]) {
        case 0: n[at + 1] = s[1]; n[at] = (s[1] & 1u) || s[at + 2] == kClaims ? 0 : 1; go(n); break;
        case 1:  // compare-and-swap
          if (s[0] == kNobody) { n[0] = id | kSlotMaking; n[at] = 2; n[at + 2] += 1; }
          else n[at] = 0;
          go(n);
          break;
        case 2: n[at] = s[1] == s[at + 1] ? 3 : 4; go(n); break;
        case 3: n[0] = id; n[at] = 0; go(n); break;
        case 4: n[0] = kNobody; n[at] = 0; go(n); break;
      }
    }
  }
  printf("%zu %lld %lld\n", seen.size(), clashes, stale);
  return 0;
}
