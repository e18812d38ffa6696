// What the word of a slot says in which the wavefronts of a team keep a list of evaluated nodes (device_core.h, team_help):
//   kNobody           free
//   id | kSlotMaking  a helper makes the list of node id; only that helper changes the word
//   an id below 2^28  its list is there, in bits 28 to 30 how many eights of nodes it has (0: eight); only the search changes the word
//   all ones          no slot
// A helper takes a free slot by compare-and-swap, so nobody else stores to one, not even kNobody: a helper that has taken it in the
// meantime and sees that it may not begin would give it back after the next one had taken it, and two would write one list.
#pragma once
#include <stdint.h>

#ifndef CUHNSW_HOST_DEVICE
#ifndef __HIPCC__
#define CUHNSW_HOST_DEVICE
#else
#define CUHNSW_HOST_DEVICE __host__ __device__
#endif
#endif

namespace cuhnsw_amd {

constexpr uint32_t kNobody = 0x7FFFFFFFu, kSlotMaking = 0x80000000u, kNoSlot = 0xFFFFFFFFu, kTeamId = 0x0FFFFFFFu;

CUHNSW_HOST_DEVICE inline bool slot_being_made(uint32_t word) { return (word & kSlotMaking) != 0u && word != kNoSlot; }
CUHNSW_HOST_DEVICE inline bool slot_holds_list(uint32_t word) { return (word & kSlotMaking) == 0u && word != kNobody; }
// the word of a list of n nodes (up to 64: a list that stayed out would have its candidate taken up again by the next helper, over and
// over), whose it is, and its eights of nodes (a list without any counts as one)
CUHNSW_HOST_DEVICE inline uint32_t slot_word(uint32_t id, int n) { return id | (uint32_t)((n > 0 ? (n + 7) >> 3 : 1) & 7) << 28; }
CUHNSW_HOST_DEVICE inline bool slot_is_of(uint32_t word, uint32_t id) { return (word & (kTeamId | kSlotMaking)) == id; }
CUHNSW_HOST_DEVICE inline int slot_eights(uint32_t word) { return (word >> 28) != 0u ? (int)(word >> 28) : 8; }

}  // namespace cuhnsw_amd
