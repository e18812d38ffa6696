// Where an id goes in the visited filter of the sorted-set search (device_core.h, visit_lossy): `sets` sets of four 16-bit
// tags, set and tag together naming the id.  Any number of sets will do, so that the filter takes the LDS that the wavefronts
// at work leave (engine.h, fit_filter) and not the power of two below: it is read for every link of a search, so a place is
// two instructions at the vector unit's full rate, as a mask and a shift were.
//
// The id times an odd number, modulo 2^24, is another 24-bit number for every id (place), and neighbouring ids lie far apart.  The
// sets cut the 24-bit numbers into stretches of equal length (within one), less than 2^16 long: a number's last 16 bits tell
// it from all others of its stretch, and there are 16 bits that no number of the stretch ends in, which stand for "empty"
// there.  More than 2^24 elements: the same with as many bits as it takes (the product in 32 bits: a quarter of the rate).
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

constexpr uint32_t kFilterSpread = 0x9E3779u;  // (2^24 over the golden ratio)
constexpr int kMostFilterSets = 16384;

struct FilterShape {
  uint32_t code = 0;  // sets << 8 (bits 8 to 23), bits beyond 24 that ids have (from bit 24 on); 0 = no filter
  CUHNSW_HOST_DEVICE int sets() const { return (int)((code & 0xFFFFFFu) >> 8); }
  CUHNSW_HOST_DEVICE int more_bits() const { return (int)(code >> 24); }
  CUHNSW_HOST_DEVICE uint32_t bytes() const { return 8u * (uint32_t)((sets() + 1) & ~1); }
};

// The shape with that many sets, or more where ids of n elements need them; none where they need too many.
inline FilterShape filter_shape(int sets, int n) {
  int more = 0;
  while (((uint32_t)n >> more) > (1u << 24)) ++more;
  const int least = (256 << more) + (4 << more);  // (a stretch of 65 536 is one too long)
  sets = sets < least ? least : sets;
  FilterShape f;
  if (sets <= kMostFilterSets) f.code = (uint32_t)sets << 8 | (uint32_t)more << 24;
  return f;
}

// the id's number, of which the tag is the last 16 bits
template <bool WIDE>
CUHNSW_HOST_DEVICE inline uint32_t filter_place(uint32_t id) {
  return WIDE ? id * kFilterSpread : (id & 0xFFFFFFu) * kFilterSpread;  // (24 by 24 bits)
}
template <bool WIDE>
CUHNSW_HOST_DEVICE inline uint32_t filter_set(FilterShape f, uint32_t place) {
  if (WIDE) place >>= f.more_bits();
#if defined(__HIP_DEVICE_COMPILE__)
  uint32_t set;
  asm("v_mul_hi_u32_u24 %0, %1, %2" : "=v"(set) : "s"(f.code), "v"(place));  // (looks at 24 bits of either)
  return set;
#else
  return (uint32_t)(((uint64_t)(f.code & 0xFFFFFFu) * (place & 0xFFFFFFu)) >> 32);
#endif
}
// 16 bits that no number of the set ends in: those of the middle of its stretch with the highest of them turned (a stretch is
// at most 64 528 long whatever more_bits is, as the fewest sets grow with it, and the middle is found within a few)
CUHNSW_HOST_DEVICE inline uint32_t filter_empty_tag(FilterShape f, uint32_t set) {
  const float stretch = (float)(1u << 24) / (float)f.sets() * (float)(1 << f.more_bits());
  return ((uint32_t)(((float)set + 0.5f) * stretch) ^ 0x8000u) & 0xFFFFu;
}

}  // namespace cuhnsw_amd
