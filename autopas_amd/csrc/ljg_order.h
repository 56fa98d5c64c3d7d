// ljg_order.h -- the order of a tower's particles, shared by the sorts and by the host's tests (no HIP needed).
#pragma once

#include <cstdint>

#ifdef __HIPCC__
#define LJG_HD __host__ __device__
#else
#define LJG_HD
#endif

namespace ljg {

// Particle a before particle b: by z, then id, then old slot.  Total for every input: a z that is not a number comes
// after all numbers, and equal ids fall back to the slots, which are distinct.  The sorts that rank (a place is the
// number of particles before) need that: two particles that are each not before the other would share a place and
// leave another place of the tower unwritten, which the permutation then reads as an old slot.
// (Without branches: it stands in every stage of the sorting networks.)
LJG_HD inline bool tower_before(double za, int64_t ia, int32_t sa, double zb, int64_t ib, int32_t sb) {
  const bool na = za != za, nb = zb != zb;
  const bool same = (za == zb) | (na & nb);
  return (za < zb) | (nb & !na) | (same & ((ia < ib) | ((ia == ib) & (sa < sb))));
}

// The FP32 word that the register sorts compare first: monotone in that order (rounding is, and what is not a
// number goes to the end), so unequal words decide and equal ones are decided by tower_before.
LJG_HD inline float tower_key32(double z) { return z != z ? __builtin_inff() : (float)z; }

}  // namespace ljg
