// qcu_hash.h -- content hash of an external gauge field, entry by entry.
#pragma once
#include "qcu_common.h"

namespace qcu {

// The bit patterns (a, b) of entry k, mixed with its position.  a goes through a
// product of its own before b enters: in a sum of multiples of both the top bits
// (the signs) of a and b cancel, and a negated entry would hash like the old one.
// Adding b, the shifts and the odd factors are one to one, so entries that differ
// in one part always hash differently.
QCU_HD unsigned long long hash_mix(unsigned long long a, unsigned long long b, unsigned long long k) {
  unsigned long long x = a + k * 0x9E3779B97F4A7C15ull;
  x ^= x >> 32;
  x *= 0xC2B2AE3D27D4EB4Full;
  x ^= x >> 29;
  x += b;
  x ^= x >> 30;
  x *= 0xBF58476D1CE4E5B9ull;
  x ^= x >> 32;
  x *= 0x94D049BB133111EBull;
  return x ^ (x >> 29);
}

}  // namespace qcu
