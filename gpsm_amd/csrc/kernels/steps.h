// Index loops of a wave over ranges of 32-bit indices.
#pragma once
#include <cstdint>

namespace gpsm {

// Calls f(x) for x = lo, lo + 64, ... below hi.  The index has 64 bits: a
// 32-bit one wraps where hi is within a step of 2^32 (an adjacency may hold
// 2^32 - 1 entries) and the loop would not end.
template <typename F>
constexpr void for_steps(uint64_t lo, uint64_t hi, F f) {
  for (uint64_t x = lo; x < hi; x += 64) f(x);
}

}  // namespace gpsm
