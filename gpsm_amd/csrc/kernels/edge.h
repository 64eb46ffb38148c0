// Edge-membership test of the join kernels.
#pragma once
#include "wave.h"

namespace gpsm {

// Edge {a, b}: one bit of a hub's adjacency bitmap when either end is a hub,
// else a binary search in the entries of b towards the label of a (key a_lo).
template <bool BYTES>
__device__ __forceinline__ bool has_edge(const Pieces& pieces, const uint32_t* __restrict__ col,
                                         const uint32_t* __restrict__ hub_of, const uint32_t* __restrict__ hub_bits,
                                         uint32_t W, uint32_t a, uint32_t a_lo, uint32_t b,
                                         unsigned long long& bytes) {
  const uint32_t ha = hub_of[a], hb = hub_of[b];
  if (BYTES) bytes += 8;
  if (ha != ~0u || hb != ~0u) {
    if (BYTES) bytes += 4;
    return ha != ~0u ? bit_of(hub_bits + (size_t)ha * W, b) != 0 : bit_of(hub_bits + (size_t)hb * W, a) != 0;
  }
  uint32_t lo, n;
  piece(pieces, b, a_lo, lo, n);
  if (BYTES) bytes += 8;
  if (n == 0) return false;
  // branch-free search for the last entry <= a: ceil(log2 n) halvings, one
  // comparison at the end (no early exit, so no per-step exec-mask updates)
  if (BYTES) bytes += 4ull * (1 + (n > 1 ? 32 - __clz(n - 1) : 0));  // ceil(log2 n) probes + the last read
  const uint32_t* p = col + lo;
  while (n > 1) {
    const uint32_t half = n >> 1;
    p = p[half] <= a ? p + half : p;
    n -= half;
  }
  return *p == a;
}

}  // namespace gpsm
