// Stable LSD radix sort passes over 64-bit keys, 8 bits at a time, with or
// without a 32-bit value per key (the device CSR build, the tuple sort).
//
// One pass: each workgroup counts the digits of its tile of
// RADIX_TILE keys (LDS histogram), an exclusive scan of the counts in
// digit-major order gives every (digit, tile) its output start, and each
// workgroup scatters its tile stably: 256 keys at a time, in index order,
// a key's place among the equal digits of its wave comes from eight
// ballots (one per digit bit), the waves before it from per-wave digit
// counts in LDS, the chunks before it from a running count per digit.
#include <algorithm>

#include "launch.h"
#include "wave.h"

namespace gpsm {

namespace {

constexpr uint32_t RADIX_ITEMS = 16;                  // keys per thread and tile
constexpr uint32_t RADIX_TILE = 256 * RADIX_ITEMS;     // keys per workgroup

__global__ void __launch_bounds__(256) radix_hist_kernel(const unsigned long long* __restrict__ keys, uint64_t n,
                                                         uint32_t shift, uint32_t ntiles,
                                                         uint32_t* __restrict__ hist) {
  __shared__ uint32_t cnt[256];
  cnt[threadIdx.x] = 0;
  __syncthreads();
  const uint64_t base = (uint64_t)blockIdx.x * RADIX_TILE;
  for (uint32_t j = 0; j < RADIX_ITEMS; ++j) {
    const uint64_t i = base + (uint64_t)j * 256 + threadIdx.x;
    if (i < n) atomicAdd(&cnt[(uint32_t)(keys[i] >> shift) & 255u], 1u);
  }
  __syncthreads();
  hist[(size_t)threadIdx.x * ntiles + blockIdx.x] = cnt[threadIdx.x];  // digit-major
}

// PAYLOAD: each key moves with its 32-bit value.
template <bool PAYLOAD>
__global__ void __launch_bounds__(256) radix_scatter_kernel(const unsigned long long* __restrict__ in,
                                                            unsigned long long* __restrict__ out,
                                                            const uint32_t* __restrict__ vin,
                                                            uint32_t* __restrict__ vout, uint64_t n,
                                                            uint32_t shift, uint32_t ntiles,
                                                            const uint32_t* __restrict__ start) {
  __shared__ uint32_t run[256];     // output position of the next key of each digit
  __shared__ uint32_t wc[4][256];   // this chunk's keys per (wave, digit)
  const uint32_t lane = lane_id(), w = threadIdx.x / WAVE;
  const unsigned long long below = lane ? (~0ULL >> (WAVE - lane)) : 0ULL;
  run[threadIdx.x] = start[(size_t)threadIdx.x * ntiles + blockIdx.x];
  const uint64_t base = (uint64_t)blockIdx.x * RADIX_TILE;
  for (uint32_t j = 0; j < RADIX_ITEMS; ++j) {
    const uint64_t i = base + (uint64_t)j * 256 + threadIdx.x;
    const bool valid = i < n;
    const unsigned long long key = valid ? in[i] : 0ULL;
    const uint32_t d = (uint32_t)(key >> shift) & 255u;
    // the lanes of this wave holding the same digit
    unsigned long long same = __ballot(valid);
#pragma unroll
    for (uint32_t b = 0; b < 8; ++b) {
      const unsigned long long ones = __ballot(valid && ((d >> b) & 1u));
      same &= ((d >> b) & 1u) ? ones : ~ones;
    }
    const uint32_t rank = (uint32_t)__popcll(same & below);
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) wc[w][lane + 64 * k] = 0;
    if (valid && rank == 0) wc[w][d] = (uint32_t)__popcll(same);
    __syncthreads();  // also publishes run (first chunk) and the previous chunk's counts
    if (valid) {
      uint32_t pos = run[d] + rank;
      for (uint32_t x = 0; x < w; ++x) pos += wc[x][d];
      out[pos] = key;
      if constexpr (PAYLOAD) vout[pos] = vin[i];
    }
    __syncthreads();
    run[threadIdx.x] += wc[0][threadIdx.x] + wc[1][threadIdx.x] + wc[2][threadIdx.x] + wc[3][threadIdx.x];
    __syncthreads();
  }
}

}  // namespace

uint64_t radix_hist_words(uint64_t n) {
  return 256ull * std::max<uint64_t>(1, (n + RADIX_TILE - 1) / RADIX_TILE);
}

void launch_radix_pass(const unsigned long long* in, unsigned long long* out, const uint32_t* vin, uint32_t* vout,
                       uint64_t n, uint32_t shift, uint32_t* hist, uint32_t* hstart, uint32_t* scratch,
                       uint64_t scratch_words, hipStream_t s) {
  if (!n) return;
  const uint32_t ntiles = (uint32_t)((n + RADIX_TILE - 1) / RADIX_TILE);
  hipLaunchKernelGGL(radix_hist_kernel, dim3(ntiles), dim3(256), 0, s, in, n, shift, ntiles, hist);
  launch_exclusive_scan(hist, hstart, radix_hist_words(n), nullptr, scratch, scratch_words, s);
  if (vin)
    hipLaunchKernelGGL(radix_scatter_kernel<true>, dim3(ntiles), dim3(256), 0, s, in, out, vin, vout, n, shift, ntiles,
                       hstart);
  else
    hipLaunchKernelGGL(radix_scatter_kernel<false>, dim3(ntiles), dim3(256), 0, s, in, out, vin, vout, n, shift,
                       ntiles, hstart);
}

}  // namespace gpsm
