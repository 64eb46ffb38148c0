// The sorted tuple list of a match (the reference's rows are in join order;
// here they are returned in lexicographic order of the query's vertices).
//
// A row is one number of q * bits bits, column 0 the most significant, bits
// the width of a vertex id.  Few rows (launch-bound) are placed by counting,
// for each, the rows below it: rows^2 comparisons in one launch, 5 us at 2000
// rows.  More are sorted by radix passes over that number, 8 bits at a time
// from its low end, on (64-bit part, row index) pairs; the rows themselves are
// gathered once at the end.  Sorting 2.28e6 rows of 4 columns on the host
// (std::sort of row indices) took 150 ms of a 160 ms call.
#include <algorithm>
#include <utility>

#include "launch.h"
#include "wave.h"

namespace gpsm {

namespace {

// Bits [lo, lo + n) (n <= 64) of a row's number.
__device__ __forceinline__ unsigned long long row_bits(const uint32_t* __restrict__ t, uint32_t q, uint32_t bits,
                                                       uint32_t lo, uint32_t n) {
  unsigned long long v = 0;
  // column q - 1 - k holds bits [k * bits, (k + 1) * bits)
  for (uint32_t k = lo / bits; k < q && k * bits < lo + n; ++k) {
    const unsigned long long x = t[q - 1 - k];
    const uint32_t at = k * bits;
    v |= at >= lo ? x << (at - lo) : x >> (lo - at);
  }
  return n < 64 ? v & ((1ull << n) - 1) : v;
}

__device__ __forceinline__ bool row_less(const uint32_t* __restrict__ a, const uint32_t* __restrict__ b, uint32_t q) {
  for (uint32_t c = 0; c < q; ++c)
    if (a[c] != b[c]) return a[c] < b[c];
  return false;
}

// 64 rows per workgroup; wave w counts the rows below them among the rows
// 64w .. 64w + 63 of every RANK_ROWS.  Rows are compared by their top 128 bits
// from LDS, then (more bits than that, an equal row other than itself) column
// by column.  With 64 bits there and 256 rows at a time 1129 rows of 6 14-bit
// columns took 105 us (a row met itself once, in another iteration than any
// other lane), 64 us with 128 bits, 21 us so.
constexpr uint32_t RANK_ROWS = 1024;

__global__ void __launch_bounds__(RANK_ROWS) rank_tuples_kernel(const uint32_t* __restrict__ tuples, uint32_t q,
                                                                uint32_t bits,
                                                                const unsigned long long* __restrict__ count,
                                                                uint32_t cap, uint32_t* __restrict__ out) {
  const unsigned long long total = *count;
  if (total > cap || (uint64_t)blockIdx.x * WAVE >= total) return;
  const uint32_t n = (uint32_t)total;
  __shared__ unsigned long long key[RANK_ROWS], rest[RANK_ROWS];
  __shared__ uint32_t part[RANK_ROWS / WAVE][WAVE];
  const uint32_t lane = lane_id(), w = threadIdx.x / WAVE;
  const uint32_t width = q * bits, top = min(width, 64u), next = min(width - top, 64u);
  const uint32_t i = blockIdx.x * WAVE + lane;
  const bool mine = i < n;
  const uint32_t* ri = tuples + (size_t)min(i, n - 1) * q;
  const unsigned long long ki = row_bits(ri, q, bits, width - top, top);
  const unsigned long long li = next ? row_bits(ri, q, bits, width - top - next, next) : 0ull;
  uint32_t below = 0;
  for (uint32_t j0 = 0; j0 < n; j0 += RANK_ROWS) {
    const uint32_t j = j0 + threadIdx.x;
    __syncthreads();
    if (j < n) {
      key[threadIdx.x] = row_bits(tuples + (size_t)j * q, q, bits, width - top, top);
      rest[threadIdx.x] = next ? row_bits(tuples + (size_t)j * q, q, bits, width - top - next, next) : 0ull;
    }
    __syncthreads();
    const uint32_t m = min(WAVE * (w + 1), n - j0);
    for (uint32_t x = WAVE * w; x < m; ++x) {
      const unsigned long long kj = key[x], lj = rest[x];
      below += kj < ki || (kj == ki && lj < li);
    }
    if (width > 128)
      for (uint32_t x = WAVE * w; x < m; ++x)
        if (key[x] == ki && rest[x] == li && j0 + x != i && row_less(tuples + (size_t)(j0 + x) * q, ri, q)) ++below;
  }
  part[w][lane] = below;
  __syncthreads();
  uint32_t at = 0;
  for (uint32_t x = 0; x < RANK_ROWS / WAVE; ++x) at += part[x][lane];
  if (mine)
    for (uint32_t c = w; c < q; c += RANK_ROWS / WAVE) out[(size_t)at * q + c] = ri[c];
}

__global__ void tuple_keys_kernel(const uint32_t* __restrict__ tuples, uint64_t n, uint32_t q, uint32_t bits,
                                  uint32_t lo, uint32_t nbits, const uint32_t* idx_in,
                                  unsigned long long* __restrict__ keys, uint32_t* idx_out) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    const uint32_t r = idx_in ? idx_in[i] : (uint32_t)i;
    keys[i] = row_bits(tuples + (size_t)r * q, q, bits, lo, nbits);
    if (!idx_in) idx_out[i] = r;
  }
}

// One thread per word of the result (consecutive words to consecutive lanes).
__global__ void gather_tuples_kernel(const uint32_t* __restrict__ tuples, uint64_t n, uint32_t q,
                                     const uint32_t* __restrict__ idx, uint32_t* __restrict__ out) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x, words = n * q;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < words; i += stride) {
    const uint64_t r = i / q;
    out[i] = tuples[(size_t)idx[r] * q + (uint32_t)(i - r * q)];
  }
}

uint32_t grid_for(uint64_t items) {
  return (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>((items + 255) / 256, 16384));
}

}  // namespace

void launch_rank_tuples(const uint32_t* tuples, uint32_t q, uint32_t bits, const unsigned long long* count,
                        uint32_t cap, uint32_t* out, hipStream_t s) {
  hipLaunchKernelGGL(rank_tuples_kernel, dim3((cap + WAVE - 1) / WAVE), dim3(RANK_ROWS), 0, s, tuples, q, bits, count,
                     cap, out);
}

uint64_t tuple_sort_words(uint64_t n) {
  // keys twice, row indices twice, digit counts and their starts, scan scratch
  return 4 * n + 2 * ((n + 1) & ~1ull) + 2 * radix_hist_words(n) + scan_scratch_words(radix_hist_words(n));
}

void launch_sort_tuples(const uint32_t* tuples, uint64_t n, uint32_t q, uint32_t bits, uint32_t* scratch,
                        uint32_t* out, hipStream_t s) {
  const uint64_t ni = (n + 1) & ~1ull, nh = radix_hist_words(n);
  unsigned long long* ka = reinterpret_cast<unsigned long long*>(scratch);
  unsigned long long* kb = ka + n;
  uint32_t* ia = reinterpret_cast<uint32_t*>(kb + n);
  uint32_t* ib = ia + ni;
  uint32_t* hist = ib + ni;
  uint32_t* hstart = hist + nh;
  uint32_t* scan = hstart + nh;
  const uint32_t width = q * bits;
  for (uint32_t lo = 0; lo < width; lo += 64) {
    const uint32_t nb = std::min(64u, width - lo);
    hipLaunchKernelGGL(tuple_keys_kernel, dim3(grid_for(n)), dim3(256), 0, s, tuples, n, q, bits, lo, nb,
                       lo ? ia : nullptr, ka, ia);
    for (uint32_t shift = 0; shift < nb; shift += 8) {
      launch_radix_pass(ka, kb, ia, ib, n, shift, hist, hstart, scan, scan_scratch_words(nh), s);
      std::swap(ka, kb);
      std::swap(ia, ib);
    }
  }
  hipLaunchKernelGGL(gather_tuples_kernel, dim3(grid_for(n * q)), dim3(256), 0, s, tuples, n, q, ia, out);
}

}  // namespace gpsm
