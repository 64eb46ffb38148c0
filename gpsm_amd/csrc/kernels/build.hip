// Undirected CSR built on the device from an edge list (the reference
// builds it on the host from per-vertex in/out vectors and sorts each row,
// graph/Graph.cpp:30-104; its own note at graph/Graph.cpp:26-28 asks for a
// GPU build).  Every edge {a, b} becomes the two keys a<<cb|b and b<<cb|a, cb
// the bits of a vertex (five 8-bit passes for 2^20 vertices; seven with the
// column in a word of its own: 8.9 against 8.4 ms for a graph of 1M vertices);
// an LSD radix sort of the 64-bit keys orders them by (row, column), a scan of
// "first of its run" flags drops duplicates, and the row offsets are lower
// bounds of v<<cb.  Self-loops become the key n<<cb, which sorts after every
// real row and is left out of the offsets.
#include <algorithm>

#include "gpsm.h"
#include "launch.h"
#include "pool.h"
#include "stager.h"
#include "wave.h"

namespace gpsm {

namespace {

__global__ void edge_keys_kernel(const uint32_t* __restrict__ src, const uint32_t* __restrict__ dst, uint64_t m,
                                 uint32_t n, uint32_t cb, unsigned long long* __restrict__ keys,
                                 uint32_t* __restrict__ bad) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < m; i += stride) {
    const uint32_t a = src[i], b = dst[i];
    unsigned long long k0 = (unsigned long long)n << cb, k1 = k0;
    if (a >= n || b >= n) {
      atomicOr(bad, 1u);
    } else if (a != b) {
      k0 = ((unsigned long long)a << cb) | b;
      k1 = ((unsigned long long)b << cb) | a;
    }
    keys[2 * i] = k0;
    keys[2 * i + 1] = k1;
  }
}

// row[v] = first key position with row >= v, for v = 0..n (a lower bound).
__global__ void row_offsets_kernel(const unsigned long long* __restrict__ keys, uint64_t count, uint32_t n,
                                   uint32_t cb, uint32_t* __restrict__ row) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t v = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; v <= n; v += stride) {
    const unsigned long long target = v << cb;
    uint64_t lo = 0, hi = count;
    while (lo < hi) {
      const uint64_t mid = (lo + hi) >> 1;
      if (keys[mid] < target) lo = mid + 1;
      else hi = mid;
    }
    row[v] = (uint32_t)lo;
  }
}

__global__ void columns_kernel(const unsigned long long* __restrict__ keys, uint64_t adj, uint32_t cb,
                               uint32_t* __restrict__ col) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < adj; i += stride)
    col[i] = (uint32_t)(keys[i] & ((1ull << cb) - 1));
}

// flags[i] = 1 where key i starts a run of equal keys (the keys sorted)
__global__ void run_heads_kernel(const unsigned long long* __restrict__ keys, uint64_t n,
                                 uint32_t* __restrict__ flags) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
    flags[i] = (i == 0 || keys[i] != keys[i - 1]) ? 1u : 0u;
}

__global__ void keep_heads_kernel(const unsigned long long* __restrict__ keys, uint64_t n,
                                  const uint32_t* __restrict__ flags, const uint32_t* __restrict__ pos,
                                  unsigned long long* __restrict__ uniq) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
    if (flags[i]) uniq[pos[i]] = keys[i];
}

uint32_t grid_for(uint64_t items) {
  const uint64_t g = (items + 255) / 256;
  return (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>(g, 16384));
}

}  // namespace

int build_csr_from_edges(uint32_t n, uint64_t m, const uint32_t* src, const uint32_t* dst, BlockPool& pool,
                         Stager& stager, hipStream_t s, uint32_t** row, uint32_t** col, uint64_t* adj_out) {
  *row = *col = nullptr;
  *adj_out = 0;
  const uint64_t M2 = 2 * m;
  if (M2 > 0xFFFFFFFFull) return GPSM_EINVAL;  // positions are 32-bit
  uint32_t *d_src = nullptr, *d_dst = nullptr, *d_bad = nullptr, *hist = nullptr, *hstart = nullptr;
  uint32_t *flags = nullptr, *fpos = nullptr, *scratch = nullptr;
  unsigned long long *keys = nullptr, *sorted = nullptr, *d_count = nullptr;
  int rc = GPSM_OK;
  auto cleanup = [&]() {
    pool.give(d_src);
    pool.give(d_dst);
    pool.give(d_bad);
    pool.give(hist);
    pool.give(hstart);
    pool.give(flags);
    pool.give(fpos);
    pool.give(scratch);
    pool.give(keys);
    pool.give(sorted);
    pool.give(d_count);
  };
  // bits of a column, and of a row up to the sentinel n
  uint32_t cb = 1;
  while (cb < 32 && ((uint64_t)n >> cb)) ++cb;
  const uint32_t end_bit = 2 * cb;
  const uint64_t nhist = radix_hist_words(M2);
  const uint64_t sw = scan_scratch_words(std::max<uint64_t>(nhist, M2)) + 2;
  if (!pool.take(&d_bad, 1) || !pool.take(&d_count, 1) || !pool.take(row, (size_t)n + 1) ||
      (M2 && (!pool.take(&d_src, m) || !pool.take(&d_dst, m) || !pool.take(&keys, M2) || !pool.take(&sorted, M2) ||
              !pool.take(&hist, nhist) || !pool.take(&hstart, nhist) || !pool.take(&flags, M2) ||
              !pool.take(&fpos, M2) || !pool.take(&scratch, sw)))) {
    pool.give(*row);
    *row = nullptr;
    cleanup();
    return GPSM_ENOMEM;
  }
  uint32_t bad = 0;
  unsigned long long count = 0;
  if (hipMemsetAsync(d_bad, 0, sizeof(uint32_t), s) != hipSuccess ||
      hipMemsetAsync(d_count, 0, sizeof(unsigned long long), s) != hipSuccess)
    rc = GPSM_EDEVICE;
  // the sorted, deduplicated keys end up in `keys` (the passes ping-pong)
  unsigned long long* uniq = keys;
  if (!rc && M2) {
    if (stager.to_device(d_src, src, sizeof(uint32_t) * m, s) != hipSuccess ||
        stager.to_device(d_dst, dst, sizeof(uint32_t) * m, s) != hipSuccess) {
      rc = GPSM_EDEVICE;
    } else {
      hipLaunchKernelGGL(edge_keys_kernel, dim3(grid_for(m)), dim3(256), 0, s, d_src, d_dst, m, n, cb, keys, d_bad);
      unsigned long long *a = keys, *b = sorted;
      for (uint32_t shift = 0; shift < end_bit; shift += 8) {
        launch_radix_pass(a, b, nullptr, nullptr, M2, shift, hist, hstart, scratch + 2, sw - 2, s);
        std::swap(a, b);
      }
      // a holds the sorted keys; the first key of each run of equal keys is kept, in order, in b
      hipLaunchKernelGGL(run_heads_kernel, dim3(grid_for(M2)), dim3(256), 0, s, a, M2, flags);
      launch_exclusive_scan(flags, fpos, M2, d_count, scratch + 2, sw - 2, s);
      hipLaunchKernelGGL(keep_heads_kernel, dim3(grid_for(M2)), dim3(256), 0, s, a, M2, flags, fpos, b);
      uniq = b;
      if (hipGetLastError() != hipSuccess) rc = GPSM_EDEVICE;
    }
  }
  if (!rc && (hipMemcpyAsync(&bad, d_bad, sizeof(uint32_t), hipMemcpyDeviceToHost, s) != hipSuccess ||
              hipMemcpyAsync(&count, d_count, sizeof(count), hipMemcpyDeviceToHost, s) != hipSuccess ||
              hipStreamSynchronize(s) != hipSuccess))
    rc = GPSM_EDEVICE;
  if (!rc && bad) rc = GPSM_EINVAL;  // an endpoint >= n
  if (!rc) {
    hipLaunchKernelGGL(row_offsets_kernel, dim3(grid_for((uint64_t)n + 1)), dim3(256), 0, s, uniq, count, n, cb, *row);
    uint32_t adj32 = 0;
    if (hipMemcpyAsync(&adj32, *row + n, sizeof(uint32_t), hipMemcpyDeviceToHost, s) != hipSuccess ||
        hipStreamSynchronize(s) != hipSuccess) {
      rc = GPSM_EDEVICE;
    } else {
      *adj_out = adj32;
      if (!pool.take(col, std::max<uint64_t>(adj32, 1))) {
        rc = GPSM_ENOMEM;
      } else {
        if (adj32)
          hipLaunchKernelGGL(columns_kernel, dim3(grid_for(adj32)), dim3(256), 0, s, uniq, (uint64_t)adj32, cb, *col);
        if (hipStreamSynchronize(s) != hipSuccess || hipGetLastError() != hipSuccess) rc = GPSM_EDEVICE;
      }
    }
  }
  if (rc) (void)hipStreamSynchronize(s);  // nothing queued still uses what is given back
  cleanup();
  if (rc) {
    pool.give(*row);
    pool.give(*col);
    *row = *col = nullptr;
  }
  return rc;
}

}  // namespace gpsm
