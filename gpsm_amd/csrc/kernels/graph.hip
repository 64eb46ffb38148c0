// Graph-resident structures built once at upload.
//
// Neighbour keys: ckey[e] = key[col[e]], the label/degree key of every
// adjacency entry's target, stored beside col (4 bytes per entry).
//
// Hub adjacency bitmaps: one n-bit bitmap per hub (a vertex above the hub
// degree), so that the join's edge-membership test of a pair touching a hub
// is one bit instead of a binary search in an adjacency list of up to 10^5
// entries (the R-MAT graph's largest), which costs ~17 dependent loads.
#include <algorithm>

#include "launch.h"
#include "wave.h"

namespace gpsm {

namespace {

// One wave per (hub, 64-entry block of its adjacency): grid-stride over the
// blocks of all hubs, found with a binary search over their prefix sums.
__global__ void __launch_bounds__(256) hub_bits_kernel(const uint32_t* __restrict__ row,
                                                       const uint32_t* __restrict__ col,
                                                       const uint32_t* __restrict__ hubs,
                                                       const uint32_t* __restrict__ block_base, uint32_t nhub,
                                                       uint32_t W, uint32_t* __restrict__ bits) {
  const uint32_t lane = lane_id();
  const uint64_t wave = ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) / WAVE;
  const uint64_t nwaves = ((uint64_t)gridDim.x * blockDim.x) / WAVE;
  const uint32_t nblocks = block_base[nhub];
  for (uint64_t it = wave; it < nblocks; it += nwaves) {
    const uint32_t h = uniform(seg_search(block_base, nhub + 1, (uint32_t)it));
    const uint32_t v = hubs[h];
    const uint32_t e = row[v] + ((uint32_t)it - block_base[h]) * WAVE + lane;
    if (e < row[v + 1]) {
      const uint32_t w = col[e];
      atomicOr(bits + (size_t)h * W + (w >> 5), 1u << (w & 31));
    }
  }
}

// Label statistics and hub counts of a graph, and its rows' order, in one
// pass each.  Host loops over the vertices and a std::sort of the labels took
// 29 of the 34.5 ms of building a 1M-vertex, 8M-edge graph from its edge list
// (5.3 ms now, 2.9 of them the edge list's copy).
//
// hist[l] for labels l < LABEL_HIST, hist[LABEL_HIST]: vertices with a larger
// label; hubs[k]: vertices whose degree exceeds min_degree * 2^j for exactly
// j = 0 .. k - 1.
__global__ void __launch_bounds__(256) vertex_stats_kernel(const uint32_t* __restrict__ row,
                                                           const uint32_t* __restrict__ label, uint32_t n,
                                                           uint32_t min_degree, uint32_t* __restrict__ hist,
                                                           uint32_t* __restrict__ hubs) {
  __shared__ uint32_t h[LABEL_HIST + 1];
  __shared__ uint32_t hb[HUB_STEPS];
  for (uint32_t i = threadIdx.x; i <= LABEL_HIST; i += blockDim.x) h[i] = 0;
  if (threadIdx.x < HUB_STEPS) hb[threadIdx.x] = 0;
  __syncthreads();
  const uint32_t stride = gridDim.x * blockDim.x;
  for (uint64_t v = blockIdx.x * blockDim.x + threadIdx.x; v < n; v += stride) {
    atomicAdd(&h[min(label[v], LABEL_HIST)], 1u);
    const uint32_t deg = row[v + 1] - row[v];
    uint32_t k = 0;
    for (uint64_t d = min_degree; deg > d; d *= 2) ++k;
    if (k) atomicAdd(&hb[k], 1u);
  }
  __syncthreads();
  for (uint32_t i = threadIdx.x; i <= LABEL_HIST; i += blockDim.x)
    if (h[i]) atomicAdd(&hist[i], h[i]);
  if (threadIdx.x < HUB_STEPS && hb[threadIdx.x]) atomicAdd(&hubs[threadIdx.x], hb[threadIdx.x]);
}

// *bad |= 1 if a row is not strictly ascending, names a vertex >= n or its own.
__global__ void check_rows_kernel(const uint32_t* __restrict__ row, const uint32_t* __restrict__ col, uint32_t n,
                                  uint32_t* __restrict__ bad) {
  // one wave per 64 rows, flattened over their entries by a search in the offsets
  const uint64_t wave = ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) / WAVE;
  const uint64_t nwaves = (uint64_t)gridDim.x * blockDim.x / WAVE;
  const uint32_t lane = lane_id();
  bool wrong = false;
  for (uint64_t v0 = wave * WAVE; v0 < n; v0 += nwaves * WAVE) {
    const uint32_t nv = (uint32_t)min((uint64_t)WAVE, n - v0);
    const uint32_t e1 = row[v0 + nv];
    for (uint32_t e = row[v0] + lane; e < e1; e += WAVE) {
      const uint32_t i = seg_search(row + v0, nv, e);  // the last row starting at or before e: it holds e
      const uint32_t c = col[e];
      wrong |= c >= n || c == v0 + i || (e > row[v0 + i] && col[e - 1] >= c);
    }
  }
  if (wrong) atomicOr(bad, 1u);
}

// key[v] = (dense label << KEY_DEG_BITS) | min(degree, KEY_DEG_MASK): the
// dense label is 1 + the label's place among the nl distinct ones.
__global__ void vertex_keys_kernel(const uint32_t* __restrict__ row, const uint32_t* __restrict__ label, uint32_t n,
                                   const uint32_t* __restrict__ value, uint32_t nl, uint32_t* __restrict__ key) {
  const uint32_t stride = gridDim.x * blockDim.x;
  for (uint64_t v = blockIdx.x * blockDim.x + threadIdx.x; v < n; v += stride)
    key[v] = ((seg_search(value, nl, label[v]) + 1) << KEY_DEG_BITS) | min(row[v + 1] - row[v], KEY_DEG_MASK);
}

// The filter's vertex ranges: each block of FCHUNK_VERTS vertices is cut
// greedily into ranges of at most FCHUNK_ENTRIES adjacency entries (a vertex
// with more is a range of its own).  ends[b * FCHUNK_VERTS + i]: end of range i
// of block b; count[b]: its ranges.
__global__ void __launch_bounds__(256) range_ends_kernel(const uint32_t* __restrict__ row, uint32_t n,
                                                         uint32_t* __restrict__ ends, uint32_t* __restrict__ count,
                                                         uint32_t* __restrict__ parts) {
  __shared__ uint32_t off[FCHUNK_VERTS + 1];
  const uint32_t v0 = blockIdx.x * FCHUNK_VERTS, nv = min(FCHUNK_VERTS, n - v0);
  for (uint32_t i = threadIdx.x; i <= nv; i += blockDim.x) off[i] = row[v0 + i];
  __syncthreads();
  if (threadIdx.x) return;
  uint32_t k = 0;
  for (uint32_t v = 0; v < nv; ++k) {
    uint32_t lo = v + 1, hi = nv;  // the last end whose entries fit, at least one vertex
    while (lo < hi) {
      const uint32_t mid = (lo + hi + 1) >> 1;
      if (off[mid] - off[v] <= FCHUNK_ENTRIES) lo = mid;
      else hi = mid - 1;
    }
    ends[(size_t)v0 + k] = v0 + lo;
    const uint32_t entries = off[lo] - off[v];  // over the limit: one vertex
    if (entries > FCHUNK_ENTRIES) atomicAdd(parts, (entries + HUB_PART - 1) / HUB_PART);
    v = lo;
  }
  count[blockIdx.x] = k;
}

// fchunk and wrange from the blocks' ranges; base[b]: ranges before block b.
__global__ void __launch_bounds__(256) ranges_kernel(const uint32_t* __restrict__ ends,
                                                     const uint32_t* __restrict__ count,
                                                     const uint32_t* __restrict__ base,
                                                     const uint32_t* __restrict__ row, uint32_t n,
                                                     uint32_t* __restrict__ fchunk, uint32_t* __restrict__ wrange,
                                                     uint2* __restrict__ hparts, uint32_t* __restrict__ next) {
  const uint32_t b = blockIdx.x, v0 = b * FCHUNK_VERTS, c = count[b], r0 = base[b];
  const uint32_t* e = ends + v0;
  for (uint32_t i = threadIdx.x; i < c; i += blockDim.x) {
    fchunk[r0 + i + 1] = e[i];
    const uint32_t v = e[i] - 1, entries = row[v + 1] - row[v];
    if (entries > FCHUNK_ENTRIES) {
      const uint32_t np = (entries + HUB_PART - 1) / HUB_PART, at = atomicAdd(next, np);
      for (uint32_t k = 0; k < np; ++k) hparts[at + k] = make_uint2(v, k);
    }
  }
  if (b == 0 && threadIdx.x == 0) fchunk[0] = 0;
  for (uint32_t i = threadIdx.x; i < FCHUNK_VERTS / 32; i += blockDim.x) {
    const uint32_t v = v0 + 32 * i;
    if (v >= n) break;
    uint32_t lo = 0, hi = c;  // ranges ending at or before v
    while (lo < hi) {
      const uint32_t mid = (lo + hi) >> 1;
      if (e[mid] <= v) lo = mid + 1;
      else hi = mid;
    }
    wrange[v / 32] = r0 + lo;
  }
}

__global__ void hub_flags_kernel(const uint32_t* __restrict__ row, uint32_t n, uint32_t degree,
                                 uint32_t* __restrict__ flag) {
  const uint32_t stride = gridDim.x * blockDim.x;
  for (uint64_t v = blockIdx.x * blockDim.x + threadIdx.x; v < n; v += stride)
    flag[v] = row[v + 1] - row[v] > degree;
}

// hub_of[v] = pos[v] for hubs (pos: hubs before v), ~0 for others; the hubs and
// their 64-entry adjacency blocks (one more entry, 0, for a scan's total).
__global__ void hub_list_kernel(const uint32_t* __restrict__ row, uint32_t n, uint32_t degree, uint32_t nhub,
                                const uint32_t* __restrict__ pos, uint32_t* __restrict__ hub_of,
                                uint32_t* __restrict__ hubs, uint32_t* __restrict__ blocks) {
  const uint32_t stride = gridDim.x * blockDim.x;
  for (uint64_t v = blockIdx.x * blockDim.x + threadIdx.x; v < n; v += stride) {
    const uint32_t deg = row[v + 1] - row[v];
    if (deg > degree) {
      hub_of[v] = pos[v];
      hubs[pos[v]] = (uint32_t)v;
      blocks[pos[v]] = (deg + WAVE - 1) / WAVE;
    } else {
      hub_of[v] = ~0u;
    }
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) blocks[nhub] = 0;
}

__global__ void neighbour_keys_kernel(const uint32_t* __restrict__ col, const uint32_t* __restrict__ key,
                                     uint64_t adj, uint32_t* __restrict__ ckey) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; e < adj; e += stride) ckey[e] = key[col[e]];
}

uint32_t grid_for(uint64_t items) {
  return (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>((items + 255) / 256, 16384));
}

uint32_t range_blocks(uint32_t n) { return (uint32_t)(((uint64_t)n + FCHUNK_VERTS - 1) / FCHUNK_VERTS); }

}  // namespace

void launch_vertex_stats(const uint32_t* row, const uint32_t* label, uint32_t n, uint32_t min_degree, uint32_t* hist,
                         uint32_t* hubs, hipStream_t s) {
  hipLaunchKernelGGL(vertex_stats_kernel, dim3(std::min(grid_for(n), 1024u)), dim3(256), 0, s, row, label, n,
                     min_degree, hist, hubs);
}

void launch_check_rows(const uint32_t* row, const uint32_t* col, uint32_t n, uint32_t* bad, hipStream_t s) {
  hipLaunchKernelGGL(check_rows_kernel, dim3(grid_for(n)), dim3(256), 0, s, row, col, n, bad);
}

void launch_vertex_keys(const DevGraph& g, const uint32_t* label, const uint32_t* value, uint32_t nl, hipStream_t s) {
  hipLaunchKernelGGL(vertex_keys_kernel, dim3(grid_for(g.n)), dim3(256), 0, s, g.row, label, g.n, value, nl, g.key);
}

uint64_t range_words(uint32_t n) {
  const uint64_t nb = range_blocks(n);
  return nb * FCHUNK_VERTS + 2 * ((nb + 1) & ~1ull) + scan_scratch_words(nb);
}

void launch_range_ends(const uint32_t* row, uint32_t n, uint32_t* scratch, unsigned long long* total, uint32_t* parts,
                       hipStream_t s) {
  const uint32_t nb = range_blocks(n);
  const uint64_t ne = ((uint64_t)nb + 1) & ~1ull;
  uint32_t* count = scratch + (uint64_t)nb * FCHUNK_VERTS;
  hipLaunchKernelGGL(range_ends_kernel, dim3(nb), dim3(256), 0, s, row, n, scratch, count, parts);
  launch_exclusive_scan(count, count + ne, nb, total, count + 2 * ne, scan_scratch_words(nb), s);
}

void launch_ranges(const DevGraph& g, const uint32_t* scratch, uint32_t* next, hipStream_t s) {
  const uint32_t nb = range_blocks(g.n);
  const uint32_t* count = scratch + (uint64_t)nb * FCHUNK_VERTS;
  hipLaunchKernelGGL(ranges_kernel, dim3(nb), dim3(256), 0, s, scratch, count, count + (((uint64_t)nb + 1) & ~1ull),
                     g.row, g.n, g.fchunk, g.wrange, g.hparts, next);
}

uint64_t hub_words(uint32_t n, uint64_t nhub) {
  return 2 * (((uint64_t)n + 1) & ~1ull) + 3 * ((nhub + 2) & ~1ull) +
         scan_scratch_words(std::max<uint64_t>(n, nhub + 1));
}

void launch_hubs(const DevGraph& g, uint32_t* scratch, hipStream_t s) {
  const uint64_t nv = ((uint64_t)g.n + 1) & ~1ull, nh = ((uint64_t)g.nhub + 2) & ~1ull;
  uint32_t* flag = scratch;
  uint32_t* pos = flag + nv;
  uint32_t* hubs = pos + nv;
  uint32_t* blocks = hubs + nh;
  uint32_t* base = blocks + nh;
  uint32_t* scan = base + nh;
  const uint64_t sw = scan_scratch_words(std::max<uint64_t>(g.n, (uint64_t)g.nhub + 1));
  hipLaunchKernelGGL(hub_flags_kernel, dim3(grid_for(g.n)), dim3(256), 0, s, g.row, g.n, g.hub_degree, flag);
  launch_exclusive_scan(flag, pos, g.n, nullptr, scan, sw, s);
  hipLaunchKernelGGL(hub_list_kernel, dim3(grid_for(g.n)), dim3(256), 0, s, g.row, g.n, g.hub_degree, g.nhub, pos,
                     g.hub_of, hubs, blocks);
  launch_exclusive_scan(blocks, base, (uint64_t)g.nhub + 1, nullptr, scan, sw, s);
  launch_hub_bits(g, hubs, base, (uint32_t)std::min<uint64_t>(g.adj / WAVE + g.nhub, 0xFFFFFFFFull), s);
}

void launch_neighbour_keys(const DevGraph& g, hipStream_t s) {
  if (!g.adj) return;
  uint64_t grid = (g.adj + 255) / 256;
  if (grid > 16384) grid = 16384;
  hipLaunchKernelGGL(neighbour_keys_kernel, dim3((uint32_t)grid), dim3(256), 0, s, g.col, g.key, g.adj, g.ckey);
}

void launch_hub_bits(const DevGraph& g, const uint32_t* hubs, const uint32_t* block_base, uint32_t nblocks,
                     hipStream_t s) {
  if (!g.nhub || !nblocks) return;
  const uint32_t block = 256;
  uint64_t grid = ((uint64_t)nblocks * WAVE + block - 1) / block;
  if (grid > 65536) grid = 65536;
  hipLaunchKernelGGL(hub_bits_kernel, dim3((uint32_t)grid), dim3(block), 0, s, g.row, g.col, hubs, block_base,
                     g.nhub, g.W, g.hub_bits);
}

}  // namespace gpsm
