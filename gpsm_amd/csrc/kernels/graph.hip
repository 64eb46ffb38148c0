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
#include "steps.h"
#include "wave.h"

namespace gpsm {

namespace {

// Calls f(segment, entry) for every entry of segments off[0] .. off[nseg] (off[0]
// = 0), one wave per ENTRY_BLOCK consecutive entries: its first and last
// segment by a search in all offsets, an entry's by one between them.  (With a
// wave per 64 segments the first rows of a graph whose ids descend by degree,
// a million entries, were one wave's: 8.6 ms of a 1M-vertex graph's upload.)
constexpr uint32_t ENTRY_BLOCK = 1024;

template <typename F>
__device__ __forceinline__ void for_entries(const uint32_t* __restrict__ off, uint32_t nseg, F f) {
  const uint32_t lane = lane_id(), total = off[nseg];
  const uint64_t wave = ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) / WAVE;
  const uint64_t nwaves = (uint64_t)gridDim.x * blockDim.x / WAVE;
  for (uint64_t e0 = wave * ENTRY_BLOCK; e0 < total; e0 += nwaves * ENTRY_BLOCK) {
    const uint32_t e1 = (uint32_t)min((uint64_t)total, e0 + ENTRY_BLOCK);
    const uint32_t lo = seg_search(off, nseg, (uint32_t)e0);
    const uint32_t ns = seg_search(off + lo, nseg - lo, e1 - 1) + 1;
    for_steps(e0, e1, [&](uint64_t x) {
      const uint64_t e = x + lane;
      if (e < e1) f(lo + seg_search(off + lo, ns, (uint32_t)e), (uint32_t)e);
    });
  }
}

// A hub's entry sets its neighbour's bit.
__global__ void __launch_bounds__(256) hub_bits_kernel(const uint32_t* __restrict__ lrow, uint32_t npieces, uint32_t n,
                                                       const uint32_t* __restrict__ col,
                                                       const uint32_t* __restrict__ hub_of, uint32_t W,
                                                       uint32_t* __restrict__ bits) {
  for_entries(lrow, npieces, [&](uint32_t p, uint32_t e) {
    const uint32_t h = hub_of[p % n], w = col[e];
    if (h != ~0u) atomicOr(bits + (size_t)h * W + (w >> 5), 1u << (w & 31));
  });
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
  bool wrong = false;
  for_entries(row, n, [&](uint32_t v, uint32_t e) {
    const uint32_t c = col[e];
    wrong |= c >= n || c == v || (e > row[v] && col[e - 1] >= c);
  });
  if (wrong) atomicOr(bad, 1u);
}

// place[v] = (place of id v's label among the nl distinct ones) << 32 | v, to
// be sorted by label.
__global__ void label_places_kernel(const uint32_t* __restrict__ label, uint32_t n, const uint32_t* __restrict__ value,
                                    uint32_t nl, unsigned long long* __restrict__ place) {
  const uint32_t stride = gridDim.x * blockDim.x;
  for (uint64_t v = blockIdx.x * blockDim.x + threadIdx.x; v < n; v += stride)
    place[v] = ((unsigned long long)seg_search(value, nl, label[v]) << 32) | v;
}

// ids, pos and key of the sorted places; deg[i]: vertex i's degree, deg[n] = 0.
// key[i] = (dense label << KEY_DEG_BITS) | min(degree, KEY_DEG_MASK): the dense
// label is 1 + the label's place.
__global__ void numbering_kernel(const unsigned long long* __restrict__ place, const uint32_t* __restrict__ row0,
                                 uint32_t n, uint32_t* __restrict__ ids, uint32_t* __restrict__ pos,
                                 uint32_t* __restrict__ key, uint32_t* __restrict__ deg) {
  const uint32_t stride = gridDim.x * blockDim.x;
  for (uint64_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    const unsigned long long p = place[i];
    const uint32_t v = (uint32_t)p, d = row0[v + 1] - row0[v];
    ids[i] = v;
    pos[v] = (uint32_t)i;
    key[i] = (((uint32_t)(p >> 32) + 1) << KEY_DEG_BITS) | min(d, KEY_DEG_MASK);
    deg[i] = d;
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) deg[n] = 0;
}

// The entries of vertex 0, 1, ... as (label group, vertex, label, neighbour)
// keys: the vertex and the neighbour in pb bits, the label in lb (0: left
// out).
__global__ void row_entries_kernel(const uint32_t* __restrict__ row0, const uint32_t* __restrict__ col0,
                                   const uint32_t* __restrict__ ids, const uint32_t* __restrict__ pos,
                                   const uint32_t* __restrict__ key, const uint32_t* __restrict__ row, uint32_t n,
                                   uint32_t pb, uint32_t lb, uint32_t gshift,
                                   unsigned long long* __restrict__ entry) {
  for_entries(row, n, [&](uint32_t v, uint32_t e) {
    const uint32_t x = pos[col0[row0[ids[v]] + (e - row[v])]];
    const uint32_t l = (key[x] >> KEY_DEG_BITS) - 1;
    unsigned long long k = ((unsigned long long)(l >> gshift) << pb) | v;
    if (lb) k = (k << lb) | l;
    entry[e] = (k << pb) | x;
  });
}

// lrow[p] for the pieces p = 256 b .. 256 b + 255 of a workgroup, and the end:
// entries before the piece, searched between the workgroup's first and last.
__global__ void __launch_bounds__(256) pieces_kernel(const unsigned long long* __restrict__ entry, uint32_t adj,
                                                     uint32_t n, uint64_t npieces, uint32_t pb, uint32_t lb,
                                                     uint32_t* __restrict__ lrow) {
  __shared__ uint32_t bound[2];
  // the key of piece p's first possible entry
  auto first_key = [&](uint64_t p) { return (((p / n) << pb) | (p % n)) << (lb + pb); };
  auto before = [&](unsigned long long k, uint32_t lo, uint32_t hi) {
    while (lo < hi) {
      const uint32_t mid = lo + ((hi - lo) >> 1);
      if (entry[mid] < k) lo = mid + 1;
      else hi = mid;
    }
    return lo;
  };
  for (uint64_t p0 = (uint64_t)blockIdx.x * 256; p0 <= npieces; p0 += (uint64_t)gridDim.x * 256) {
    if (threadIdx.x < 2) {
      const uint64_t p = p0 + 256 * threadIdx.x;
      bound[threadIdx.x] = p >= npieces ? adj : before(first_key(p), 0, adj);
    }
    __syncthreads();
    const uint64_t p = p0 + threadIdx.x;
    if (p <= npieces) lrow[p] = p == npieces ? adj : before(first_key(p), bound[0], bound[1]);
    __syncthreads();
  }
}

__global__ void entry_columns_kernel(const unsigned long long* __restrict__ entry, uint64_t adj, uint32_t pb,
                                     uint32_t* __restrict__ col) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; e < adj; e += stride)
    col[e] = (uint32_t)(entry[e] & ((1ull << pb) - 1));
}

__global__ void label_ranges_kernel(const uint32_t* __restrict__ fchunk, uint32_t nfchunk,
                                    const uint32_t* __restrict__ start, uint32_t nl, uint32_t* __restrict__ range) {
  const uint32_t l = blockIdx.x * blockDim.x + threadIdx.x;
  if (l >= nl) return;
  range[2 * l] = seg_search(fchunk, nfchunk + 1, start[l]);
  range[2 * l + 1] = seg_search(fchunk, nfchunk + 1, start[l + 1] - 1) + 1;
}

// Two words of every row's bitmap by id per wave: lane l gathers the bit of
// id 64 p + l, one ballot makes the words.  Within a label the ids are in the
// vertices' order, so a row's bits, all of one label, are read almost in order.
__global__ void id_bitmaps_kernel(const uint32_t* __restrict__ pos, const uint32_t* __restrict__ bitmaps, uint32_t n,
                                  uint32_t W, uint32_t nrows, uint32_t* __restrict__ out) {
  const uint64_t wave = ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) / WAVE;
  const uint64_t nwaves = (uint64_t)gridDim.x * blockDim.x / WAVE;
  const uint32_t lane = lane_id();
  for (uint64_t p = wave; p < ((uint64_t)n + WAVE - 1) / WAVE; p += nwaves) {
    const uint64_t id = p * WAVE + lane;
    const uint32_t v = id < n ? pos[id] : 0u;
    for (uint32_t r = 0; r < nrows; ++r) {
      const bool set = id < n && bit_of(bitmaps + (size_t)r * W, v);
      const unsigned long long m = __ballot(set);
      if (lane < 2 && 2 * p + lane < W) out[(size_t)r * W + 2 * p + lane] = (uint32_t)(m >> (32 * lane));
    }
  }
}

__global__ void to_ids_kernel(const uint32_t* __restrict__ ids, uint32_t* __restrict__ v, uint64_t n) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) v[i] = ids[v[i]];
}

// The filter's vertex ranges: each block of FCHUNK_VERTS vertices is cut
// greedily into ranges of at most verts vertices and FCHUNK_ENTRIES adjacency
// entries (a vertex
// with more is a range of its own).  ends[b * FCHUNK_VERTS + i]: end of range i
// of block b; count[b]: its ranges.
__global__ void __launch_bounds__(256) range_ends_kernel(const uint32_t* __restrict__ row, uint32_t n, uint32_t verts,
                                                         uint32_t* __restrict__ ends, uint32_t* __restrict__ count,
                                                         uint32_t* __restrict__ parts) {
  __shared__ uint32_t off[FCHUNK_VERTS + 1];
  const uint32_t v0 = blockIdx.x * FCHUNK_VERTS, nv = min(FCHUNK_VERTS, n - v0);
  for (uint32_t i = threadIdx.x; i <= nv; i += blockDim.x) off[i] = row[v0 + i];
  __syncthreads();
  if (threadIdx.x) return;
  uint32_t k = 0;
  for (uint32_t v = 0; v < nv; ++k) {
    uint32_t lo = v + 1, hi = min(nv, v + verts);  // the last end whose entries fit, at least one vertex
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

// hub_of[v] = before[v] (hubs before v) for hubs, ~0 for others.
__global__ void hub_list_kernel(const uint32_t* __restrict__ row, uint32_t n, uint32_t degree,
                                const uint32_t* __restrict__ before, uint32_t* __restrict__ hub_of) {
  const uint32_t stride = gridDim.x * blockDim.x;
  for (uint64_t v = blockIdx.x * blockDim.x + threadIdx.x; v < n; v += stride)
    hub_of[v] = row[v + 1] - row[v] > degree ? before[v] : ~0u;
}

__global__ void neighbour_keys_kernel(const uint32_t* __restrict__ col, const uint32_t* __restrict__ key,
                                     uint64_t adj, uint32_t* __restrict__ ckey) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; e < adj; e += stride) ckey[e] = key[col[e]];
}

uint32_t grid_for(uint64_t items) {
  return (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>((items + 255) / 256, 16384));
}

// Workgroups of 256 threads, a wave per ENTRY_BLOCK entries.
uint32_t entry_grid(uint64_t adj) { return grid_for((adj + ENTRY_BLOCK - 1) / ENTRY_BLOCK * WAVE); }

// Bits of x.
uint32_t bits_of(uint32_t x) { return x ? 32 - (uint32_t)__builtin_clz(x) : 0; }

uint32_t range_blocks(uint32_t n) { return (uint32_t)(((uint64_t)n + FCHUNK_VERTS - 1) / FCHUNK_VERTS); }

}  // namespace

void launch_vertex_stats(const uint32_t* row, const uint32_t* label, uint32_t n, uint32_t min_degree, uint32_t* hist,
                         uint32_t* hubs, hipStream_t s) {
  hipLaunchKernelGGL(vertex_stats_kernel, dim3(std::min(grid_for(n), 1024u)), dim3(256), 0, s, row, label, n,
                     min_degree, hist, hubs);
}

void launch_check_rows(const uint32_t* row, const uint32_t* col, uint32_t n, uint64_t adj, uint32_t* bad,
                       hipStream_t s) {
  hipLaunchKernelGGL(check_rows_kernel, dim3(entry_grid(adj)), dim3(256), 0, s, row, col, n, bad);
}

uint64_t relabel_words(uint32_t n, uint64_t adj) {
  const uint64_t m = std::max<uint64_t>(n, adj);
  return 4 * m + 2 * radix_hist_words(m) + scan_scratch_words(std::max(radix_hist_words(m), (uint64_t)n + 1)) +
         (((uint64_t)n + 2) & ~1ull);
}

void launch_relabel(const DevGraph& g, const uint32_t* label, const uint32_t* value, uint32_t nl, uint32_t* scratch,
                    hipStream_t s) {
  // row == row0: the vertices keep their ids, only the keys are made
  const bool sorted = g.row != g.row0;
  const uint64_t m = sorted ? std::max<uint64_t>(g.n, g.adj) : g.n, hw = radix_hist_words(m);
  unsigned long long* a = reinterpret_cast<unsigned long long*>(scratch);
  unsigned long long* b = a + m;
  uint32_t* hist = reinterpret_cast<uint32_t*>(b + m);  // hw is even
  uint32_t* hstart = hist + hw;
  uint32_t* deg = hstart + hw;
  uint32_t* scan = deg + (((uint64_t)g.n + 2) & ~1ull);
  const uint64_t sw = scan_scratch_words(std::max(hw, (uint64_t)g.n + 1));
  hipLaunchKernelGGL(label_places_kernel, dim3(grid_for(g.n)), dim3(256), 0, s, label, g.n, value, nl, a);
  for (uint32_t shift = 32; sorted && (uint64_t)(nl - 1) >> (shift - 32); shift += 8) {
    launch_radix_pass(a, b, nullptr, nullptr, g.n, shift, hist, hstart, scan, sw, s);
    std::swap(a, b);
  }
  hipLaunchKernelGGL(numbering_kernel, dim3(grid_for(g.n)), dim3(256), 0, s, a, g.row0, g.n, g.ids, g.pos, g.key, deg);
  if (!sorted) return;
  launch_exclusive_scan(deg, g.row, (uint64_t)g.n + 1, nullptr, scan, sw, s);
  if (!g.adj) {
    if (g.ngroup > 1) launch_fill_u32(g.lrow, 0u, (uint64_t)g.n * g.ngroup + 1, s);
    return;
  }
  // A vertex's entries come in the ids' order, in which those of one label
  // ascend: where every label is a group of its own, a stable sort by the group
  // is all (one pass for 256 labels).  Else by (group, vertex, label), or by
  // the whole key where the label's bits do not fit.
  const uint32_t pb = bits_of(g.n - 1), gb = bits_of(g.ngroup - 1);
  const bool exact = g.gshift == 0;
  uint32_t lb = exact ? 0 : bits_of(nl - 1);
  if (gb + 2 * pb + lb > 64) lb = 0;
  hipLaunchKernelGGL(row_entries_kernel, dim3(entry_grid(g.adj)), dim3(256), 0, s, g.row0, g.col0, g.ids, g.pos, g.key,
                     g.row, g.n, pb, lb, g.gshift, a);
  for (uint32_t shift = exact ? 2 * pb : lb ? pb : 0; shift < gb + 2 * pb + lb; shift += 8) {
    launch_radix_pass(a, b, nullptr, nullptr, g.adj, shift, hist, hstart, scan, sw, s);
    std::swap(a, b);
  }
  if (g.ngroup > 1) {
    const uint64_t np = (uint64_t)g.n * g.ngroup;
    hipLaunchKernelGGL(pieces_kernel, dim3(grid_for(np + 1)), dim3(256), 0, s, a, (uint32_t)g.adj, g.n, np, pb, lb,
                       g.lrow);
  }
  hipLaunchKernelGGL(entry_columns_kernel, dim3(grid_for(g.adj)), dim3(256), 0, s, a, g.adj, pb, g.col);
}

void choose_pieces(DevGraph& g, uint32_t nl) {
  g.gshift = 0;
  for (;; ++g.gshift) {
    g.ngroup = ((nl - 1) >> g.gshift) + 1;
    const uint64_t words = (uint64_t)g.ngroup * g.n;
    if (g.ngroup == 1 || (g.ngroup <= PIECE_GROUPS && words <= 4 * g.adj + g.n && words < 1ull << 32 &&
                          bits_of(g.ngroup - 1) + 2 * bits_of(g.n - 1) <= 64))
      return;
  }
}

void launch_label_ranges(const DevGraph& g, const uint32_t* start, uint32_t nl, uint32_t* range, hipStream_t s) {
  hipLaunchKernelGGL(label_ranges_kernel, dim3((nl + 255) / 256), dim3(256), 0, s, g.fchunk, g.nfchunk, start, nl,
                     range);
}

void launch_id_bitmaps(const DevGraph& g, const uint32_t* bitmaps, uint32_t nrows, uint32_t* out, hipStream_t s) {
  hipLaunchKernelGGL(id_bitmaps_kernel, dim3(grid_for(g.n)), dim3(256), 0, s, g.pos, bitmaps, g.n, g.W, nrows, out);
}

void launch_to_ids(const DevGraph& g, uint32_t* v, uint64_t n, hipStream_t s) {
  if (!n) return;
  hipLaunchKernelGGL(to_ids_kernel, dim3(grid_for(n)), dim3(256), 0, s, g.ids, v, n);
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
  hipLaunchKernelGGL(range_ends_kernel, dim3(nb), dim3(256), 0, s, row, n, range_verts(n), scratch, count, parts);
  launch_exclusive_scan(count, count + ne, nb, total, count + 2 * ne, scan_scratch_words(nb), s);
}

void launch_ranges(const DevGraph& g, const uint32_t* scratch, uint32_t* next, hipStream_t s) {
  const uint32_t nb = range_blocks(g.n);
  const uint32_t* count = scratch + (uint64_t)nb * FCHUNK_VERTS;
  hipLaunchKernelGGL(ranges_kernel, dim3(nb), dim3(256), 0, s, scratch, count, count + (((uint64_t)nb + 1) & ~1ull),
                     g.row, g.n, g.fchunk, g.wrange, g.hparts, next);
}

uint64_t hub_words(uint32_t n) { return 2 * (((uint64_t)n + 1) & ~1ull) + scan_scratch_words(n); }

void launch_hubs(const DevGraph& g, uint32_t* scratch, hipStream_t s) {
  const uint64_t nv = ((uint64_t)g.n + 1) & ~1ull;
  uint32_t* flag = scratch;
  uint32_t* before = flag + nv;
  hipLaunchKernelGGL(hub_flags_kernel, dim3(grid_for(g.n)), dim3(256), 0, s, g.row, g.n, g.hub_degree, flag);
  launch_exclusive_scan(flag, before, g.n, nullptr, before + nv, scan_scratch_words(g.n), s);
  hipLaunchKernelGGL(hub_list_kernel, dim3(grid_for(g.n)), dim3(256), 0, s, g.row, g.n, g.hub_degree, before,
                     g.hub_of);
  const uint64_t np = (uint64_t)g.n * g.ngroup;
  hipLaunchKernelGGL(hub_bits_kernel, dim3(entry_grid(g.adj)), dim3(256), 0, s, g.lrow, (uint32_t)np, g.n,
                     g.col, g.hub_of, g.W, g.hub_bits);
}

void launch_neighbour_keys(const DevGraph& g, hipStream_t s) {
  if (!g.adj) return;
  uint64_t grid = (g.adj + 255) / 256;
  if (grid > 16384) grid = 16384;
  hipLaunchKernelGGL(neighbour_keys_kernel, dim3((uint32_t)grid), dim3(256), 0, s, g.col, g.key, g.adj, g.ckey);
}

}  // namespace gpsm
