// Scan and compaction on gfx950: the reference's kernel_collect
// (transform_kernel + thrust::exclusive_scan + scatter_kernel,
// match/Match.cu:463-526) and its unbuilt Blelloch prefix scan / stream
// compaction (util/prefix_scan.cu:158-427, util/compact_scan.cu:7-70).
//
// Candidate sets are bitmaps here, so "collect" is a popcount scan.  Each
// bitmap row is cut into segments of SEG_WORDS words, so that a batch of a
// few hundred rows still fills 256 CUs: a first pass popcounts every
// segment (one workgroup per (row, segment)), a row's segment counts are
// scanned in place into row-relative offsets (one workgroup per row; the
// total is the row's candidate count), and the second pass (one workgroup
// per four consecutive segments of a row) takes the group's base from them
// and compacts the four one after the other (each
// thread owns eight consecutive words, one block scan places them), ids
// staged in LDS and written back coalesced.  The same pass writes the rank
// index (set bits before each word, row-relative) the join uses to find a vertex's candidate-edge list.
#include <algorithm>

#include "launch.h"
#include "wave.h"

namespace gpsm {

namespace {

__global__ void __launch_bounds__(256) seg_popcount_kernel(const uint32_t* __restrict__ bitmaps, uint32_t W,
                                                           uint32_t nseg, uint32_t* __restrict__ segc) {
  __shared__ uint32_t part[4];
  const uint32_t r = blockIdx.x / nseg, sg = blockIdx.x % nseg;
  const uint32_t* bm = bitmaps + (size_t)r * W;
  const uint32_t base = sg * SEG_WORDS;
  uint32_t v[SEG_WORDS / 256];
  if (base + SEG_WORDS <= W) {  // a whole segment: the loads unconditional, all in flight together
#pragma unroll
    for (uint32_t j = 0; j < SEG_WORDS / 256; ++j) v[j] = bm[base + j * 256 + threadIdx.x];
  } else {
#pragma unroll
    for (uint32_t j = 0; j < SEG_WORDS / 256; ++j) {
      const uint32_t i = base + j * 256 + threadIdx.x;
      v[j] = i < W ? bm[i] : 0u;
    }
  }
  uint32_t c = 0;
#pragma unroll
  for (uint32_t j = 0; j < SEG_WORDS / 256; ++j) c += __popc(v[j]);
  c = wave_sum(c);
  if (lane_id() == 0) part[threadIdx.x / WAVE] = c;
  __syncthreads();
  if (threadIdx.x == 0) segc[blockIdx.x] = part[0] + part[1] + part[2] + part[3];
}

// Exclusive scan of p[0..n) in place by one workgroup of NT threads, in
// chunks of NT * ITEMS values in striped order (thread t holds p[c + j * NT
// + t]): a wave scan per row j, one wave scan of the (row, wave) totals in
// element order, a running carry across chunks.  Returns the total (in
// every thread).  Contains __syncthreads.
template <typename T, uint32_t NT, uint32_t ITEMS>
__device__ __forceinline__ T block_scan_in_place(T* __restrict__ p, uint32_t n) {
  constexpr uint32_t NW = NT / WAVE;
  static_assert(NT % WAVE == 0 && ITEMS * NW == WAVE, "one wave scans the (row, wave) totals");
  __shared__ T wt[ITEMS * NW + 1];  // (row j, wave w) at j * NW + w, then the chunk total
  const uint32_t lane = lane_id(), w = threadIdx.x / WAVE;
  T carry = 0;
  for (uint32_t base = 0; base < n; base += NT * ITEMS) {
    T v[ITEMS];
#pragma unroll
    for (uint32_t j = 0; j < ITEMS; ++j) {
      const uint32_t i = base + j * NT + threadIdx.x;
      v[j] = i < n ? p[i] : T(0);
    }
#pragma unroll
    for (uint32_t j = 0; j < ITEMS; ++j) {
      T incl;
      if constexpr (sizeof(T) == 8) incl = wave_incl_scan64(v[j]);
      else incl = wave_incl_scan(v[j]);
      if (lane == WAVE - 1) wt[j * NW + w] = incl;
      v[j] = incl - v[j];  // exclusive within the wave's 64 values of row j
    }
    __syncthreads();
    if (w == 0) {
      const T x = wt[lane];
      T incl;
      if constexpr (sizeof(T) == 8) incl = wave_incl_scan64(x);
      else incl = wave_incl_scan(x);
      wt[lane] = incl - x;
      if (lane == WAVE - 1) wt[ITEMS * NW] = incl;
    }
    __syncthreads();
#pragma unroll
    for (uint32_t j = 0; j < ITEMS; ++j) {
      const uint32_t i = base + j * NT + threadIdx.x;
      if (i < n) p[i] = carry + wt[j * NW + w] + v[j];
    }
    carry += wt[ITEMS * NW];
    __syncthreads();  // the next chunk rewrites wt
  }
  return carry;
}

// Row r's segment popcounts become their exclusive prefix sums (in place),
// and counts[r] their total: one workgroup per row, 4096 segments per step.
// The compaction then reads a group's row-relative base with one load.
// (One thread per row adding its counts took 0.5 ms for the 8192 segments
// of a 2^29-bit row, and each compaction workgroup re-added the counts
// before its group.)
__global__ void __launch_bounds__(256) seg_offsets_kernel(uint32_t* __restrict__ segc, uint32_t nseg,
                                                          uint32_t* __restrict__ counts) {
  const uint32_t t = block_scan_in_place<uint32_t, 256, 16>(segc + (size_t)blockIdx.x * nseg, nseg);
  if (threadIdx.x == 0) counts[blockIdx.x] = t;
}

// A workgroup compacts COMPACT_GROUP consecutive segments of one row, one
// after the other: thread t holds the words j * 256 + t of a segment (eight
// loads in flight, and the next segment's eight issued before the current
// one is scanned); a wave scan per row j of its words' popcounts and one
// scan of the (row, wave) totals give every word its output position,
// which is its rank-index entry, and the ids
// go through LDS (in rounds of STAGE_IDS output positions when the segment
// holds more) and are written back coalesced.  The row's set bits before
// the group come from the segment popcounts; within the group the
// workgroup carries them.  Measured per batch on the 1M Chung-Lu mix: 0.29
// ms for one segment per workgroup, eight consecutive words per thread and
// dense segments written by the threads; 0.27 ms for four segments; 0.23 ms
// with dense segments staged in rounds (stages of 4096 and 2048 ids 0.25
// and 0.41 ms; sixteen segments per workgroup 0.31 ms); 0.19 ms with the
// words in striped order.
constexpr uint32_t CW = 8;             // words per thread
constexpr uint32_t STAGE_IDS = 8192;   // ids staged in LDS per round
constexpr uint32_t COMPACT_GROUP = 4;  // segments per workgroup
static_assert(SEG_WORDS == 256 * CW && CW * 4 < WAVE, "a segment is CW words per thread; one wave scans the totals");

// Words of a segment in striped order: thread t holds words j * 256 + t,
// j < CW (every load instruction reads 256 contiguous bytes per wave).
__device__ __forceinline__ void load_words(const uint32_t* __restrict__ bm, uint32_t W, uint32_t s0,
                                           uint32_t (&w)[CW]) {
  if (s0 + SEG_WORDS <= W) {
#pragma unroll
    for (uint32_t j = 0; j < CW; ++j) w[j] = bm[s0 + j * 256 + threadIdx.x];
  } else {
#pragma unroll
    for (uint32_t j = 0; j < CW; ++j) {
      const uint32_t i = s0 + j * 256 + threadIdx.x;
      w[j] = i < W ? bm[i] : 0u;
    }
  }
}

__global__ void __launch_bounds__(256) compact_rows_kernel(const uint32_t* __restrict__ bitmaps, uint32_t W,
                                                           uint32_t nseg,
                                                           const uint32_t* __restrict__ segc,
                                                           const uint64_t* __restrict__ coff,
                                                           uint32_t* __restrict__ clist,
                                                           uint32_t* __restrict__ bprefix) {
  __shared__ uint32_t stage[STAGE_IDS];
  __shared__ uint32_t wt[CW * 4 + 1];  // (row j, wave) popcount totals, then their offsets; [CW * 4] = segment total
  __shared__ uint32_t rel;
  const uint32_t lane = lane_id(), wv = threadIdx.x / WAVE;
  const uint32_t ngrp = (nseg + COMPACT_GROUP - 1) / COMPACT_GROUP;
  const uint32_t r = blockIdx.x / ngrp, sg0 = (blockIdx.x % ngrp) * COMPACT_GROUP;
  const uint32_t sg1 = min(nseg, sg0 + COMPACT_GROUP);
  const uint32_t* bm = bitmaps + (size_t)r * W;
  uint32_t* bp = bprefix + (size_t)r * W;
  uint32_t* out = clist + coff[r];
  if (threadIdx.x == 0) rel = segc[(size_t)r * nseg + sg0];  // set bits of the row's segments before the group
  uint32_t w[CW];
  load_words(bm, W, sg0 * SEG_WORDS, w);
  for (uint32_t sg = sg0; sg < sg1; ++sg) {
    const uint32_t s0 = sg * SEG_WORDS;
    uint32_t nx[CW] = {};
    if (sg + 1 < sg1) load_words(bm, W, s0 + SEG_WORDS, nx);
    // positions: per row j a wave scan of the 64 words' popcounts, then one
    // scan of the (row, wave) totals in word order
    uint32_t pos[CW];
#pragma unroll
    for (uint32_t j = 0; j < CW; ++j) {
      const uint32_t c = __popc(w[j]);
      const uint32_t incl = wave_incl_scan(c);
      if (lane == WAVE - 1) wt[j * 4 + wv] = incl;
      pos[j] = incl - c;
    }
    __syncthreads();  // also publishes rel
    if (wv == 0) {
      const uint32_t x = lane < CW * 4 ? wt[lane] : 0u;
      const uint32_t incl = wave_incl_scan(x);
      if (lane < CW * 4) wt[lane] = incl - x;
      if (lane == CW * 4 - 1) wt[CW * 4] = incl;
    }
    __syncthreads();
    const uint32_t carry = rel, total = wt[CW * 4];
#pragma unroll
    for (uint32_t j = 0; j < CW; ++j) {
      pos[j] += wt[j * 4 + wv];
      const uint32_t wi = s0 + j * 256 + threadIdx.x;
      if (bprefix && wi < W) bp[wi] = carry + pos[j];
    }
    // ids through LDS, in rounds of STAGE_IDS output positions when the
    // segment holds more, written back coalesced
    for (uint32_t base = 0; base < total; base += STAGE_IDS) {
      const uint32_t lim = base + STAGE_IDS;
#pragma unroll
      for (uint32_t j = 0; j < CW; ++j) {
        const uint32_t pc = __popc(w[j]);
        if (pos[j] + pc > base && pos[j] < lim) {
          const uint32_t id0 = (s0 + j * 256 + threadIdx.x) * 32;
          uint32_t p = pos[j];
          for (uint32_t x = w[j]; x; x &= x - 1, ++p)
            if (p >= base && p < lim) stage[p - base] = id0 + (uint32_t)(__ffs(x) - 1);
        }
      }
      __syncthreads();
      const uint32_t n = min(STAGE_IDS, total - base);
      for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) out[carry + base + i] = stage[i];
      __syncthreads();
    }
    // every thread has read wt (and stage): the last round ends with a
    // barrier, and a segment without set bits has none
    if (total == 0) __syncthreads();
    if (threadIdx.x == 0) rel = carry + total;  // read after the next segment's first barrier
#pragma unroll
    for (uint32_t j = 0; j < CW; ++j) w[j] = nx[j];
  }
}

// Exclusive scan of generic u32 arrays (wrapping u32 values, u64 total) in one
// pass: a workgroup takes the next tile (a counter, so that every tile before
// its own is taken by a workgroup that runs), publishes the tile's sum, adds up
// the tiles before it - 64 at a time, back to the first that has published its
// inclusive sum - and publishes its own.  It waits only for tiles taken before
// its own, whose sums are published before anything is waited for.
// A state is one word (2 bits what it holds, 62 bits of sum: at most 2^30
// values of 32 bits a launch), read and written whole at agent scope.
// The sums first and the tiles in a second pass read everything twice: 95 +
// 14 + 119 us for 1e8 values, 245 us with the call; in one pass 217 us.  The
// known sum moves on by the 64 tiles of one look per exchange of states across
// the XCDs, about 1.4 us, so tiles are large: 271 us with 8192 values, 228 with
// 16384, 217 with 32768, 255 with 49152 (too few waves).  Looking at 128 or 256
// tiles at a time is slower (233, 241 us at 16384): more reads of the states
// that others write.
constexpr uint32_t SCAN_NT = 1024, SCAN_QUADS = 8;
constexpr uint32_t SCAN_TILE = SCAN_NT * SCAN_QUADS * 4;
constexpr uint64_t SCAN_MOST = 1ull << 30;  // values a launch
constexpr unsigned long long ST_SUM = 1ull << 62, ST_INCL = 2ull << 62, ST_VALUE = ST_SUM - 1;

// Before the states in scratch: the tile counter, the sum of earlier launches.
struct ScanHead {
  unsigned int next, pad;
  unsigned long long carry;
};

__device__ __forceinline__ uint4 load_quad(const uint32_t* in, uint64_t i, uint64_t n, bool wide) {
  if (wide && i + 4 <= n) return *reinterpret_cast<const uint4*>(in + i);
  uint4 v;
  v.x = i < n ? in[i] : 0u;
  v.y = i + 1 < n ? in[i + 1] : 0u;
  v.z = i + 2 < n ? in[i + 2] : 0u;
  v.w = i + 3 < n ? in[i + 3] : 0u;
  return v;
}

// wide: in and out are 16-byte aligned.  first: no earlier launch's sum.
__global__ void __launch_bounds__(SCAN_NT) scan_kernel(const uint32_t* in, uint32_t* out, uint64_t n, bool wide,
                                                       bool first, ScanHead* head,
                                                       unsigned long long* __restrict__ state,
                                                       unsigned long long* __restrict__ total) {
  constexpr uint32_t NW = SCAN_NT / WAVE;
  __shared__ uint32_t wt[SCAN_QUADS * NW];  // (quad k, wave w) totals at k * NW + w, then their offsets
  __shared__ unsigned long long part[NW], before;
  __shared__ uint32_t taken;
  const uint32_t lane = lane_id(), w = threadIdx.x / WAVE;
  if (threadIdx.x == 0) taken = gridDim.x > 1 ? atomicAdd(&head->next, 1u) : 0u;
  __syncthreads();
  const uint32_t tile = taken;
  const uint64_t base = (uint64_t)tile * SCAN_TILE;
  uint4 v[SCAN_QUADS];
#pragma unroll
  for (uint32_t k = 0; k < SCAN_QUADS; ++k)
    v[k] = load_quad(in, base + ((uint64_t)k * SCAN_NT + threadIdx.x) * 4, n, wide);
  unsigned long long mine = 0;
  uint32_t ex[SCAN_QUADS];
#pragma unroll
  for (uint32_t k = 0; k < SCAN_QUADS; ++k) {
    mine += (unsigned long long)v[k].x + v[k].y + ((unsigned long long)v[k].z + v[k].w);
    const uint32_t s = v[k].x + v[k].y + v[k].z + v[k].w, incl = wave_incl_scan(s);
    if (lane == WAVE - 1) wt[k * NW + w] = incl;
    ex[k] = incl - s;
  }
  mine = wave_sum64(mine);
  if (lane == 0) part[w] = mine;
  __syncthreads();
  if (w == 0) {
    static_assert(SCAN_QUADS * NW % WAVE == 0, "one wave scans the (quad, wave) totals");
    uint32_t run = 0;
#pragma unroll
    for (uint32_t c = 0; c < SCAN_QUADS * NW; c += WAVE) {
      const uint32_t x = wt[c + lane], incl = wave_incl_scan(x);
      wt[c + lane] = run + incl - x;
      run += __shfl(incl, WAVE - 1, WAVE);
    }
    unsigned long long sum = 0;
    for (uint32_t i = 0; i < NW; ++i) sum += part[i];
    unsigned long long excl = 0;
    if (gridDim.x > 1) {
      if (lane == 0)
        __hip_atomic_store(&state[tile], (tile ? ST_SUM : ST_INCL) | sum, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      for (uint32_t hi = tile; hi > 0;) {  // tiles below hi are still to be added
        const unsigned long long st =
            lane < hi ? __hip_atomic_load(&state[hi - 1 - lane], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : ST_INCL;
        const unsigned long long incl_at = __ballot((st & ST_INCL) != 0), none = __ballot(st == 0);
        // lanes up to the first inclusive sum count
        const unsigned long long use = incl_at ? (incl_at & (0ull - incl_at)) * 2 - 1 : ~0ull;
        if (none & use) {
          __builtin_amdgcn_s_sleep(1);
          continue;
        }
        excl += wave_sum64((use >> lane) & 1 ? st & ST_VALUE : 0ull);
        hi = incl_at ? 0u : hi - WAVE;
      }
      if (tile && lane == 0)
        __hip_atomic_store(&state[tile], ST_INCL | (excl + sum), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    const unsigned long long carry = first ? 0ull : head->carry;
    if (lane == 0) {
      before = carry + excl;
      if (tile == gridDim.x - 1 && total) *total = carry + excl + sum;
    }
  }
  __syncthreads();
  const uint32_t off = (uint32_t)before;
#pragma unroll
  for (uint32_t k = 0; k < SCAN_QUADS; ++k) {
    const uint64_t i = base + ((uint64_t)k * SCAN_NT + threadIdx.x) * 4;
    uint4 o;
    o.x = off + wt[k * NW + w] + ex[k];
    o.y = o.x + v[k].x;
    o.z = o.y + v[k].y;
    o.w = o.z + v[k].z;
    if (wide && i + 4 <= n) {
      *reinterpret_cast<uint4*>(out + i) = o;
    } else {
      if (i < n) out[i] = o.x;
      if (i + 1 < n) out[i + 1] = o.y;
      if (i + 2 < n) out[i + 2] = o.z;
      if (i + 3 < n) out[i + 3] = o.w;
    }
  }
}

// The sum so far is carried to the next launch, whose tiles start over.
__global__ void scan_next_kernel(ScanHead* head, const unsigned long long* __restrict__ sum) {
  head->carry = *sum;
  head->next = 0;
}

__global__ void fill_u32_kernel(uint32_t* __restrict__ p, uint32_t v, uint64_t n) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) p[i] = v;
}

}  // namespace

// Fill kernel instead of hipMemsetAsync so that captured graphs hold only
// kernel nodes.
void launch_fill_u32(uint32_t* p, uint32_t v, uint64_t n, hipStream_t s) {
  if (!n) return;
  uint64_t grid = (n + 255) / 256;
  if (grid > 8192) grid = 8192;
  hipLaunchKernelGGL(fill_u32_kernel, dim3((uint32_t)grid), dim3(256), 0, s, p, v, n);
}

void launch_row_popcount(const DevGraph& g, const uint32_t* bitmaps, uint32_t nrows, uint32_t* segc,
                         uint32_t* counts, hipStream_t s) {
  if (!nrows) return;
  const uint32_t nseg = segs_of(g.W);
  hipLaunchKernelGGL(seg_popcount_kernel, dim3(nrows * nseg), dim3(256), 0, s, bitmaps, g.W, nseg, segc);
  hipLaunchKernelGGL(seg_offsets_kernel, dim3(nrows), dim3(256), 0, s, segc, nseg, counts);
}

void launch_compact_rows(const DevGraph& g, const uint32_t* bitmaps, uint32_t nrows, const uint32_t* segc,
                         const uint64_t* coff, uint32_t* clist, uint32_t* bprefix, hipStream_t s) {
  if (!nrows) return;
  const uint32_t nseg = segs_of(g.W);
  const uint32_t ngrp = (nseg + COMPACT_GROUP - 1) / COMPACT_GROUP;
  hipLaunchKernelGGL(compact_rows_kernel, dim3(nrows * ngrp), dim3(256), 0, s, bitmaps, g.W, nseg, segc, coff,
                     clist, bprefix);
}

namespace {
uint64_t scan_tiles(uint64_t n) { return (std::min(n, SCAN_MOST) + SCAN_TILE - 1) / SCAN_TILE; }
constexpr uint64_t kScanHead = (sizeof(ScanHead) + sizeof(unsigned long long)) / sizeof(uint32_t);  // and a total
}  // namespace

uint64_t scan_scratch_words(uint64_t n) { return kScanHead + 2 * scan_tiles(n); }

void launch_exclusive_scan(const uint32_t* in, uint32_t* out, uint64_t n, unsigned long long* total,
                           uint32_t* scratch, uint64_t scratch_words, hipStream_t s) {
  if (!n || scratch_words < scan_scratch_words(n)) return;
  ScanHead* head = reinterpret_cast<ScanHead*>(scratch);
  unsigned long long* sum = reinterpret_cast<unsigned long long*>(head + 1);
  unsigned long long* state = sum + 1;
  const bool wide = ((reinterpret_cast<uintptr_t>(in) | reinterpret_cast<uintptr_t>(out)) & 15) == 0;
  for (uint64_t at = 0; at < n; at += SCAN_MOST) {
    const uint64_t m = std::min(SCAN_MOST, n - at), tiles = scan_tiles(m);
    const bool last = at + m == n;
    if (at) {
      hipLaunchKernelGGL(scan_next_kernel, dim3(1), dim3(1), 0, s, head, sum);
      launch_fill_u32(reinterpret_cast<uint32_t*>(state), 0u, 2 * tiles, s);
    } else if (tiles > 1) {
      launch_fill_u32(scratch, 0u, kScanHead + 2 * tiles, s);
    }
    hipLaunchKernelGGL(scan_kernel, dim3((uint32_t)tiles), dim3(SCAN_NT), 0, s, in + at, out + at, m, wide, at == 0,
                       head, state, last ? total : sum);
  }
}

uint64_t compact_scratch_words(uint64_t nbits) {
  const uint64_t W = (nbits + 31) / 32;
  return 2 + segs_of((uint32_t)W) + 1;
}

void launch_compact_bitmap(const uint32_t* bits, uint64_t nbits, uint32_t* ids, unsigned long long* count,
                           uint32_t* scratch, hipStream_t s) {
  // one row of ceil(nbits/32) words through the row compaction; scratch
  // holds the row offset (2 words), the segment counts and the row count
  DevGraph g;
  g.W = (uint32_t)((nbits + 31) / 32);
  uint64_t* coff = reinterpret_cast<uint64_t*>(scratch);
  uint32_t* segc = scratch + 2;
  uint32_t* rowc = segc + segs_of(g.W);
  hipMemsetAsync(coff, 0, sizeof(uint64_t), s);
  launch_row_popcount(g, bits, 1, segc, rowc, s);
  launch_compact_rows(g, bits, 1, segc, coff, ids, nullptr, s);
  hipMemsetAsync(count, 0, sizeof(unsigned long long), s);
  hipMemcpyAsync(count, rowc, sizeof(uint32_t), hipMemcpyDeviceToDevice, s);
}

}  // namespace gpsm
