// Candidate-edge tables on gfx950 (count_kernel + thrust::exclusive_scan +
// examine_kernel, match/Match.cu:892-1139).  CET(x -> w) lists, for each
// mu in C(x) ascending, the data neighbours of mu that are in C(w), in
// adjacency (ascending) order.
//
// One wave per 64 candidates of C(x): some of the first, which on a power-law
// graph are the hubs, spread over the table's waves, and runs of consecutive
// ones (cand_index).  The wave walks the concatenated adjacency of its
// candidates towards w's label (DevGraph::lrow: C(w) holds no vertex of
// another) 64 entries per step (balanced across hub and leaf candidates) and
// tests C(w) membership in the bitmap.  Outputs are per candidate (its
// count, its list at its offset), so the assignment does not change them.
// The write pass ranks each hit inside its candidate's run with a ballot,
// so lists stay in adjacency order without a second scan.
#include "launch.h"
#include "wave.h"

namespace gpsm {

namespace {

constexpr int CET_UNROLL = 4;  // adjacency entries in flight per lane

struct CetLds {
  uint32_t pre[WAVE + 1];
  uint32_t off[WAVE];
  uint32_t cnt[WAVE];
};

// Optional work counters (profiling), per lane: of cet_count and cet_write the
// candidates loaded, of all but cet_agg the adjacency entries examined, bitmap
// probes, list entries written; cet_sum's candidates; cet_agg's candidates,
// list entries and records read.  One atomic per counter per workgroup into
// copy blockIdx % STAT_COPIES of stats.
constexpr int CET_STATS = 8;
static_assert(CET_STATS <= STAT_STRIDE, "a copy's counters");
struct CetTally {
  uint32_t cand = 0, ent = 0, probe = 0, wrote = 0, sums = 0, aggs = 0, items = 0, recs = 0;
};

__device__ __forceinline__ void flush_tally(const CetTally& t, unsigned long long* stats) {
  __shared__ unsigned long long red[4][CET_STATS];
  const unsigned long long v[CET_STATS] = {wave_sum64(t.cand), wave_sum64(t.ent),  wave_sum64(t.probe),
                                           wave_sum64(t.wrote), wave_sum64(t.sums), wave_sum64(t.aggs),
                                           wave_sum64(t.items), wave_sum64(t.recs)};
  const uint32_t w = threadIdx.x / WAVE;
  if (lane_id() == 0)
    for (int i = 0; i < CET_STATS; ++i) red[w][i] = v[i];
  __syncthreads();
  if (threadIdx.x < CET_STATS) {
    unsigned long long tot = 0;
    for (uint32_t x = 0; x < blockDim.x / WAVE; ++x) tot += red[x][threadIdx.x];
    if (tot) atomicAdd(stats + (blockIdx.x % STAT_COPIES) * STAT_STRIDE + threadIdx.x, tot);
  }
}

// Chunk j of a table with nch chunks holds every nch-th of the first CET_RUN *
// nch candidates (the hubs of a graph whose ids descend by degree are among
// them, and one piece of theirs can hold thousands of entries), and of the rest
// runs of CET_RUN consecutive ones, whose pieces are next to each other.
constexpr uint32_t CET_RUN = 16;
__device__ __forceinline__ uint32_t cand_index(uint32_t j, uint32_t nch, uint32_t lane) {
  const uint32_t r = lane / CET_RUN;
  return r == 0 ? j + lane * nch : (CET_RUN + (r - 1) * CET_RUN) * nch + j * CET_RUN + lane % CET_RUN;
}

__device__ __forceinline__ void load_chunk(const Pieces& pieces, const uint32_t* __restrict__ clist,
                                           const CetDesc& d, uint32_t j, uint32_t nch, CetLds& L, bool& mine,
                                           uint32_t& D) {
  const uint32_t lane = lane_id();
  const uint32_t ci = cand_index(j, nch, lane);
  mine = ci < d.ncand;
  const uint32_t id = mine ? clist[d.clist_off + ci] : 0u;
  uint32_t off = 0, deg = 0;
  if (mine) piece(pieces, id, d.w_lo, off, deg);
  const uint32_t incl = wave_incl_scan(deg);
  D = uniform(__shfl(incl, WAVE - 1, WAVE));
  L.pre[lane] = incl - deg;
  L.off[lane] = off;
  L.cnt[lane] = 0;
  wave_sync();
}

// Eight waves per SIMD (64 VGPRs, no spill; seven at the compiler's own
// choice): 9-11% faster on the 1M Chung-Lu mix and the R-MAT 22 shapes.
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(8))) cet_count_kernel(Pieces pieces, const uint32_t* __restrict__ col,
                                                        const uint32_t* __restrict__ bitmaps, uint32_t W,
                                                        const uint32_t* __restrict__ clist, CetDesc* descs,
                                                        const uint32_t* __restrict__ chunk_base, uint32_t ndesc,
                                                        uint32_t* __restrict__ offsets,
                                                        unsigned long long* __restrict__ stats) {
  __shared__ CetLds lds[4];
  CetTally tl;
  CetLds& L = lds[threadIdx.x / WAVE];
  const uint32_t lane = lane_id();
  const uint32_t wave = (blockIdx.x * blockDim.x + threadIdx.x) / WAVE;
  const uint32_t nwaves = (gridDim.x * blockDim.x) / WAVE;
  const uint32_t nitems = chunk_base[ndesc];
  for (uint32_t it = wave; it < nitems; it += nwaves) {
    const uint32_t di = uniform(seg_search(chunk_base, ndesc + 1, it));
    const CetDesc d = descs[di];
    const uint32_t j = it - chunk_base[di], nch = chunk_base[di + 1] - chunk_base[di];
    bool mine;
    uint32_t D;
    load_chunk(pieces, clist, d, j, nch, L, mine, D);
    tl.cand += mine;
    const uint32_t* bm_w = bitmaps + (size_t)d.w_slot * W;
    uint32_t tot = 0;
    for (uint32_t f = 0; f < D; f += WAVE * CET_UNROLL) {
      // CET_UNROLL entries per lane: all adjacency loads, then their probes
      uint32_t cis[CET_UNROLL], mvs[CET_UNROLL], es[CET_UNROLL];
#pragma unroll
      for (int u = 0; u < CET_UNROLL; ++u) cis[u] = f + u * WAVE + lane;
      halving_search<CET_UNROLL>(L.pre, WAVE, cis);
#pragma unroll
      for (int u = 0; u < CET_UNROLL; ++u) es[u] = L.off[cis[u]] + (f + u * WAVE + lane - L.pre[cis[u]]);
#pragma unroll
      for (int u = 0; u < CET_UNROLL; ++u) {
        if (f + u * WAVE + lane < D) {
          mvs[u] = col[es[u]];
        } else {
          cis[u] = WAVE;
        }
      }
      // the probes' bitmap words loaded together, then tested
      uint32_t pw[CET_UNROLL];
#pragma unroll
      for (int u = 0; u < CET_UNROLL; ++u)
        pw[u] = cis[u] != WAVE ? bm_w[mvs[u] >> 5] >> (mvs[u] & 31) : 0u;
      if (stats) {
#pragma unroll
        for (int u = 0; u < CET_UNROLL; ++u) {
          tl.ent += cis[u] != WAVE;
          tl.probe += cis[u] != WAVE;
        }
      }
#pragma unroll
      for (int u = 0; u < CET_UNROLL; ++u)
        if (pw[u] & 1u) {
          ++tot;
          atomicAdd(&L.cnt[cis[u]], 1u);
        }
    }
    wave_sync();
    if (mine) offsets[d.off_base + cand_index(j, nch, lane)] = L.cnt[lane];
    tot = wave_sum(tot);
    if (lane == 0 && tot) atomicAdd(reinterpret_cast<unsigned long long*>(&descs[di].total), (unsigned long long)tot);
    wave_sync();
  }
  if (stats) flush_tally(tl, stats);
}

// One workgroup per table scans its per-candidate counts in place, in tiles
// of 256 x OFF_ITEMS: each thread sums OFF_ITEMS consecutive counts (loads
// in flight together), one block scan places the thread sums, and each
// thread writes its run.  A table of 10^5 candidates takes 49 tiles instead
// of 391 block scans of 256.
constexpr uint32_t OFF_ITEMS = 8;

__global__ void __launch_bounds__(256) cet_offsets_kernel(const CetDesc* __restrict__ descs,
                                                          uint32_t* __restrict__ offsets) {
  __shared__ uint32_t tmp[8];
  const CetDesc d = descs[blockIdx.x];
  uint32_t* o = offsets + d.off_base;
  uint32_t carry = 0;
  for (uint32_t t0 = 0; t0 < d.ncand; t0 += blockDim.x * OFF_ITEMS) {
    const uint32_t i0 = t0 + threadIdx.x * OFF_ITEMS;
    uint32_t v[OFF_ITEMS], sum = 0;
#pragma unroll
    for (uint32_t j = 0; j < OFF_ITEMS; ++j) {
      v[j] = i0 + j < d.ncand ? o[i0 + j] : 0u;
      sum += v[j];
    }
    uint32_t total;
    uint32_t run = carry + block_excl_scan(sum, tmp, &total);
#pragma unroll
    for (uint32_t j = 0; j < OFF_ITEMS; ++j) {
      if (i0 + j < d.ncand) o[i0 + j] = min(run, d.list_cap);
      run += v[j];
    }
    carry += total;
  }
  if (threadIdx.x == 0) o[d.ncand] = min(carry, d.list_cap);
}

__global__ void __launch_bounds__(256) cet_write_kernel(Pieces pieces, const uint32_t* __restrict__ col,
                                                        const uint32_t* __restrict__ bitmaps, uint32_t W,
                                                        const uint32_t* __restrict__ clist,
                                                        const CetDesc* __restrict__ descs,
                                                        const uint32_t* __restrict__ chunk_base, uint32_t ndesc,
                                                        const uint32_t* __restrict__ offsets,
                                                        uint32_t* __restrict__ lists,
                                                        unsigned long long* __restrict__ stats) {
  __shared__ CetLds lds[4];
  CetTally tl;
  CetLds& L = lds[threadIdx.x / WAVE];
  const uint32_t lane = lane_id();
  const uint32_t wave = (blockIdx.x * blockDim.x + threadIdx.x) / WAVE;
  const uint32_t nwaves = (gridDim.x * blockDim.x) / WAVE;
  const uint32_t nitems = chunk_base[ndesc];
  for (uint32_t it = wave; it < nitems; it += nwaves) {
    const uint32_t di = uniform(seg_search(chunk_base, ndesc + 1, it));
    const CetDesc d = descs[di];
    const uint32_t j = it - chunk_base[di], nch = chunk_base[di + 1] - chunk_base[di];
    bool mine;
    uint32_t D;
    load_chunk(pieces, clist, d, j, nch, L, mine, D);
    tl.cand += mine;
    // each lane's list starts at its candidate's offset; cnt advances it
    L.cnt[lane_id()] = mine ? offsets[d.off_base + cand_index(j, nch, lane_id())] : 0u;
    wave_sync();
    const uint32_t* bm_w = bitmaps + (size_t)d.w_slot * W;
    uint32_t* out = lists + d.list_base;
    for (uint32_t f = 0; f < D; f += WAVE * CET_UNROLL) {
      // CET_UNROLL sub-steps of 64 entries: all adjacency loads, their probes,
      // then the writes sub-step by sub-step (lists stay in adjacency order)
      uint32_t cis[CET_UNROLL], mvs[CET_UNROLL];
      bool hits[CET_UNROLL];
      uint32_t es[CET_UNROLL];
#pragma unroll
      for (int u = 0; u < CET_UNROLL; ++u) cis[u] = f + u * WAVE + lane;
      halving_search<CET_UNROLL>(L.pre, WAVE, cis);
#pragma unroll
      for (int u = 0; u < CET_UNROLL; ++u) es[u] = L.off[cis[u]] + (f + u * WAVE + lane - L.pre[cis[u]]);
#pragma unroll
      for (int u = 0; u < CET_UNROLL; ++u) {
        mvs[u] = 0;
        hits[u] = false;
        if (f + u * WAVE + lane < D) mvs[u] = col[es[u]];
      }
      // the probes' bitmap words loaded together, then tested
      uint32_t pw[CET_UNROLL];
#pragma unroll
      for (int u = 0; u < CET_UNROLL; ++u)
        pw[u] = f + u * WAVE + lane < D ? bm_w[mvs[u] >> 5] >> (mvs[u] & 31) : 0u;
#pragma unroll
      for (int u = 0; u < CET_UNROLL; ++u) hits[u] = (pw[u] & 1u) != 0;
      if (stats) {
#pragma unroll
        for (int u = 0; u < CET_UNROLL; ++u) {
          tl.ent += f + u * WAVE + lane < D;
          tl.probe += f + u * WAVE + lane < D;
        }
      }
#pragma unroll
      for (int u = 0; u < CET_UNROLL; ++u) {
        const uint32_t fu = f + u * WAVE, ci = cis[u];
        const unsigned long long hm = __ballot(hits[u]);
        if (hits[u]) {
          // lanes of this sub-step that belong to candidate ci start at seg_lo
          const uint32_t seg_lo = L.pre[ci] > fu ? L.pre[ci] - fu : 0u;
          const unsigned long long below = (lane ? (~0ULL >> (WAVE - lane)) : 0ULL) & (~0ULL << seg_lo);
          const uint32_t rank = __popcll(hm & below);
          const uint32_t pos = L.cnt[ci] + rank;
          if (pos < d.list_cap) {
            out[pos] = mvs[u];
            ++tl.wrote;
          }
        }
        wave_sync();
        if (hits[u]) atomicAdd(&L.cnt[ci], 1u);
        wave_sync();
      }
    }
  }
  if (stats) flush_tally(tl, stats);
}

// cell[seg] += x for every lane, lanes of one seg consecutive (seg
// non-decreasing over the wave's lanes, all active): one wave scan, then two
// LDS atomics per segment boundary, whatever the segments' lengths.
__device__ __forceinline__ void seg_add(unsigned long long* cell, uint32_t seg, bool tail, uint32_t next,
                                        unsigned long long x) {
  const unsigned long long incl = wave_incl_scan64(x);
  if (tail) {
    atomicAdd(&cell[seg], incl);
    if (next != WAVE) atomicAdd(&cell[next], 0ull - incl);
  }
}

// Records of the last join levels' tables: one wave per 64 candidates of
// C(x) (cand_index), flattened over their adjacency as in cet_count, but an
// entry in C(w) adds its hash term (computed here, about 30 VALU
// instructions, only in lanes with a hit) to its candidate's sum and is not
// written: the join reads 32 bytes per candidate instead of 12 per list
// entry.  Bound by the random probes of C(w), like cet_count.
struct SumLds {
  CetLds c;
  unsigned long long s[WAVE];
};

__global__ void __launch_bounds__(256) cet_sum_kernel(Pieces pieces, const uint32_t* __restrict__ col,
                                                      const uint32_t* __restrict__ ids,
                                                      const uint32_t* __restrict__ bitmaps, uint32_t W,
                                                      const uint32_t* __restrict__ clist,
                                                      const CetDesc* __restrict__ descs,
                                                      const uint32_t* __restrict__ chunk_base, uint32_t ndesc,
                                                      CetAgg* __restrict__ aggs,
                                                      unsigned long long* __restrict__ stats) {
  __shared__ SumLds lds[4];
  CetTally tl;
  SumLds& L = lds[threadIdx.x / WAVE];
  const uint32_t lane = lane_id();
  const uint32_t wave = (blockIdx.x * blockDim.x + threadIdx.x) / WAVE;
  const uint32_t nwaves = (gridDim.x * blockDim.x) / WAVE;
  const uint32_t nitems = chunk_base[ndesc];
  for (uint32_t it = wave; it < nitems; it += nwaves) {
    const uint32_t di = uniform(seg_search(chunk_base, ndesc + 1, it));
    const CetDesc d = descs[di];
    const uint32_t j = it - chunk_base[di], nch = chunk_base[di + 1] - chunk_base[di];
    bool mine;
    uint32_t D;
    L.s[lane] = 0;
    load_chunk(pieces, clist, d, j, nch, L.c, mine, D);
    tl.sums += mine;
    const uint32_t* bm_w = bitmaps + (size_t)d.w_slot * W;
    for (uint32_t f = 0; f < D; f += WAVE * CET_UNROLL) {
      uint32_t cis[CET_UNROLL], mvs[CET_UNROLL], pw[CET_UNROLL];
#pragma unroll
      for (int u = 0; u < CET_UNROLL; ++u) cis[u] = f + u * WAVE + lane;
      halving_search<CET_UNROLL>(L.c.pre, WAVE, cis);  // an index past D falls in the last candidate
#pragma unroll
      for (int u = 0; u < CET_UNROLL; ++u) {
        const uint32_t g = f + u * WAVE + lane;
        const uint32_t e = L.c.off[cis[u]] + (g - L.c.pre[cis[u]]);
        mvs[u] = g < D ? col[e] : 0u;
      }
#pragma unroll
      for (int u = 0; u < CET_UNROLL; ++u) {
        const bool in = f + u * WAVE + lane < D;
        pw[u] = in ? bm_w[mvs[u] >> 5] >> (mvs[u] & 31) : 0u;
        if (stats) {
          tl.ent += in;
          tl.probe += in;
        }
      }
#pragma unroll
      for (int u = 0; u < CET_UNROLL; ++u) {
        const bool hit = (pw[u] & 1u) != 0;
        const unsigned long long hm = __ballot(hit);
        if (!hm) continue;  // the whole wave
        const uint32_t fu = f + u * WAVE, ci = cis[u];
        const uint32_t next = __shfl_down(ci, 1, WAVE);
        const bool tail = lane == WAVE - 1 || next != ci;
        seg_add(L.s, ci, tail, lane == WAVE - 1 ? (uint32_t)WAVE : next, hit ? tuple_term(d.term_qid, ids[mvs[u]]) : 0ull);
        if (tail) {
          const uint32_t seg_lo = L.c.pre[ci] > fu ? L.c.pre[ci] - fu : 0u;
          if (seg_lo < WAVE) {
            const unsigned long long seg = (~0ULL << seg_lo) & (~0ULL >> (WAVE - 1 - lane));
            atomicAdd(&L.c.cnt[ci], (uint32_t)__popcll(hm & seg));
          }
        }
      }
    }
    wave_sync();
    if (mine) {
      CetAgg r;
      r.s = L.s[lane];
      r.a = r.b = 0;
      r.off = 0;
      r.len = L.c.cnt[lane];
      aggs[d.agg_base + cand_index(j, nch, lane)] = r;
    }
    wave_sync();
  }
  if (stats) flush_tally(tl, stats);
}

// Records of the level before the last: one wave per 64 candidates
// (cand_index), flattened over their lists.  A list entry costs its hash term and,
// where w's parent is the entry itself (AGG_CHAIN), its rank in C(y) and its
// 32-byte record of the last table.
constexpr int AGG_UNROLL = 2;  // list entries in flight per lane

struct AggLds {
  uint32_t pre[WAVE];
  uint32_t off[WAVE];
  unsigned long long s[WAVE], a[WAVE], b[WAVE];
};

// STATS: with the work counters, whose registers the timed variant keeps free.
template <bool STATS>
__global__ void __launch_bounds__(256) cet_agg_kernel(const uint32_t* __restrict__ ids,
                                                      const uint32_t* __restrict__ bitmaps,
                                                      const uint32_t* __restrict__ bprefix, uint32_t W,
                                                      const AggDesc* __restrict__ descs, uint32_t ndesc,
                                                      const uint32_t* __restrict__ chunk_base,
                                                      const uint32_t* __restrict__ offsets,
                                                      const uint32_t* __restrict__ lists, CetAgg* aggs,
                                                      unsigned long long* __restrict__ stats) {
  __shared__ AggLds lds[4];
  CetTally tl;
  AggLds& L = lds[threadIdx.x / WAVE];
  const uint32_t lane = lane_id();
  const uint32_t wave = (blockIdx.x * blockDim.x + threadIdx.x) / WAVE;
  const uint32_t nwaves = (gridDim.x * blockDim.x) / WAVE;
  const uint32_t nitems = chunk_base[ndesc];
  for (uint32_t it = wave; it < nitems; it += nwaves) {
    const uint32_t di = uniform(seg_search(chunk_base, ndesc + 1, it));
    const AggDesc d = descs[di];
    const uint32_t j = it - chunk_base[di], nch = chunk_base[di + 1] - chunk_base[di];
    const uint32_t ci = cand_index(j, nch, lane);
    const bool mine = ci < d.ncand;
    const uint32_t off = mine ? offsets[d.off_base + ci] : 0u;
    const uint32_t len = mine ? offsets[d.off_base + ci + 1] - off : 0u;
    const uint32_t incl = wave_incl_scan(len);
    const uint32_t D = uniform(__shfl(incl, WAVE - 1, WAVE));
    if (STATS) {
      tl.aggs += mine;
      tl.items += len;
      if (d.mode == AGG_CHAIN) tl.recs += len;
      if (d.mode == AGG_SIBLING) tl.probe += len;
    }
    L.pre[lane] = incl - len;
    L.off[lane] = off;
    L.s[lane] = L.a[lane] = L.b[lane] = 0;
    wave_sync();
    const uint32_t* bm_y = bitmaps + (size_t)d.y_slot * W;
    const uint32_t* bp_y = bprefix + (size_t)d.y_slot * W;
    const uint32_t* bm_w = bitmaps + (size_t)d.w_slot * W;
    const uint32_t* lst = lists + d.list_base;
    for (uint32_t f = 0; f < D; f += WAVE * AGG_UNROLL) {
      uint32_t cis[AGG_UNROLL], v[AGG_UNROLL];
      unsigned long long t[AGG_UNROLL], xa[AGG_UNROLL], xb[AGG_UNROLL];
#pragma unroll
      for (int u = 0; u < AGG_UNROLL; ++u) cis[u] = f + u * WAVE + lane;
      halving_search<AGG_UNROLL>(L.pre, WAVE, cis);
#pragma unroll
      for (int u = 0; u < AGG_UNROLL; ++u) {
        // an index past D (in the last candidate) reads no entry and adds
        // nothing; vertex 0 stands in for it (C(y) is not empty, so rank 0
        // has a record)
        const uint32_t g = f + u * WAVE + lane;
        v[u] = g < D ? lst[L.off[cis[u]] + (g - L.pre[cis[u]])] : 0u;
      }
#pragma unroll
      for (int u = 0; u < AGG_UNROLL; ++u) {
        const bool in = f + u * WAVE + lane < D;
        const uint32_t id = ids[v[u]];
        xa[u] = xb[u] = 0;
        if (d.mode == AGG_CHAIN) {  // uniform
          const CetAgg r = aggs[d.w_agg_base + rank_of(bm_y, bp_y, v[u])];
          xa[u] = in ? r.len : 0u;
          xb[u] = in ? r.s : 0ull;
        } else if (d.mode == AGG_SIBLING) {
          const bool hit = in && bit_of(bm_w, v[u]);
          xa[u] = hit;
          xb[u] = hit ? tuple_term(d.w_qid, id) : 0ull;
        }
        t[u] = in ? tuple_term(d.y_qid, id) : 0ull;
        xb[u] *= t[u];
      }
#pragma unroll
      for (int u = 0; u < AGG_UNROLL; ++u) {
        if (f + u * WAVE >= D) continue;  // uniform
        const uint32_t next = __shfl_down(cis[u], 1, WAVE);
        const bool tail = lane == WAVE - 1 || next != cis[u];
        const uint32_t nx = lane == WAVE - 1 ? (uint32_t)WAVE : next;
        seg_add(L.s, cis[u], tail, nx, t[u]);
        if (d.mode != AGG_SUM) {
          seg_add(L.a, cis[u], tail, nx, xa[u]);
          seg_add(L.b, cis[u], tail, nx, xb[u]);
        }
      }
    }
    wave_sync();
    if (mine) {
      CetAgg r;
      r.s = L.s[lane];
      r.a = L.a[lane];
      r.b = L.b[lane];
      r.off = off;
      r.len = len;
      aggs[d.agg_base + ci] = r;
    }
    wave_sync();
  }
  if constexpr (STATS) flush_tally(tl, stats);
}

// One thread per term: the table by a binary search over the term ranges.
__global__ void __launch_bounds__(256) cet_terms_kernel(const uint32_t* __restrict__ ids,
                                                        const uint32_t* __restrict__ lists,
                                                        const CetDesc* __restrict__ descs,
                                                        const uint32_t* __restrict__ term_desc,
                                                        const uint64_t* __restrict__ term_start, uint32_t nd,
                                                        uint64_t nterms, unsigned long long* __restrict__ terms) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; t < nterms; t += stride) {
    uint32_t lo = 0, hi = nd;  // last range with start <= t
    while (hi - lo > 1) {
      const uint32_t mid = (lo + hi) >> 1;
      if (term_start[mid] <= t) lo = mid;
      else hi = mid;
    }
    const CetDesc& d = descs[term_desc[lo]];
    const uint64_t e = t - term_start[lo];
    terms[t] = e < d.list_cap ? tuple_term(d.term_qid, ids[lists[d.list_base + e]]) : 0ull;
  }
}

}  // namespace

void launch_cet_count(const DevGraph& g, const uint32_t* bitmaps, const uint32_t* clist, CetDesc* descs,
                      uint32_t ndesc, uint32_t* offsets, const uint32_t* chunk_base, uint32_t grid, hipStream_t s,
                      unsigned long long* stats) {
  if (!ndesc) return;
  hipLaunchKernelGGL(cet_count_kernel, dim3(grid), dim3(256), 0, s, pieces_of(g), g.col, bitmaps, g.W, clist,
                     descs, chunk_base, ndesc, offsets, stats);
}

void launch_cet_offsets(CetDesc* descs, uint32_t ndesc, uint32_t* offsets, hipStream_t s) {
  if (!ndesc) return;
  hipLaunchKernelGGL(cet_offsets_kernel, dim3(ndesc), dim3(256), 0, s, descs, offsets);
}

void launch_cet_terms(const DevGraph& g, const uint32_t* lists, const CetDesc* descs, const uint32_t* term_desc,
                      const uint64_t* term_start, uint32_t nterm_desc, uint64_t nterms, unsigned long long* terms,
                      hipStream_t s) {
  if (!nterm_desc || !nterms) return;
  uint64_t grid = (nterms + 255) / 256;
  if (grid > 16384) grid = 16384;
  hipLaunchKernelGGL(cet_terms_kernel, dim3((uint32_t)grid), dim3(256), 0, s, g.ids, lists, descs, term_desc, term_start,
                     nterm_desc, nterms, terms);
}

void launch_cet_sums(const DevGraph& g, const uint32_t* bitmaps, const uint32_t* clist, const CetDesc* descs,
                     uint32_t ndesc, const uint32_t* chunk_base, CetAgg* aggs, uint32_t grid, hipStream_t s,
                     unsigned long long* stats) {
  if (!ndesc) return;
  hipLaunchKernelGGL(cet_sum_kernel, dim3(grid), dim3(256), 0, s, pieces_of(g), g.col, g.ids, bitmaps, g.W, clist, descs,
                     chunk_base, ndesc, aggs, stats);
}

void launch_cet_aggs(const DevGraph& g, const uint32_t* bitmaps, const uint32_t* bprefix, const AggDesc* descs,
                     uint32_t ndesc, const uint32_t* chunk_base, const uint32_t* offsets, const uint32_t* lists,
                     CetAgg* aggs, uint32_t grid, hipStream_t s, unsigned long long* stats) {
  if (!ndesc) return;
  hipLaunchKernelGGL(stats ? cet_agg_kernel<true> : cet_agg_kernel<false>, dim3(grid), dim3(256), 0, s, g.ids, bitmaps, bprefix, g.W, descs, ndesc,
                     chunk_base, offsets, lists, aggs, stats);
}

void launch_cet_write(const DevGraph& g, const uint32_t* bitmaps, const uint32_t* clist, const CetDesc* descs,
                      uint32_t ndesc, const uint32_t* offsets, uint32_t* lists, const uint32_t* chunk_base, uint32_t grid,
                      hipStream_t s, unsigned long long* stats) {
  if (!ndesc) return;
  hipLaunchKernelGGL(cet_write_kernel, dim3(grid), dim3(256), 0, s, pieces_of(g), g.col, bitmaps, g.W, clist,
                     descs, chunk_base, ndesc, offsets, lists, stats);
}

}  // namespace gpsm
