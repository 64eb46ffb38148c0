// Candidate-vertex filtering on gfx950: the start vertex's label/degree check
// (check_kernel, match/Match.cu:431-461), exploration (explore_kernel,
// :528-659) and neighbourhood refinement (refine_kernel, :761-846), for any
// number of queries per launch.
//
// Layout: candidate sets are bitmaps (1 bit per data vertex, 32-bit words);
// the reference used one byte per (query vertex, data vertex).
// Parallel decomposition: one wave per (op, vertex range).  The ranges are
// fixed per data graph (DevGraph::fchunk): at most FCHUNK_VERTS vertices and
// FCHUNK_ENTRIES adjacency entries each, so a power-law graph's hubs (which a Chung-Lu or
// R-MAT generator gives the lowest ids) do not pile onto one wave.  The wave
// compacts the range's candidates into LDS (the reference's kernel_collect,
// fused), then, neighbour by neighbour of the query vertex, walks the entries
// of 64 candidates at a time towards that neighbour's label, concatenated,
// 64 entries per lane step (lane t takes entry t; a binary search in the 64
// prefix sums finds its candidate), so hub and leaf candidates share lanes
// evenly instead of one 32-lane warp per candidate.
#include <type_traits>

#include "launch.h"
#include "steps.h"
#include "wave.h"

namespace gpsm {

namespace {

constexpr int MAX_CAND = FCHUNK_VERTS;  // candidates of one vertex range
static_assert(FCHUNK_VERTS <= 32 * (WAVE - 1), "a range's bitmap words fit one wave");

// Start-vertex candidates of every op.  A wave owns 64 consecutive bitmap
// words (2048 vertices); lane l loads the keys of vertices base + l + 64 j,
// j < 32 (each load instruction reads 256 contiguous bytes), keeps them in
// registers, and for each op of its group one ballot per j gives the two
// words 2j and 2j + 1, which lanes 2j and 2j + 1 keep.  The keys are read
// once for all ops, and each op's 64 words leave as one coalesced store.
constexpr uint32_t INIT_OPS = 16;  // ops per wave

__global__ void __launch_bounds__(256) init_kernel(const uint32_t* __restrict__ key, uint32_t n, uint32_t W,
                                                   const InitOp* __restrict__ ops, uint32_t nops,
                                                   uint32_t* __restrict__ bitmaps) {
  const uint32_t lane = lane_id();
  const uint32_t blocks = (W + WAVE - 1) / WAVE, groups = (nops + INIT_OPS - 1) / INIT_OPS;
  const uint64_t wave = ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) / WAVE;
  if (wave >= (uint64_t)blocks * groups) return;  // the whole wave
  const uint32_t wb = (uint32_t)(wave % blocks), og = (uint32_t)(wave / blocks);
  const uint32_t v0 = wb * WAVE * 32;
  uint32_t k[32];
#pragma unroll
  for (uint32_t j = 0; j < 32; ++j) {
    const uint32_t v = v0 + j * WAVE + lane;
    k[j] = v < n ? key[v] : 0u;  // key 0 matches no op (dense labels start at 1)
  }
  const uint32_t w = wb * WAVE + lane;
  const uint32_t o_end = min(nops, (og + 1) * INIT_OPS);
  for (uint32_t o = og * INIT_OPS; o < o_end; ++o) {
    const uint32_t lo = uniform(ops[o].lo), hi = uniform(ops[o].hi), slot = uniform(ops[o].slot);
    uint32_t word = 0;
#pragma unroll
    for (uint32_t j = 0; j < 32; ++j) {
      const unsigned long long m = __ballot(k[j] >= lo && k[j] <= hi);
      if (lane == 2 * j) word = (uint32_t)m;
      if (lane == 2 * j + 1) word = (uint32_t)(m >> 32);
    }
    if (w < W) bitmaps[(size_t)slot * W + w] = word;
  }
}

// The (op, vertex range) pairs of a superstep whose range holds at least one
// candidate of the op's C(u), appended to items[] (order arbitrary: a
// superstep's updates are atomic bit operations on distinct slots per
// query, so the order of its items does not change the result).  Once the
// sets are small most ranges are empty, and the superstep then costs one
// coalesced pass over the bitmap words instead of one wave per pair.
// One wave per (op, 256 consecutive ranges); lane l reads words l, l + 64,
// ... of the ranges' span, eight loads in flight, together with the range of
// each word's first vertex (wrange), and a nonzero word marks its range
// (and, when it runs past that range's end, the next ones it has bits in).
// The four waves of a workgroup take consecutive range groups of one op,
// and the list is appended to with one atomic per workgroup: appends to a
// single counter serialise, and one per wave cost as much as the scan.
constexpr uint32_t AR_GROUP = 4 * WAVE;  // vertex ranges per wave
constexpr int AR_UNROLL = 8;             // bitmap words in flight per lane

__global__ void __launch_bounds__(256) active_ranges_kernel(const uint32_t* __restrict__ fchunk,
                                                             const uint32_t* __restrict__ wrange, uint32_t max_ranges,
                                                             const FilterOp* __restrict__ ops, uint32_t nops,
                                                             const uint32_t* __restrict__ bitmaps, uint32_t W,
                                                             const uint32_t* __restrict__ rflags,
                                                             uint2* __restrict__ items, uint32_t* __restrict__ nitems) {
  __shared__ uint32_t s_lo[4][AR_GROUP + 1];
  __shared__ uint32_t s_act[4][AR_GROUP];
  __shared__ uint32_t s_wtot[4], s_wbase[4];
  const uint32_t lane = lane_id(), wv = threadIdx.x / WAVE;
  const uint32_t groups = (max_ranges + AR_GROUP - 1) / AR_GROUP;
  const uint32_t wgs_per_op = (groups + 3) / 4;
  const uint32_t o_wg = blockIdx.x / wgs_per_op;  // the workgroup's op
  const uint32_t g = (blockIdx.x % wgs_per_op) * 4 + wv;
  uint32_t* lo_b = s_lo[wv];
  uint32_t* act = s_act[wv];
#pragma unroll
  for (uint32_t j = 0; j < AR_GROUP / WAVE; ++j) act[j * WAVE + lane] = 0;
  const uint32_t o = o_wg;
  uint32_t c0 = 0, nc = 0;
  if (o < nops && g < groups) {  // uniform per wave
    const uint32_t nrange = uniform(ops[o].nrange);
    c0 = uniform(ops[o].range0) + g * AR_GROUP;
    const uint32_t need = uniform(ops[o].need);
    // an op whose previous refine round removed nothing lists no range
    if (g * AR_GROUP < nrange && (need == ~0u || uniform(rflags[need]) != 0))
      nc = min(AR_GROUP, nrange - g * AR_GROUP);
  }
  if (nc) {
    for (uint32_t j = lane; j <= nc; j += WAVE) lo_b[j] = fchunk[c0 + j];
    wave_sync();
    const uint32_t v_begin = lo_b[0], v_end = lo_b[nc];
    const uint32_t w_begin = v_begin >> 5, w_last = (v_end - 1) >> 5;
    const uint32_t* bm = bitmaps + (size_t)uniform(ops[o].u_slot) * W;
    for (uint32_t w0 = w_begin; w0 <= w_last; w0 += WAVE * AR_UNROLL) {
      uint32_t xs[AR_UNROLL], rs[AR_UNROLL];
#pragma unroll
      for (int u = 0; u < AR_UNROLL; ++u) {
        const uint32_t w = w0 + u * WAVE + lane;
        xs[u] = 0;
        rs[u] = 0;
        if (w <= w_last) {
          xs[u] = bm[w];
          rs[u] = wrange[w];
        }
      }
#pragma unroll
      for (int u = 0; u < AR_UNROLL; ++u) {
        const uint32_t w = w0 + u * WAVE + lane;
        uint32_t x = xs[u];
        if (w == w_begin) x &= ~0u << (v_begin & 31);
        if (w == w_last && (v_end & 31)) x &= (1u << (v_end & 31)) - 1u;
        // range a holds the lowest remaining set bit: the word's first range
        // (c0 or later once the bits below v_begin are masked), then forward
        uint32_t a = rs[u] > c0 ? rs[u] - c0 : 0u;
        while (x) {
          const uint32_t v = w * 32 + (uint32_t)(__ffs(x) - 1);
          while (lo_b[a + 1] <= v) ++a;
          act[a] = 1;
          const uint32_t next = lo_b[a + 1];  // first vertex after range a (> v)
          if (next >= w * 32 + 32) break;
          x &= ~0u << (next - w * 32);
        }
      }
    }
  }
  wave_sync();
  // lane l owns ranges l, l + 64, l + 128, l + 192 of the wave's group
  uint32_t mine = 0;
#pragma unroll
  for (uint32_t j = 0; j < AR_GROUP / WAVE; ++j) mine += act[j * WAVE + lane] != 0;
  const uint32_t incl = wave_incl_scan(mine);
  if (lane == WAVE - 1) s_wtot[wv] = incl;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t tot = 0;
    for (uint32_t x = 0; x < blockDim.x / WAVE; ++x) {
      s_wbase[x] = tot;
      tot += s_wtot[x];
    }
    const uint32_t base = tot ? atomicAdd(nitems, tot) : 0u;
    for (uint32_t x = 0; x < blockDim.x / WAVE; ++x) s_wbase[x] += base;
  }
  __syncthreads();
  uint32_t pos = s_wbase[wv] + incl - mine;
#pragma unroll
  for (uint32_t j = 0; j < AR_GROUP / WAVE; ++j)
    if (act[j * WAVE + lane]) items[pos++] = make_uint2(o, c0 + j * WAVE + lane);
}

constexpr int UNROLL = 4;  // adjacency entries in flight per lane

struct WaveLds {
  uint32_t cand[MAX_CAND];
  uint32_t pre[WAVE + 1];
  uint32_t base[WAVE];
  uint32_t hit[WAVE];
};

// One step over the next entries of T flattened ones: UNROLL in flight per
// lane, or one where that takes them all (pieces are short: most steps do).
// The number of entries it covers.
template <typename Step>
__device__ __forceinline__ uint32_t step_entries(uint32_t T, Step step) {
  if (T <= WAVE) {
    step(std::integral_constant<int, 1>());
    return WAVE;
  }
  step(std::integral_constant<int, UNROLL>());
  return UNROLL * WAVE;
}

// Which candidates meet their op's neighbours.  list null: every (op, range)
// pair is an item (nops * chunks of them, the ops whose need flag is clear
// leave theirs).  A refine op drops the others.  An explore op drops them too
// and leaves behind what the neighbours' sets are filled from (fill_kernel):
// a candidate that meets v_0 .. v_{i-1} but not v_i still hands its matches
// to those before v_i (match/Match.cu:547-600), so its bit goes to their
// bitmaps at e_slot (v_0 .. v_{nv-2}: no candidate that fails has met all);
// counts[cnt] counts the candidates that meet v_0.
__global__ void __launch_bounds__(256) filter_step_kernel(Pieces pieces, const uint32_t* __restrict__ col,
                                                          const uint32_t* __restrict__ ckey, uint32_t W,
                                                          const uint32_t* __restrict__ fchunk,
                                                          const uint2* __restrict__ list,
                                                          const uint32_t* __restrict__ nlist, uint32_t max_ranges,
                                                          uint32_t nops, const FilterOp* __restrict__ ops,
                                                          const uint32_t* __restrict__ nbr_slot,
                                                          const uint32_t* __restrict__ nbr_lo,
                                                          const uint32_t* __restrict__ nbr_hi,
                                                          uint32_t* __restrict__ bitmaps,
                                                          uint32_t* __restrict__ rflags,
                                                          uint32_t* __restrict__ counts,
                                                          unsigned long long* __restrict__ stats) {
  extern __shared__ unsigned char lds_raw[];
  WaveLds& L = reinterpret_cast<WaveLds*>(lds_raw)[threadIdx.x / WAVE];
  const uint32_t lane = lane_id();
  const uint32_t items = list ? uniform(*nlist) : nops * max_ranges;
  const uint32_t wave = uniform((blockIdx.x * blockDim.x + threadIdx.x) / WAVE);
  const uint32_t nwaves = (gridDim.x * blockDim.x) / WAVE;
  // per-lane tallies for the optional byte accounting, over all items
  uint32_t t_piece = 0, t_ent = 0, t_probe = 0;

  // the next item's list entry is loaded while the current one runs
  uint2 nxt = list && wave < items ? list[wave] : make_uint2(0u, 0u);
  for (uint32_t it = wave; it < items; it += nwaves) {
    uint32_t o, c;
    if (list) {
      const uint2 item = nxt;
      if (it + nwaves < items) nxt = list[it + nwaves];
      o = uniform(item.x);
      c = uniform(item.y);
    } else {
      o = it / max_ranges;
      c = it % max_ranges;
      if (c >= uniform(ops[o].nrange)) continue;
      c += uniform(ops[o].range0);
      const uint32_t need = uniform(ops[o].need);
      if (need != ~0u && uniform(rflags[need]) == 0) continue;
    }
    const uint32_t type = uniform(ops[o].type);
    const uint32_t nv = uniform(ops[o].nv);
    const uint32_t nb = uniform(ops[o].nbr_off);
    uint32_t* bm_u = bitmaps + (size_t)uniform(ops[o].u_slot) * W;

    // collect: candidates of vertex range [v_lo, v_hi), ascending; lane l
    // reads bitmap word w_lo + l and keeps the range's bits of it
    const uint32_t v_lo = uniform(fchunk[c]), v_hi = uniform(fchunk[c + 1]);
    const uint32_t w_lo = v_lo >> 5, nw = ((v_hi - 1) >> 5) - w_lo + 1;
    const uint32_t wi = w_lo + lane;
    uint32_t w = 0;
    if (lane < nw) {
      w = bm_u[wi];
      if (lane == 0) w &= ~0u << (v_lo & 31);
      if (lane == nw - 1 && (v_hi & 31)) w &= (1u << (v_hi & 31)) - 1u;
    }
    const uint32_t pc = __popc(w);
    const uint32_t incl = wave_incl_scan(pc);
    const uint32_t C = uniform(__shfl(incl, WAVE - 1, WAVE));
    if (C == 0) continue;
    {
      uint32_t pos = incl - pc, x = w;
      while (x) {
        const uint32_t b = __ffs(x) - 1;
        x &= x - 1;
        L.cand[pos++] = wi * 32 + b;
      }
    }
    wave_sync();

    uint32_t met = 0;  // explore: candidates that meet v_0
    for (uint32_t s0 = 0; s0 < C; s0 += WAVE) {
      // lane = one candidate of the sub-chunk; the neighbours v_i one after
      // the other, each in the candidates' pieces towards its label
      const bool mine = s0 + lane < C;
      const uint32_t id = mine ? L.cand[s0 + lane] : 0u;
      uint32_t ff = mine ? nv : 0u;  // the first neighbour without a match
      uint32_t off = 0, len = 0;
      piece(pieces, id, nbr_lo[nb], off, len);
      for (uint32_t i = 0; i < nv; ++i) {
        const uint32_t lo = uniform(nbr_lo[nb + i]), hi = uniform(nbr_hi[nb + i]);
        const uint32_t* bm = bitmaps + (size_t)uniform(nbr_slot[nb + i]) * W;
        // the next neighbour's pieces load behind this one's entries
        uint32_t noff = 0, nlen = 0;
        if (i + 1 < nv) piece(pieces, id, nbr_lo[nb + i + 1], noff, nlen);
        const bool alive = mine && ff == nv;
        if (stats) t_piece += alive;
        L.hit[lane] = 0;
        uint32_t cur = 0;  // entries of this candidate already examined
        bool h = !alive;
        wave_sync();
        // every step re-flattens the remaining entries of the candidates
        // without a match, so one that has it stops costing lanes
        for (;;) {
          const uint32_t rem = h ? 0u : len - cur;
          const uint32_t rincl = wave_incl_scan(rem);
          const uint32_t T = uniform(__shfl(rincl, WAVE - 1, WAVE));
          if (T == 0) break;
          const uint32_t rpre = rincl - rem;
          L.pre[lane] = rpre;
          L.base[lane] = off + cur;
          wave_sync();
          const uint32_t span = step_entries(T, [&](auto U) {
            constexpr int N = decltype(U)::value;
            // an entry index past T reads entry T - 1 (in bounds): the same
            // answer again, and every lane loads, no branch per entry
            uint32_t cis[N], gi[N], es[N];
#pragma unroll
            for (int u = 0; u < N; ++u) cis[u] = gi[u] = min(u * WAVE + lane, T - 1);
            halving_search<N>(L.pre, WAVE, cis);
#pragma unroll
            for (int u = 0; u < N; ++u) es[u] = L.base[cis[u]] + (gi[u] - L.pre[cis[u]]);
            if (type == OP_REFINE) {
              // refine: in C(v_i)
              uint32_t mvs[N], wv[N];
#pragma unroll
              for (int u = 0; u < N; ++u) mvs[u] = col[es[u]];
#pragma unroll
              for (int u = 0; u < N; ++u) wv[u] = bm[mvs[u] >> 5];
#pragma unroll
              for (int u = 0; u < N; ++u)
                if ((wv[u] >> (mvs[u] & 31)) & 1u) L.hit[cis[u]] = 1;
              t_probe += min((T + WAVE - 1 - lane) / WAVE, (uint32_t)N);
            } else {
              // explore: the entry's key (read in place of the column index:
              // no extra bytes) in v_i's label/degree range
              uint32_t ks[N];
#pragma unroll
              for (int u = 0; u < N; ++u) ks[u] = ckey[es[u]];
#pragma unroll
              for (int u = 0; u < N; ++u)
                if (ks[u] >= lo && ks[u] <= hi) L.hit[cis[u]] = 1;
            }
            t_ent += min((T + WAVE - 1 - lane) / WAVE, (uint32_t)N);
          });
          wave_sync();
          cur += rpre >= span ? 0u : min(rem, span - rpre);
          h = !alive || L.hit[lane] != 0;
        }
        if (alive && !h) ff = i;
        off = noff;
        len = nlen;
        if (!__any(mine && ff == nv)) break;
      }

      if (type == OP_REFINE) {
        const bool drop = mine && ff < nv;
        if (drop) clear_bit(bm_u, id);
        if (__ballot(drop) && lane == 0) rflags[uniform(ops[o].mark)] = 1u;
      } else {
        // first neighbour without a match: mu leaves C(u), its matches of the
        // neighbours before it stay
        if (mine && ff < nv) {
          clear_bit(bm_u, id);
          uint32_t* e = bitmaps + (size_t)ops[o].e_slot * W;
          for (uint32_t i = 0; i < ff; ++i) set_bit(e + (size_t)i * W, id);  // ff < nv: e_slot has nv - 1 rows
        }
        met += (uint32_t)__popcll(__ballot(mine && ff > 0));
      }
      wave_sync();
    }
    if (met && lane == 0) atomicAdd(&counts[ops[o].cnt], met);
  }
  if (stats) {
    // one atomic per counter per workgroup, spread over STAT_COPIES copies
    __shared__ unsigned long long red[4][5];
    const unsigned long long v[5] = {wave_sum64(t_piece), wave_sum64(t_ent), 0, wave_sum64(t_probe), 0};
    const uint32_t w = threadIdx.x / WAVE;
    if (lane == 0)
      for (int i = 0; i < 5; ++i) red[w][i] = v[i];
    __syncthreads();
    if (threadIdx.x < 5) {
      unsigned long long tot = 0;
      for (uint32_t x = 0; x < blockDim.x / WAVE; ++x) tot += red[x][threadIdx.x];
      if (tot) atomicAdd(stats + (blockIdx.x % STAT_COPIES) * STAT_STRIDE + threadIdx.x, tot);
    }
  }
}

// The vertices an explore op's neighbour v receives: those in v's label and
// degree range with a neighbour in C(u) (or in e_slot's bitmap).  One wave
// per (fill, vertex range), whichever way is cheaper for the fill:
//  pull  the range's vertices of v's label look for a neighbour in C(u) and
//        stop at the first, as a refine op does; the range's words are
//        written once;
//  push  the range's candidates of C(u) set the bits of their matches (read
//        first, an atomic only where clear); a vertex with more entries than
//        a range holds goes in parts of HUB_PART, one wave each.
// Pushing alone took 85-340 us per op on the 1M Chung-Lu graph for some 1e5
// vertices found, bound by the atomics: the lines of one 125 KB bitmap move
// between the L2s of eight XCDs.  Pulling them takes 11-28 us.  A vertex of v's
// label without a neighbour in C(u) is walked to its end, so where v's label
// has more than FILL_PULL times as many vertices as C(u) they are pushed.
struct FillLds {
  uint32_t cand[MAX_CAND];
  uint32_t pre[WAVE + 1];
  uint32_t base[WAVE];
  uint32_t hit[WAVE];
  uint32_t word[WAVE];
};

__global__ void __launch_bounds__(256) fill_kernel(const uint32_t* __restrict__ row, Pieces pieces,
                                                   const uint32_t* __restrict__ col,
                                                   const uint32_t* __restrict__ key,
                                                   const uint32_t* __restrict__ ckey, uint32_t W,
                                                   const uint32_t* __restrict__ fchunk, uint32_t max_ranges,
                                                   const uint2* __restrict__ hparts, uint32_t nhp,
                                                   const FillOp* __restrict__ fills, uint32_t nfill,
                                                   const uint32_t* __restrict__ counts, uint32_t* bitmaps, unsigned long long* __restrict__ stats) {
  extern __shared__ unsigned char lds_raw[];
  FillLds& L = reinterpret_cast<FillLds*>(lds_raw)[threadIdx.x / WAVE];
  const uint32_t lane = lane_id();
  const uint64_t wave = ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) / WAVE;
  const uint64_t nwaves = ((uint64_t)gridDim.x * blockDim.x) / WAVE;
  const uint64_t pairs = (uint64_t)nfill * max_ranges, items = pairs + (uint64_t)nfill * nhp;
  uint32_t t_piece = 0, t_ent = 0, t_key = 0, t_probe = 0, t_set = 0;
  for (uint64_t it = wave; it < items; it += nwaves) {
    const bool part = it >= pairs;
    const uint64_t x = part ? it - pairs : it;
    const uint32_t per = part ? nhp : max_ranges;
    const uint32_t f = uniform((uint32_t)(x / per));
    uint32_t c = uniform((uint32_t)(x % per));
    const FillOp& op = fills[f];
    const uint32_t lo = uniform(op.lo), hi = uniform(op.hi), met = uniform(counts[op.cnt]);
    if (met == 0) continue;
    const bool pull = (uint64_t)met * FILL_PULL >= uniform(op.nlabel);
    if (part && pull) continue;
    const uint32_t* bm_u = bitmaps + (size_t)uniform(op.u_slot) * W;
    const uint32_t e_slot = uniform(op.e_slot), u_lo = uniform(op.u_lo);
    const uint32_t* bm_e = e_slot != ~0u ? bitmaps + (size_t)e_slot * W : nullptr;
    uint32_t* bm_v = bitmaps + (size_t)uniform(op.v_slot) * W;
    uint32_t v_lo, v_hi, first = 0;  // first: where a part's entries start
    if (part) {
      const uint2 hp = hparts[c];
      v_lo = uniform(hp.x);
      v_hi = v_lo + 1;
      first = uniform(hp.y) * HUB_PART;
    } else {
      if (c >= uniform(op.nrange[pull])) continue;
      c += uniform(op.range0[pull]);
      v_lo = uniform(fchunk[c]);
      v_hi = uniform(fchunk[c + 1]);
    }
    const uint32_t w_lo = v_lo >> 5, nw = ((v_hi - 1) >> 5) - w_lo + 1;
    uint32_t C = 0;
    if (pull) {
      // the range's vertices with v's label and degree, ascending
      for_steps(v_lo, v_hi, [&](uint64_t v0) {
        const uint64_t v = v0 + lane;
        const uint32_t k = v < v_hi ? key[v] : 0u;
        if (stats) t_key += v < v_hi;
        const unsigned long long m = __ballot(k >= lo && k <= hi && v < v_hi);
        if ((m >> lane) & 1ULL) L.cand[C + (uint32_t)__popcll(lane ? m & (~0ULL >> (WAVE - lane)) : 0ULL)] = (uint32_t)v;
        C += (uint32_t)__popcll(m);
      });
      L.word[lane] = 0;
    } else {
      uint32_t w = 0;
      if (lane < nw) {
        w = bm_u[w_lo + lane];
        if (bm_e) w |= bm_e[w_lo + lane];
        if (lane == 0) w &= ~0u << (v_lo & 31);
        if (lane == nw - 1 && (v_hi & 31)) w &= (1u << (v_hi & 31)) - 1u;
      }
      const uint32_t pc = __popc(w);
      const uint32_t incl = wave_incl_scan(pc);
      C = uniform(__shfl(incl, WAVE - 1, WAVE));
      uint32_t pos = incl - pc;
      for (; w; w &= w - 1) L.cand[pos++] = (w_lo + lane) * 32 + (uint32_t)(__ffs(w) - 1);
    }
    if (C == 0) continue;
    wave_sync();
    for (uint32_t s0 = 0; s0 < C; s0 += WAVE) {
      const bool mine = s0 + lane < C;
      const uint32_t id = mine ? L.cand[s0 + lane] : 0u;
      uint32_t off = 0, len = 0;
      if (stats) t_piece += mine;
      if (mine) {
        piece(pieces, id, pull ? u_lo : lo, off, len);
        off += first;
        if (part) len = len > first ? min(len - first, HUB_PART) : 0u;
        else if (!pull && row[id + 1] - row[id] > FCHUNK_ENTRIES) len = 0;  // pushed by its parts
      }
      if (pull) {
        L.hit[lane] = 0;
        uint32_t cur = 0;
        bool h = false;
        wave_sync();
        for (;;) {
          const uint32_t rem = h ? 0u : len - cur;
          const uint32_t rincl = wave_incl_scan(rem);
          const uint32_t T = uniform(__shfl(rincl, WAVE - 1, WAVE));
          if (T == 0) break;
          const uint32_t rpre = rincl - rem;
          L.pre[lane] = rpre;
          L.base[lane] = off + cur;
          wave_sync();
          uint32_t cis[UNROLL], gi[UNROLL], mvs[UNROLL], wv[UNROLL];
#pragma unroll
          for (int u = 0; u < UNROLL; ++u) cis[u] = gi[u] = min(u * WAVE + lane, T - 1);
          halving_search<UNROLL>(L.pre, WAVE, cis);
#pragma unroll
          for (int u = 0; u < UNROLL; ++u) mvs[u] = col[L.base[cis[u]] + (gi[u] - L.pre[cis[u]])];
#pragma unroll
          for (int u = 0; u < UNROLL; ++u) {
            wv[u] = bm_u[mvs[u] >> 5];
            if (bm_e) wv[u] |= bm_e[mvs[u] >> 5];
          }
          // an index past T repeats entry T - 1: the same answer again
#pragma unroll
          for (int u = 0; u < UNROLL; ++u)
            if ((wv[u] >> (mvs[u] & 31)) & 1u) L.hit[cis[u]] = 1;
          wave_sync();
          const uint32_t span = UNROLL * WAVE;
          cur += rpre >= span ? 0u : min(rem, span - rpre);
          h = L.hit[lane] != 0;
          if (stats) {
            t_ent += min((T + WAVE - 1 - lane) / WAVE, (uint32_t)UNROLL);
            t_probe += min((T + WAVE - 1 - lane) / WAVE, (uint32_t)UNROLL);
          }
        }
        if (h) atomicOr(&L.word[(id >> 5) - w_lo], 1u << (id & 31));
        t_set += h;
      } else {
        const uint32_t incl = wave_incl_scan(len);
        const uint32_t T = uniform(__shfl(incl, WAVE - 1, WAVE));
        L.pre[lane] = incl - len;
        L.base[lane] = off;
        wave_sync();
        for (uint32_t f0 = 0; f0 < T; f0 += UNROLL * WAVE) {
          uint32_t cis[UNROLL], gi[UNROLL], mvs[UNROLL], cw[UNROLL];
          bool want[UNROLL];
#pragma unroll
          for (int u = 0; u < UNROLL; ++u) cis[u] = gi[u] = min(f0 + u * WAVE + lane, T - 1);
          halving_search<UNROLL>(L.pre, WAVE, cis);
#pragma unroll
          for (int u = 0; u < UNROLL; ++u) {
            const uint32_t e = L.base[cis[u]] + (gi[u] - L.pre[cis[u]]);
            mvs[u] = col[e];
            const uint32_t k = ckey[e];
            want[u] = f0 + u * WAVE + lane < T && k >= lo && k <= hi;
          }
          // a bit is set (one atomic) only where it is still clear
#pragma unroll
          for (int u = 0; u < UNROLL; ++u)
            cw[u] = want[u] ? __hip_atomic_load(bm_v + (mvs[u] >> 5), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : ~0u;
#pragma unroll
          for (int u = 0; u < UNROLL; ++u) {
            const uint32_t m = 1u << (mvs[u] & 31);
            if (want[u] && !(cw[u] & m)) atomicOr(bm_v + (mvs[u] >> 5), m);
            if (stats) {
              const bool in = f0 + u * WAVE + lane < T;
              t_ent += in;
              t_key += in;
              t_set += want[u];
            }
          }
        }
      }
      wave_sync();
    }
    if (pull) {
      // two ranges may share a word
      const uint32_t w = lane < nw ? L.word[lane] : 0u;
      if (w) atomicOr(bm_v + w_lo + lane, w);
    }
    wave_sync();
  }
  if (stats) {
    const unsigned long long v[5] = {wave_sum64(t_piece), wave_sum64(t_ent), wave_sum64(t_key), wave_sum64(t_probe),
                                     wave_sum64(t_set)};
    if (lane == 0)
      for (int i = 0; i < 5; ++i)
        if (v[i]) atomicAdd(stats + (blockIdx.x % STAT_COPIES) * STAT_STRIDE + i, v[i]);
  }
}

}  // namespace

void launch_init(const DevGraph& g, const InitOp* ops, uint32_t nops, uint32_t* bitmaps, hipStream_t s) {
  if (!nops) return;
  const uint64_t waves = (uint64_t)((g.W + WAVE - 1) / WAVE) * ((nops + INIT_OPS - 1) / INIT_OPS);
  hipLaunchKernelGGL(init_kernel, dim3((uint32_t)((waves + 3) / 4)), dim3(256), 0, s, g.key, g.n, g.W, ops, nops,
                     bitmaps);
}

void launch_filter_step(const DevGraph& g, const FilterOp* ops, uint32_t nops, const uint32_t* nbr_slot,
                        const uint32_t* nbr_lo, const uint32_t* nbr_hi, const FillOp* fills, uint32_t nfill,
                        uint32_t* bitmaps, uint32_t max_ranges, uint32_t block, uint32_t resident, uint2* items,
                        uint32_t* nitems, uint32_t* rflags, uint32_t* counts, unsigned long long* stats,
                        hipStream_t s) {
  if (!nops) return;
  const uint64_t pairs = (uint64_t)nops * max_ranges;
  const bool direct = pairs <= FILTER_DIRECT;
  if (!direct) {
    const uint32_t wgs_per_op = ((max_ranges + AR_GROUP - 1) / AR_GROUP + 3) / 4;
    // four waves per workgroup: the kernel's LDS and its per-workgroup append assume 256 threads
    hipLaunchKernelGGL(active_ranges_kernel, dim3(nops * wgs_per_op), dim3(256), 0, s, g.fchunk, g.wrange, max_ranges,
                       ops, nops, bitmaps, g.W, rflags, items, nitems);
  }
  // the list's length is known on the device only: a grid of at most
  // FILTER_OVERSUB times as many workgroups as are resident at once strides
  // over it (waves past its end leave at once).
  // Workgroups beyond the resident ones start as earlier ones finish, which
  // evens out uneven items (R-MAT hub ranges); with far more, the waves in
  // flight touch more bitmaps at a time.  Measured per batch: 1x resident
  // 10.9 ms (1M Chung-Lu mix) / 24.0 ms (R-MAT 22 shapes), 8x 11.1 / 20.9,
  // 65,536 workgroups 13.3 / 19.5; items taken from a shared counter (16
  // per atomic) 14.1 / 28.4, the atomics serialising across the XCDs.
  const uint32_t wpb = block / WAVE;
  const uint64_t most = (uint64_t)resident * FILTER_OVERSUB;
  hipLaunchKernelGGL(filter_step_kernel, dim3((uint32_t)std::min((pairs + wpb - 1) / wpb, most)), dim3(block),
                     sizeof(WaveLds) * wpb, s, pieces_of(g), g.col, g.ckey, g.W, g.fchunk,
                     direct ? nullptr : items, nitems, max_ranges, nops, ops, nbr_slot, nbr_lo, nbr_hi, bitmaps, rflags, counts, stats);
  const uint64_t fwaves = (uint64_t)nfill * (max_ranges + g.nhparts);
  if (!fwaves) return;
  hipLaunchKernelGGL(fill_kernel, dim3((uint32_t)std::min((fwaves + wpb - 1) / wpb, most)), dim3(block),
                     sizeof(FillLds) * wpb, s, g.row, pieces_of(g), g.col, g.key, g.ckey, g.W, g.fchunk, max_ranges,
                     g.hparts, g.nhparts, fills, nfill, counts, bitmaps, stats);
}

uint32_t filter_resident(uint32_t block) {
  int dev = 0, ncu = 0, per_cu = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
      hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, filter_step_kernel, (int)block,
                                                   sizeof(WaveLds) * (block / WAVE)) != hipSuccess ||
      ncu < 1 || per_cu < 1) {
    (void)hipGetLastError();
    return 8192;
  }
  return (uint32_t)ncu * (uint32_t)per_cu;
}

}  // namespace gpsm
