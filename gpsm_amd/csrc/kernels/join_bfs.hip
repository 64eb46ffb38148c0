// Breadth-first join of plans with back edges (join_kernel, expand_kernel,
// link_kernel, match/Match.cu:1141-1569): every level of every such plan of a
// batch in one launch.
//
// The depth-first kernel (join.hip) shares work by rows of the first table.
// On a power-law graph a cycle or clique query has a few thousand of those,
// and the one that binds two hubs holds most of the query's work: a 6-clique
// on an R-MAT graph of 2^18 vertices took 103 ms for 3.5e8 candidates, one
// workgroup walking most of them.  Here all rows of a level are in memory
// before the next level starts, so the whole device shares them:
//  * a row (its vertices, hash product, plan and the candidate list that
//    extends it) is one record; 16 lanes take a row of at most LONG_LIST
//    candidates, four rows per wave, a workgroup takes a longer one;
//  * a row's candidates come from its parent's candidate-edge list, or, with
//    the learned order, from a back edge's bound vertex of shorter adjacency
//    (tested against C(w) and the parent's edge instead): the order's choice
//    of the vertex to expand from, made row by row;
//  * survivors are staged in LDS and finished densely, one lane each: their
//    own next list (rank index, offsets), then one record;
//  * the last level is counted and hashed, not written.
// Records are reserved in blocks per wave: one counter for a level's rows,
// added to by every wave step, would serialise on one address.
// When the next level's buffer is full a wave saves where it stands (the row,
// the step of its candidates, the survivors already written) and stops; the
// caller runs the deeper levels, empties them, and launches the level again
// from the saved places, so a join of any size runs in bounded memory and
// nothing is counted twice.
#include <algorithm>

#include "edge.h"
#include "launch.h"
#include "wave.h"

namespace gpsm {

namespace {

// row record: words 0-1 hash product, 2 plan, 3 start of the candidates, 4
// their number (0: no row), 5 their source (0: the parent's list, 1 + b: the
// adjacency of the vertex at back position b), then the level + 1 vertices
constexpr uint32_t R_PLAN = 2, R_START = 3, R_LEN = 4, R_SRC = 5, R_VAL = 6;
constexpr uint32_t GROUP = 16;         // lanes per short row (one DPP row)
constexpr uint32_t LONG_LIST = 512;    // candidates above which workgroups take the row
constexpr int BFS_UNROLL = 4;          // candidates in flight per lane
constexpr uint32_t STAGE = WAVE * BFS_UNROLL;  // staged survivors of a wave's step

struct PlanAcc {
  unsigned long long cnt, hash, rows, work;
};

struct WaveStage {
  uint32_t mv[STAGE];
  uint32_t grp[STAGE];          // group of the wave whose row the survivor extends
  const uint32_t* row[WAVE / GROUP];
};

// A wave's block of reserved row slots of the level being written.
struct Slots {
  uint32_t at, left;
};

__device__ __forceinline__ void flush_acc(const BfsArgs& a, const PlanAcc* acc) {
  for (uint32_t i = threadIdx.x; i < a.nplans; i += blockDim.x) {
    const PlanAcc& x = acc[i];
    const uint32_t nk = a.level + 1;
    JoinOut& o = a.j.out[a.j.plans[i].out];
    if (x.cnt) {
      atomicAdd(&o.count, x.cnt);
      atomicAdd(&o.level_rows[a.j.plans[i].q - 1], x.cnt);
    }
    if (x.hash) atomicAdd(&o.hash, x.hash);
    if (x.rows) atomicAdd(&o.level_rows[nk], x.rows);
    if (x.work) atomicAdd(&o.level_work[nk + 1], x.work);
    // first-table rows are work too
    const unsigned long long first = a.level == 0 ? x.rows : 0ull, done = x.work + first;
    if (first) atomicAdd(&o.level_work[1], first);
    if (done) {
      const unsigned long long before = atomicAdd(&o.work, done);
      if (a.j.budget && before + done > a.j.budget) o.aborted = 1;
    }
  }
}

// Finishes one new row per lane (has: the lane holds one): vals[0..k] are the
// vertices of the row it extends, mv the vertex at position nk = k + 1 and
// hash the row's product.  Finds the list that extends it, counts it, and
// writes its record unless it has no candidates.  All lanes of the wave call;
// false, with nothing written or counted, when the level's buffer is full.
__device__ __forceinline__ bool finish_rows(const BfsArgs& a, PlanAcc* acc, Slots& slots, bool has,
                                            const uint32_t* vals, uint32_t k, uint32_t plan, uint32_t mv,
                                            unsigned long long hash) {
  const uint32_t lane = lane_id();
  const unsigned long long bh = __ballot(has);
  if (!bh) return true;
  uint32_t st = 0, len = 0, src = 0, full = 0;
  if (has) {
    const JoinPlan& P = a.j.plans[plan];
    const uint32_t n2 = k + 2;
    const CetDesc& d = a.j.cets[P.cet[n2]];
    const uint32_t pp = P.par[n2];
    const uint32_t x = pp == k + 1 ? mv : vals[pp];
    const uint32_t j = rank_of(a.j.bitmaps + (size_t)d.x_slot * a.j.W, a.j.bprefix + (size_t)d.x_slot * a.j.NB, x);
    const uint32_t* off = a.j.offsets + d.off_base;
    st = off[j];
    full = off[j + 1] - st;
    len = full;
    // a back edge's vertex with less than half as many neighbours is the
    // cheaper source (its candidates take two tests more).  The heuristic
    // order's plans keep their expand edge, the reference's rule.
    for (uint32_t b = a.any_source ? P.back_off[n2] : P.back_off[n2 + 1]; b < P.back_off[n2 + 1]; ++b) {
      const uint32_t c = P.backs[b];
      const uint32_t u = c == k + 1 ? mv : vals[c];
      uint32_t r0, dg;
      piece(a.j.pieces, u, d.w_lo, r0, dg);
      if (full && 2 * (uint64_t)dg < len) {
        st = r0;
        len = dg;
        src = 1 + b - P.back_off[n2];
      }
    }
  }
  const bool lng = len > LONG_LIST, shrt = len && !lng;
  const unsigned long long bs = __ballot(shrt), bl = __ballot(lng);
  const unsigned long long below = lane ? (~0ULL >> (WAVE - lane)) : 0ULL;
  const uint32_t ns = (uint32_t)__popcll(bs), nl = (uint32_t)__popcll(bl);
  uint32_t lbase = 0;
  bool ok = true;
  if (nl) {
    if (lane == 0) lbase = atomicAdd(&a.cout[1], nl);
    lbase = uniform(lbase);
    ok = lbase + nl <= a.long_cap;
  }
  // slots: the wave's block, its rest first, then a new block of at least as
  // many as are missing (at most 64)
  const uint32_t old_at = slots.at, old_left = slots.left;
  uint32_t base = 0, take = 0;
  if (ok && ns > old_left) {
    take = max(a.block, ns - old_left);
    if (lane == 0) base = atomicAdd(&a.cout[0], take);
    base = uniform(base);
    ok = base + take <= a.cap;
  }
  if (!ok) {
    // what was reserved holds no rows
    if (lane < nl && lbase + lane < a.long_cap) a.long_out[(uint64_t)(lbase + lane) * a.stride_out + R_LEN] = 0;
    if (lane < take && base + lane < a.cap) a.rows_out[(uint64_t)(base + lane) * a.stride_out + R_LEN] = 0;
    return false;
  }
  uint32_t* dst = nullptr;
  if (shrt) {
    const uint32_t r = (uint32_t)__popcll(bs & below);
    dst = a.rows_out + (uint64_t)(r < old_left ? old_at + r : base + (r - old_left)) * a.stride_out;
  } else if (lng) {
    dst = a.long_out + (uint64_t)(lbase + (uint32_t)__popcll(bl & below)) * a.stride_out;
  }
  if (take) {
    slots.at = base + (ns - old_left);
    slots.left = take - (ns - old_left);
  } else {
    slots.at += ns;
    slots.left -= ns;
  }
  if (dst) {
    dst[0] = (uint32_t)hash;
    dst[1] = (uint32_t)(hash >> 32);
    dst[R_PLAN] = plan;
    dst[R_START] = st;
    dst[R_LEN] = len;
    dst[R_SRC] = src;
    for (uint32_t c = 0; c <= k; ++c) dst[R_VAL + c] = vals[c];
    dst[R_VAL + k + 1] = mv;
  }
  // rows and the work they bring, once per wave where one plan has them all
  const uint32_t p0 = (uint32_t)__shfl((int)plan, __ffsll((long long)bh) - 1, WAVE);
  if (__ballot(has && plan != p0) == 0) {
    const unsigned long long w = wave_sum64(full);
    if (lane == 0) {
      atomicAdd(&acc[p0].rows, (unsigned long long)__popcll(bh));
      if (w) atomicAdd(&acc[p0].work, w);
    }
  } else if (has) {
    atomicAdd(&acc[plan].rows, 1ull);
    if (full) atomicAdd(&acc[plan].work, (unsigned long long)full);
  }
  return true;
}

// The rest of a wave's block holds no rows.
__device__ __forceinline__ void close_slots(const BfsArgs& a, const Slots& slots) {
  for (uint32_t i = slots.at + lane_id(); i < slots.at + slots.left; i += WAVE)
    a.rows_out[(uint64_t)i * a.stride_out + R_LEN] = 0;
}

// Level-1 rows: the first tables of all plans, one thread per entry.
__global__ void __launch_bounds__(256) bfs_first_kernel(BfsArgs a) {
  extern __shared__ unsigned char lds_raw[];
  PlanAcc* acc = reinterpret_cast<PlanAcc*>(lds_raw);
  for (uint32_t i = threadIdx.x; i < a.nplans; i += blockDim.x) acc[i] = {0, 0, 0, 0};
  __syncthreads();
  Slots slots = {0, 0};
  const uint64_t total = a.first_row[a.nplans];
  for (uint64_t e0 = (uint64_t)blockIdx.x * blockDim.x; e0 < total; e0 += (uint64_t)gridDim.x * blockDim.x) {
    const uint64_t e = e0 + threadIdx.x;
    const bool has = e < total;
    uint32_t plan = 0, mu = 0, mv = 0;
    unsigned long long h = 0;
    if (has) {
      uint32_t lo = 0, hi = a.nplans;  // the last plan whose first row is at or before e
      while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (a.first_row[mid] <= e) lo = mid;
        else hi = mid;
      }
      plan = lo;
      const JoinPlan& P = a.j.plans[plan];
      const CetDesc& d0 = a.j.cets[P.first_cet];
      const uint32_t r = (uint32_t)(e - a.first_row[lo]);
      mu = a.j.clist[d0.clist_off + seg_search(a.j.offsets + d0.off_base, d0.ncand + 1, r)];
      mv = a.j.lists[d0.list_base + r];
      h = tuple_term(P.order[0], a.j.ids[mu]) * tuple_term(P.order[1], a.j.ids[mv]);
    }
    finish_rows(a, acc, slots, has, &mu, 0, plan, mv, h);
  }
  close_slots(a, slots);
  __syncthreads();
  flush_acc(a, acc);
}

// The candidates idx, idx + step, ... (BFS_UNROLL of them, below len) of a
// row: ok[u] and mv[u].  nk: the position they would bind.
__device__ __forceinline__ void test_candidates(const BfsArgs& a, const JoinPlan& P, const CetDesc& d,
                                                const uint32_t* __restrict__ vals, uint32_t nk, uint32_t st,
                                                uint32_t len, uint32_t src, uint32_t idx, uint32_t step,
                                                uint32_t (&mv)[BFS_UNROLL], bool (&ok)[BFS_UNROLL]) {
  const uint32_t* from = src ? a.j.col + st : a.j.lists + d.list_base + st;
#pragma unroll
  for (int u = 0; u < BFS_UNROLL; ++u) {
    ok[u] = idx + u * step < len;
    mv[u] = ok[u] ? from[idx + u * step] : 0u;
  }
  if (src) {
    // from an adjacency: in C(w), and adjacent to the parent
    const uint32_t* bm_w = a.j.bitmaps + (size_t)d.w_slot * a.j.W;
    uint32_t wd[BFS_UNROLL];
#pragma unroll
    for (int u = 0; u < BFS_UNROLL; ++u) wd[u] = ok[u] ? bm_w[mv[u] >> 5] >> (mv[u] & 31) : 0u;
#pragma unroll
    for (int u = 0; u < BFS_UNROLL; ++u) ok[u] = ok[u] && (wd[u] & 1u);
  }
  for (uint64_t m = len ? P.inj[nk] : 0; m; m &= m - 1) {
    const uint32_t c = vals[__ffsll((long long)m) - 1];
#pragma unroll
    for (int u = 0; u < BFS_UNROLL; ++u) ok[u] = ok[u] && mv[u] != c;
  }
  // a lane without a row (len 0) may name a plan of fewer positions
  const uint32_t bo = P.back_off[nk], nb = len ? P.back_off[nk + 1] - bo : 0u;
  for (uint32_t b = 0; b < nb; ++b) {
    // the source's own edge holds; the parent's is tested in its place
    const uint32_t bv = vals[src == 1 + b ? P.par[nk] : P.backs[bo + b]];
    const uint32_t hb = a.j.hub_of[bv];
    if (hb != ~0u) {
      const uint32_t* bm = a.j.hub_bits + (size_t)hb * a.j.W;
      uint32_t wd[BFS_UNROLL];
#pragma unroll
      for (int u = 0; u < BFS_UNROLL; ++u) wd[u] = ok[u] ? bm[mv[u] >> 5] >> (mv[u] & 31) : 0u;
#pragma unroll
      for (int u = 0; u < BFS_UNROLL; ++u) ok[u] = ok[u] && (wd[u] & 1u);
    } else {
      // a short row: its piece towards the candidates' label is shorter still
      uint32_t p0, n;
      piece(a.j.pieces, bv, d.w_lo, p0, n);
      const uint32_t* e[BFS_UNROLL];
#pragma unroll
      for (int u = 0; u < BFS_UNROLL; ++u) {
        ok[u] = ok[u] && n;
        e[u] = a.j.col + p0;
      }
      for (; n > 1; n -= n >> 1) {  // the last entry <= mv[u], as in has_edge
#pragma unroll
        for (int u = 0; u < BFS_UNROLL; ++u)
          if (ok[u]) e[u] = e[u][n >> 1] <= mv[u] ? e[u] + (n >> 1) : e[u];
      }
#pragma unroll
      for (int u = 0; u < BFS_UNROLL; ++u) ok[u] = ok[u] && *e[u] == mv[u];
    }
  }
}

// Staged survivors from .. n - 1 become rows, 64 at a time.  The first one
// not written (n when all are).
__device__ __forceinline__ uint32_t drain(const BfsArgs& a, PlanAcc* acc, Slots& slots, const WaveStage& G,
                                          uint32_t from, uint32_t n) {
  const uint32_t lane = lane_id(), nk = a.level + 1;
  for (uint32_t s0 = from; s0 < n; s0 += WAVE) {
    const bool has = s0 + lane < n;
    const uint32_t mv = has ? G.mv[s0 + lane] : 0u;
    const uint32_t* row = G.row[has ? G.grp[s0 + lane] : 0u];
    uint32_t plan = 0;
    unsigned long long h = 0;
    if (has) {
      plan = row[R_PLAN];
      h = (((unsigned long long)row[1] << 32) | row[0]) * tuple_term(a.j.plans[plan].order[nk], a.j.ids[mv]);
    }
    if (!finish_rows(a, acc, slots, has, row + R_VAL, a.level, plan, mv, h)) return s0;
  }
  return n;
}

// Adds a row's survivors to its plan's counters: the group's (or wave's) sums
// are already in the calling lane.
__device__ __forceinline__ void add_last(PlanAcc& x, unsigned long long cnt, unsigned long long hash) {
  if (cnt) atomicAdd(&x.cnt, cnt);
  if (hash) atomicAdd(&x.hash, hash);
}

// Stages the survivors of a step; their number.
__device__ __forceinline__ uint32_t stage_step(WaveStage& G, const uint32_t (&mv)[BFS_UNROLL],
                                               const bool (&ok)[BFS_UNROLL], bool keep, uint32_t grp) {
  const uint32_t lane = lane_id();
  const unsigned long long below = lane ? (~0ULL >> (WAVE - lane)) : 0ULL;
  uint32_t n = 0;
#pragma unroll
  for (int u = 0; u < BFS_UNROLL; ++u) {
    const bool put = ok[u] && keep;
    const unsigned long long bal = __ballot(put);
    if (put) {
      const uint32_t at = n + (uint32_t)__popcll(bal & below);
      G.mv[at] = mv[u];
      G.grp[at] = grp;
    }
    n += (uint32_t)__popcll(bal);
  }
  return n;
}

// Five waves per SIMD (96 VGPRs, 6 spilled): R-MAT 22 cliques 660 ms, cycles
// 1297 ms per batch, against 753 and 1375 at four (no spill) and 643 and 1338
// at six (32 spilled).  Bound by the back-edge probes: an n-bit hub bitmap is
// 32 KB on 2^18 vertices, so nearly every probe is an L2 miss of its own (79
// GB fetched in 16 ms, the copy rate of the card).
// Level a.level -> a.level + 1.  A wave's place in the level's rows is a
// cursor per kind of row: the row (or quad of rows), the step of its
// candidates, and the step's survivors already written.
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(5))) bfs_expand_kernel(BfsArgs a) {
  extern __shared__ unsigned char lds_raw[];
  PlanAcc* acc = reinterpret_cast<PlanAcc*>(lds_raw);
  __shared__ WaveStage stage[4];
  const uint32_t lane = lane_id(), wv = threadIdx.x / WAVE;
  WaveStage& G = stage[wv];
  for (uint32_t i = threadIdx.x; i < a.nplans; i += blockDim.x) acc[i] = {0, 0, 0, 0};
  __syncthreads();
  Slots slots = {0, 0};
  const uint32_t nk = a.level + 1;
  const uint32_t wave = blockIdx.x * (256 / WAVE) + wv, nwaves = gridDim.x * (256 / WAVE);
  BfsCursor* cur = a.cursors + (uint64_t)wave * 2;
  bool full = false;  // the next level's buffer is full (uniform per wave)

  // long rows: `share` workgroups each (one, unless there are fewer rows than
  // workgroups), whose waves take every (4 * share)-th step of 256 candidates
  const uint32_t nlong = min(a.cin[1], a.long_cap_in);
  const uint32_t share = nlong ? max(1u, min(64u, gridDim.x / nlong)) : 1u;
  const uint32_t first_pos = (blockIdx.x % share) * (256 / WAVE) + wv;
  const uint32_t rows_at_once = gridDim.x / share;
  uint32_t idx = blockIdx.x / share < rows_at_once ? blockIdx.x / share : ~0u, pos = first_pos, skip = 0;
  if (a.resume) idx = uniform(cur[0].idx), pos = uniform(cur[0].pos), skip = uniform(cur[0].skip);
  while (idx < nlong) {
    const uint32_t* row = a.long_in + (uint64_t)idx * a.stride_in;
    const uint32_t plan = uniform(row[R_PLAN]), st = uniform(row[R_START]), src = uniform(row[R_SRC]);
    uint32_t len = uniform(row[R_LEN]);
    if (len) {  // 0: reserved, not written
      if (a.j.budget && uniform((uint32_t)a.j.out[a.j.plans[plan].out].aborted)) len = 0;
      const JoinPlan& P = a.j.plans[plan];
      const CetDesc& d = a.j.cets[P.cet[nk]];
      const bool final = nk + 1 == P.q;
      const uint32_t qid = P.order[nk];
      if (lane == 0) G.row[0] = row;
      wave_sync();
      unsigned long long hsum = 0;
      uint32_t cnt = 0;
      for (; pos * (WAVE * BFS_UNROLL) < len; pos += share * (256 / WAVE)) {
        uint32_t mv[BFS_UNROLL];
        bool ok[BFS_UNROLL];
        test_candidates(a, P, d, row + R_VAL, nk, st, len, src, pos * (WAVE * BFS_UNROLL) + lane, WAVE, mv, ok);
        if (final) {
#pragma unroll
          for (int u = 0; u < BFS_UNROLL; ++u)
            if (ok[u]) {
              ++cnt;
              hsum += tuple_term(qid, a.j.ids[mv[u]]);
            }
        } else {
          const uint32_t n = stage_step(G, mv, ok, true, 0);
          wave_sync();
          const uint32_t done = drain(a, acc, slots, G, skip, n);
          wave_sync();
          if (done < n) {
            skip = done;
            full = true;
            break;
          }
          skip = 0;
        }
      }
      if (final) {
        const unsigned long long c = wave_sum(cnt), h = wave_sum64(hsum);
        if (lane == 0) add_last(acc[plan], c, h * (((unsigned long long)row[1] << 32) | row[0]));
      }
      if (full) break;
    }
    idx += rows_at_once;
    pos = first_pos;
    skip = 0;
  }
  if (lane == 0) cur[0] = {idx, pos, skip};

  // short rows: 16 lanes each, four per wave
  const uint32_t nshort = min(a.cin[0], a.cap_in);
  const uint32_t gi = lane / GROUP, gl = lane % GROUP;
  constexpr uint32_t PER = WAVE / GROUP;
  const uint32_t nquad = (nshort + PER - 1) / PER;
  idx = wave, pos = 0, skip = 0;
  if (a.resume) idx = uniform(cur[1].idx), pos = uniform(cur[1].pos), skip = uniform(cur[1].skip);
  while (!full && idx < nquad) {
    const uint32_t r = idx * PER + gi;
    const uint32_t* row = a.rows_in + (uint64_t)min(r, nshort - 1) * a.stride_in;
    uint32_t len = r < nshort ? row[R_LEN] : 0u;
    if (__any(len != 0)) {
      uint32_t plan = 0, st = 0, src = 0;
      if (len) {
        plan = row[R_PLAN];
        st = row[R_START];
        src = row[R_SRC];
        if (a.j.budget && a.j.out[a.j.plans[plan].out].aborted) len = 0;
      }
      const JoinPlan& P = a.j.plans[plan];
      const CetDesc& d = a.j.cets[P.cet[nk]];
      const bool final = nk + 1 == P.q;
      const uint32_t qid = P.order[nk];
      if (gl == 0) G.row[gi] = row;
      wave_sync();
      unsigned long long hsum = 0;
      uint32_t cnt = 0;
      for (; __any(pos < len); pos += GROUP * BFS_UNROLL) {
        uint32_t mv[BFS_UNROLL];
        bool ok[BFS_UNROLL];
        test_candidates(a, P, d, row + R_VAL, nk, st, len, src, pos + gl, GROUP, mv, ok);
        const uint32_t n = stage_step(G, mv, ok, !final, gi);
        if (n) {
          wave_sync();
          const uint32_t done = drain(a, acc, slots, G, skip, n);
          wave_sync();
          if (done < n) {  // this step again later: its last-level rows are not counted yet
            skip = done;
            full = true;
            break;
          }
        }
        skip = 0;
        if (final) {
#pragma unroll
          for (int u = 0; u < BFS_UNROLL; ++u)
            if (ok[u]) {
              ++cnt;
              hsum += tuple_term(qid, a.j.ids[mv[u]]);
            }
        }
      }
      // the group's sums end in its last lane
      if (__any(cnt != 0)) {
        unsigned long long c = cnt, h = hsum;
        c += dpp_or_0<0x111, 0xf>(c), h += dpp_or_0<0x111, 0xf>(h);
        c += dpp_or_0<0x112, 0xf>(c), h += dpp_or_0<0x112, 0xf>(h);
        c += dpp_or_0<0x114, 0xf>(c), h += dpp_or_0<0x114, 0xf>(h);
        c += dpp_or_0<0x118, 0xf>(c), h += dpp_or_0<0x118, 0xf>(h);
        if (gl == GROUP - 1 && c)
          add_last(acc[plan], c, h * (((unsigned long long)row[1] << 32) | row[0]));
      }
      wave_sync();
      if (full) break;
    }
    idx += nwaves;
    pos = 0;
    skip = 0;
  }
  if (lane == 0) {
    cur[1] = {idx, pos, skip};
    if (full) atomicAdd(a.pending, 1u);
  }
  if (a.rows_out) close_slots(a, slots);
  __syncthreads();
  flush_acc(a, acc);
}

}  // namespace

uint32_t bfs_row_words(uint32_t level) { return (R_VAL + level + 1 + 1) & ~1u; }

void launch_bfs_first(const BfsArgs& a, uint32_t nwg, hipStream_t s) {
  hipLaunchKernelGGL(bfs_first_kernel, dim3(nwg), dim3(256), sizeof(PlanAcc) * a.nplans, s, a);
}

void launch_bfs_expand(const BfsArgs& a, uint32_t nwg, hipStream_t s) {
  hipLaunchKernelGGL(bfs_expand_kernel, dim3(nwg), dim3(256), sizeof(PlanAcc) * a.nplans, s, a);
}

uint32_t bfs_resident_per_cu() {
  int per_cu = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, bfs_expand_kernel, 256, sizeof(PlanAcc) * BFS_PLANS) !=
          hipSuccess ||
      per_cu < 1) {
    (void)hipGetLastError();
    per_cu = 1;
  }
  return (uint32_t)per_cu;
}

}  // namespace gpsm
