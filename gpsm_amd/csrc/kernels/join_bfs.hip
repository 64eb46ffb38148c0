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
//    the learned order (finish_rows), from a back edge's bound vertex with fewer
//    neighbours of the label (tested against C(w) and the parent's edge instead);
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
static_assert(bfs_row_words(1) == ((R_VAL + 2 + 1) & ~1u), "a row's words");
constexpr uint32_t GROUP = 16;         // lanes per short row (one DPP row)
constexpr uint32_t LONG_LIST = 512;    // candidates above which workgroups take the row
constexpr int BFS_UNROLL = 4;          // candidates in flight per lane
constexpr uint32_t STAGE = WAVE * BFS_UNROLL;  // staged survivors of a wave's step

struct PlanAcc {
  unsigned long long cnt, hash, rows, work;
};

struct WaveStage {
  uint32_t mv[STAGE];
  uint32_t lane0[STAGE];  // first lane of the group whose row the survivor extends
};

// What a launch needs of a plan, in LDS: the table its rows' candidates come
// from (position nk = level + 1 is bound) and the one of the rows written.
// Read from the plans and tables themselves, a row's first candidate waited
// for six loads, each with the address of the one before, its first test for
// four more; most rows have one or two steps of candidates.
struct PlanLevel {
  uint64_t list, off;      // list arena: the lists; offsets arena: the next table's offsets
  uint32_t w_slot, w_lo;   // C(w) of the candidates, a key of their label
  uint32_t x_slot, w_lo2;  // the next table: C(x) its candidates are ranked in, a key of their label
  uint32_t inj, qid;
  uint8_t par, nb, par2, nb2, final, pad[3];
  uint8_t backs[BFS_MAXQ], backs2[BFS_MAXQ];
};

__device__ __forceinline__ void load_plans(const BfsArgs& a, PlanLevel* L) {
  const uint32_t nk = a.level + 1;
  for (uint32_t i = threadIdx.x; i < a.nplans; i += blockDim.x) {
    const JoinPlan& P = a.j.plans[i];
    PlanLevel p = {};
    if (nk < P.q) {
      p.qid = P.order[nk];
      p.final = nk + 1 == P.q;
      if (nk >= 2) {
        const CetDesc& d = a.j.cets[P.cet[nk]];
        p.list = d.list_base;
        p.w_slot = d.w_slot;
        p.w_lo = d.w_lo;
        p.inj = (uint32_t)P.inj[nk];
        p.par = (uint8_t)P.par[nk];
        p.nb = (uint8_t)(P.back_off[nk + 1] - P.back_off[nk]);
        for (uint32_t b = 0; b < p.nb; ++b) p.backs[b] = P.backs[P.back_off[nk] + b];
      }
      if (!p.final) {
        const CetDesc& d = a.j.cets[P.cet[nk + 1]];
        p.off = d.off_base;
        p.x_slot = d.x_slot;
        p.w_lo2 = d.w_lo;
        p.par2 = (uint8_t)P.par[nk + 1];
        p.nb2 = (uint8_t)(P.back_off[nk + 2] - P.back_off[nk + 1]);
        for (uint32_t b = 0; b < p.nb2; ++b) p.backs2[b] = P.backs[P.back_off[nk + 1] + b];
      }
    }
    L[i] = p;
  }
}

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

// Finishes one new row per lane (has: the lane holds one): val(c), c <= k, are
// the vertices of the row it extends (all lanes call it together), mv the
// vertex at position k + 1 and hash the row's product.  Finds the list that
// extends it, counts it, and writes its record unless it has no candidates.
// All lanes of the wave call; false, with nothing written or counted, when the
// level's buffer is full.
template <typename Val>
__device__ __forceinline__ bool finish_rows(const BfsArgs& a, const PlanLevel* plans, PlanAcc* acc, Slots& slots,
                                            bool has, Val val, uint32_t k, uint32_t plan, uint32_t mv,
                                            unsigned long long hash) {
  const uint32_t lane = lane_id();
  const unsigned long long bh = __ballot(has);
  if (!bh) return true;
  const PlanLevel& p = plans[plan];
  uint32_t st = 0, len = 0, src = 0, full = 0;
  const uint32_t pp = has ? p.par2 : 0u;
  const uint32_t bound = val(min(pp, k));
  if (has) {
    const uint32_t x = pp == k + 1 ? mv : bound;
    const uint32_t j = rank_of(a.j.bitmaps + (size_t)p.x_slot * a.j.W, a.j.bprefix + (size_t)p.x_slot * a.j.W, x);
    const uint32_t* off = a.j.offsets + p.off;
    st = off[j];
    full = off[j + 1] - st;
    len = full;
  }
  // A back edge's vertex with fewer neighbours of the label is the cheaper
  // source, although its candidates take two tests more: 32 cycles and cliques
  // on an R-MAT 18 graph take 21.6 ms from the parents' lists alone, 16.0 /
  // 14.2 / 13.6 ms with those less than 1/4, 1/2, 4/5 as long.  Rows, work,
  // counts and hashes do not depend on it, and nothing in a heuristic plan rules
  // it out.  It is off there for one reason: the 16 cliques on the R-MAT 22 graph
  // are expected to join with the learned order in at most 0.8 times the
  // heuristic order's time (tests/test_gpu_configs.py).  With it for both orders
  // they take 137 ms (learned) and 125 (heuristic), so the expectation holds
  // through this rule only: 137 and 320 ms as it is.
  const uint32_t nb = a.any_source && has ? p.nb2 : 0u;
  for (uint32_t b = 0; __any(b < nb); ++b) {
    const uint32_t c = b < nb ? p.backs2[b] : 0u;
    const uint32_t at = val(min(c, k));
    if (b < nb && full) {
      uint32_t r0, dg;
      piece(a.j.pieces, c == k + 1 ? mv : at, p.w_lo2, r0, dg);
      if ((uint64_t)dg + dg / 4 < len) {
        st = r0;
        len = dg;
        src = 1 + b;
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
    dst[R_VAL + k + 1] = mv;
  }
  if (bs | bl)
    for (uint32_t c = 0; c <= k; ++c) {
      const uint32_t v = val(c);
      if (dst) dst[R_VAL + c] = v;
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
  PlanLevel* plans = reinterpret_cast<PlanLevel*>(acc + a.nplans);
  for (uint32_t i = threadIdx.x; i < a.nplans; i += blockDim.x) acc[i] = {0, 0, 0, 0};
  load_plans(a, plans);
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
    finish_rows(a, plans, acc, slots, has, [&](uint32_t) { return mu; }, 0, plan, mv, h);
  }
  close_slots(a, slots);
  __syncthreads();
  flush_acc(a, acc);
}

// A row as its lanes hold it: lane lane0 + i has word i of the record, and lane
// lane0 + b what the test of back edge b needs (its vertex and hub index, or
// where it is none its entries towards the candidates' label).
struct RowRegs {
  uint32_t lane0, word, hub, p0, n;
  __device__ __forceinline__ uint32_t get(uint32_t i) const { return __shfl(word, lane0 + i, WAVE); }
};

// Looks the back edges' vertices up (len: lanes of a row with candidates).
__device__ __forceinline__ void load_backs(const BfsArgs& a, const PlanLevel& p, RowRegs& r, uint32_t src, bool live) {
  const uint32_t b = lane_id() - r.lane0;
  const bool mine = live && b < p.nb;
  // the source's own edge holds; the parent's is tested in its place
  const uint32_t c = mine ? (src == 1 + b ? p.par : p.backs[b]) : 0u;
  const uint32_t bv = r.get(R_VAL + c);
  r.hub = ~0u;
  r.p0 = r.n = 0;
  if (mine) {
    r.hub = a.j.hub_of[bv];
    if (r.hub == ~0u) piece(a.j.pieces, bv, p.w_lo, r.p0, r.n);
  }
}

// The candidates idx, idx + step, ... (BFS_UNROLL of them, below len) of a
// row: ok[u] and mv[u].  All lanes of the wave call (len 0: no row).
__device__ __forceinline__ void test_candidates(const BfsArgs& a, const PlanLevel& p, const RowRegs& r, uint32_t st,
                                                uint32_t len, uint32_t src, uint32_t idx, uint32_t step,
                                                uint32_t (&mv)[BFS_UNROLL], bool (&ok)[BFS_UNROLL]) {
  const uint32_t* from = src ? a.j.col + st : a.j.lists + p.list + st;
#pragma unroll
  for (int u = 0; u < BFS_UNROLL; ++u) {
    ok[u] = idx + u * step < len;
    mv[u] = ok[u] ? from[idx + u * step] : 0u;
  }
  if (src) {
    // from an adjacency: in C(w), and adjacent to the parent
    const uint32_t* bm_w = a.j.bitmaps + (size_t)p.w_slot * a.j.W;
    uint32_t wd[BFS_UNROLL];
#pragma unroll
    for (int u = 0; u < BFS_UNROLL; ++u) wd[u] = ok[u] ? bm_w[mv[u] >> 5] >> (mv[u] & 31) : 0u;
#pragma unroll
    for (int u = 0; u < BFS_UNROLL; ++u) ok[u] = ok[u] && (wd[u] & 1u);
  }
  for (uint32_t m = len ? p.inj : 0u; __any(m != 0); m &= m - 1) {
    const uint32_t c = r.get(R_VAL + (m ? (uint32_t)__ffs((int)m) - 1 : 0u));
#pragma unroll
    for (int u = 0; u < BFS_UNROLL; ++u) ok[u] = ok[u] && !(m && mv[u] == c);
  }
  const uint32_t nb = len ? p.nb : 0u;
  for (uint32_t b = 0; __any(b < nb); ++b) {
    const uint32_t hub = __shfl(r.hub, r.lane0 + b, WAVE);
    const uint32_t p0 = __shfl(r.p0, r.lane0 + b, WAVE);
    uint32_t n = __shfl(r.n, r.lane0 + b, WAVE);
    if (b >= nb) continue;
    if (hub != ~0u) {
      const uint32_t* bm = a.j.hub_bits + (size_t)hub * a.j.W;
      uint32_t wd[BFS_UNROLL];
#pragma unroll
      for (int u = 0; u < BFS_UNROLL; ++u) wd[u] = ok[u] ? bm[mv[u] >> 5] >> (mv[u] & 31) : 0u;
#pragma unroll
      for (int u = 0; u < BFS_UNROLL; ++u) ok[u] = ok[u] && (wd[u] & 1u);
    } else {
      // a short row: its piece towards the candidates' label is shorter still
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
__device__ __forceinline__ uint32_t drain(const BfsArgs& a, const PlanLevel* plans, PlanAcc* acc, Slots& slots,
                                          const WaveStage& G, const RowRegs& regs, uint32_t from, uint32_t n) {
  const uint32_t lane = lane_id();
  for (uint32_t s0 = from; s0 < n; s0 += WAVE) {
    const bool has = s0 + lane < n;
    const uint32_t mv = has ? G.mv[s0 + lane] : 0u;
    RowRegs r = regs;
    r.lane0 = has ? G.lane0[s0 + lane] : 0u;
    const uint32_t row_plan = r.get(R_PLAN), plan = has ? row_plan : 0u;
    unsigned long long h = ((unsigned long long)r.get(1) << 32) | r.get(0);
    if (has) h *= tuple_term(plans[plan].qid, a.j.ids[mv]);
    if (!finish_rows(a, plans, acc, slots, has, [&](uint32_t c) { return r.get(R_VAL + c); }, a.level, plan, mv, h))
      return s0;
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
                                               const bool (&ok)[BFS_UNROLL], bool keep, uint32_t lane0) {
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
      G.lane0[at] = lane0;
    }
    n += (uint32_t)__popcll(bal);
  }
  return n;
}

// Eight waves per SIMD: 32 cycles and cliques on an R-MAT 18 graph 20.5-24.2
// ms, 21.5-25.4 at six, 23.2-27.4 at five and four.  Bound by what a CU can
// gather: a list entry and 1 to 2 back-edge bits a candidate, 2e9 candidates
// and 4e9 loads in 20 ms; with the vertices numbered by label a hub bitmap's
// bits of one label are a few lines, and 3 GB of 32 ms' worth come from HBM.
// Level a.level -> a.level + 1.  A wave's place in the level's rows is a
// cursor per kind of row: the row (or quad of rows), the step of its
// candidates, and the step's survivors already written.
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(8))) bfs_expand_kernel(BfsArgs a) {
  extern __shared__ unsigned char lds_raw[];
  PlanAcc* acc = reinterpret_cast<PlanAcc*>(lds_raw);
  PlanLevel* plans = reinterpret_cast<PlanLevel*>(acc + a.nplans);
  __shared__ WaveStage stage[4];
  const uint32_t lane = lane_id(), wv = threadIdx.x / WAVE;
  WaveStage& G = stage[wv];
  for (uint32_t i = threadIdx.x; i < a.nplans; i += blockDim.x) acc[i] = {0, 0, 0, 0};
  load_plans(a, plans);
  __syncthreads();
  Slots slots = {0, 0};
  const uint32_t words = R_VAL + a.level + 1;  // of a row
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
    RowRegs r = {};
    r.word = lane < words ? a.long_in[(uint64_t)idx * a.stride_in + lane] : 0u;
    const uint32_t plan = uniform(r.get(R_PLAN)), st = uniform(r.get(R_START)), src = uniform(r.get(R_SRC));
    uint32_t len = uniform(r.get(R_LEN));
    if (len) {  // 0: reserved, not written
      if (a.j.budget && uniform((uint32_t)a.j.out[a.j.plans[plan].out].aborted)) len = 0;
      const PlanLevel& p = plans[plan];
      const bool final = p.final;
      const uint32_t qid = p.qid;
      load_backs(a, p, r, src, len != 0);
      unsigned long long hsum = 0;
      uint32_t cnt = 0;
      for (; pos * (WAVE * BFS_UNROLL) < len; pos += share * (256 / WAVE)) {
        uint32_t mv[BFS_UNROLL];
        bool ok[BFS_UNROLL];
        test_candidates(a, p, r, st, len, src, pos * (WAVE * BFS_UNROLL) + lane, WAVE, mv, ok);
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
          const uint32_t done = drain(a, plans, acc, slots, G, r, skip, n);
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
        const unsigned long long of_row = ((unsigned long long)r.get(1) << 32) | r.get(0);
        if (lane == 0) add_last(acc[plan], c, h * of_row);
      }
      if (full) break;
    }
    idx += rows_at_once;
    pos = first_pos;
    skip = 0;
  }
  if (lane == 0) cur[0] = {idx, pos, skip, 0};

  // short rows: 16 lanes each, four per wave; the next quad's rows load while
  // this one's candidates are tested
  const uint32_t nshort = min(a.cin[0], a.cap_in);
  const uint32_t gi = lane / GROUP, gl = lane % GROUP;
  constexpr uint32_t PER = WAVE / GROUP;
  static_assert(R_VAL + BFS_MAXQ <= GROUP, "a row's words fit its lanes");
  const uint32_t nquad = (nshort + PER - 1) / PER;
  idx = wave, pos = 0, skip = 0;
  if (a.resume) idx = uniform(cur[1].idx), pos = uniform(cur[1].pos), skip = uniform(cur[1].skip);
  auto word_of = [&](uint32_t i) {
    const uint64_t row = (uint64_t)i * PER + gi;
    return i < nquad && row < nshort && gl < words ? a.rows_in[row * a.stride_in + gl] : 0u;
  };
  uint32_t next = full ? 0u : word_of(idx);
  while (!full && idx < nquad) {
    RowRegs r = {};
    r.lane0 = gi * GROUP;
    r.word = next;
    next = word_of(idx < ~0u - nwaves ? idx + nwaves : ~0u);
    uint32_t len = r.get(R_LEN);
    if (__any(len != 0)) {
      // a reserved slot that holds no row has only its length
      const uint32_t row_plan = r.get(R_PLAN), st = r.get(R_START), row_src = r.get(R_SRC);
      const uint32_t plan = len ? row_plan : 0u, src = len ? row_src : 0u;
      // rows of a plan over its budget end here, but where part of a step is
      // written the step's rows are those it was saved with: skip counts the
      // survivors of them all
      if (len && a.j.budget &&
          (skip ? !((cur[1].rows >> gi) & 1u) : a.j.out[a.j.plans[plan].out].aborted != 0))
        len = 0;
      const PlanLevel& p = plans[plan];
      const bool final = p.final;
      const uint32_t qid = p.qid;
      load_backs(a, p, r, src, len != 0);
      unsigned long long hsum = 0;
      uint32_t cnt = 0;
      for (; __any(pos < len); pos += GROUP * BFS_UNROLL) {
        uint32_t mv[BFS_UNROLL];
        bool ok[BFS_UNROLL];
        test_candidates(a, p, r, st, len, src, pos + gl, GROUP, mv, ok);
        const uint32_t n = stage_step(G, mv, ok, !final, r.lane0);
        if (n) {
          wave_sync();
          const uint32_t done = drain(a, plans, acc, slots, G, r, skip, n);
          wave_sync();
          if (done < n) {  // this step again later: its last-level rows are not counted yet
            skip = done;
            full = true;
            const unsigned long long with = __ballot(len != 0);
            uint32_t rows = 0;
            for (uint32_t i = 0; i < PER; ++i) rows |= (uint32_t)((with >> (i * GROUP)) & 1u) << i;
            if (lane == 0) cur[1].rows = rows;
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
        const unsigned long long of_row = ((unsigned long long)r.get(1) << 32) | r.get(0);
        if (gl == GROUP - 1 && c) add_last(acc[plan], c, h * of_row);
      }
      wave_sync();
      if (full) break;
    }
    idx += nwaves;
    pos = 0;
    skip = 0;
  }
  if (lane == 0) {
    cur[1].idx = idx, cur[1].pos = pos, cur[1].skip = skip;
    if (full) atomicAdd(a.pending, 1u);
  }
  if (a.rows_out) close_slots(a, slots);
  __syncthreads();
  flush_acc(a, acc);
}

}  // namespace

void launch_bfs_first(const BfsArgs& a, uint32_t nwg, hipStream_t s) {
  hipLaunchKernelGGL(bfs_first_kernel, dim3(nwg), dim3(256), (sizeof(PlanAcc) + sizeof(PlanLevel)) * a.nplans, s, a);
}

void launch_bfs_expand(const BfsArgs& a, uint32_t nwg, hipStream_t s) {
  hipLaunchKernelGGL(bfs_expand_kernel, dim3(nwg), dim3(256), (sizeof(PlanAcc) + sizeof(PlanLevel)) * a.nplans, s, a);
}

uint32_t bfs_resident_per_cu(uint32_t nplans) {
  int per_cu = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, bfs_expand_kernel, 256,
                                                   (sizeof(PlanAcc) + sizeof(PlanLevel)) * nplans) !=
          hipSuccess ||
      per_cu < 1) {
    (void)hipGetLastError();
    per_cu = 1;
  }
  return (uint32_t)per_cu;
}

}  // namespace gpsm
