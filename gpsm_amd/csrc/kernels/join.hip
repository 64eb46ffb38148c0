// Join of candidate-edge tables on gfx950 (table_kernel, join_kernel,
// expand_kernel, link_kernel, filter_kernel; match/Match.cu:1141-1569).
//
// The reference materialises every intermediate table breadth-first, finds
// a row's vertex in the candidate list with a warp-linear scan (quadratic in
// rows x candidates), and leaves injectivity to the host.  Here:
//  * a persistent grid pulls tasks (every T-th row of one query's first
//    table) from a device counter, so hundreds of uneven queries share one
//    launch and hub rows are spread over a query's T tasks;
//  * each workgroup walks its slice depth-first through levels k = 1..q-1
//    (k+1 bound vertices) with one bounded column-major buffer per level, so
//    memory is O(cap * q^2) per workgroup whatever the result size;
//  * a row's candidate list is found in O(1) through the rank index of C(x)
//    (set bits before each word + a popcount);
//  * a window of 256 rows is expanded flattened: 256 threads take 256
//    consecutive (row, candidate) pairs, so rows of any fan-out share lanes;
//  * join-mode edges become edge-membership checks (binary search in the
//    shorter adjacency) and injectivity is checked in the same pass;
//  * the tuple hash is a product of one factor per (query vertex, image)
//    pair, so a row carries the product of its factors, and the embeddings
//    that extend a row hash to that product times a sum of last factors;
//  * where the last one or two vertices have no back edges and no tuples are
//    wanted, their levels are not enumerated: a row's embeddings are counted
//    and hashed from sums kept per candidate (CetAgg), with the injectivity
//    checks as exact corrections (count_last_level, count_last_two).  On the
//    245-query mix on the 1M Chung-Lu graph (4.57e11 candidates of the last
//    levels) the join went from 437 to 9.0 ms and the batch from 467 to 32.6
//    ms, on one 4-vertex walk of 7e8 embeddings from 3.2 to 0.06 ms;
//  * otherwise the last level is enumerated but never written: an embedding
//    costs one multiply by its last factor (precomputed per list entry); a
//    wave expanding one long row sums the factors of its valid candidates
//    and multiplies once per row.
#include <algorithm>
#include <type_traits>

#include "edge.h"
#include "launch.h"
#include "wave.h"

namespace gpsm {

namespace {

constexpr uint32_t WROWS = 256;  // rows per window = threads per workgroup
static_assert((WROWS & (WROWS - 1)) == 0, "row indices are masked with WROWS - 1");
// candidates in flight per thread: cyclic plans, tree plans (with the
// waves per SIMD of the two kernels, below)
constexpr int EXP_UNROLL = 4;
constexpr int TREE_UNROLL = 3;
// At the last level a row with at least this many candidates is expanded by
// one wave on its own (no row search per candidate, the row's values
// uniform); shorter rows share lanes through the flattened expansion.
// Measured (join per batch): 96 equals 128 on the 1M Chung-Lu mix and is 1%
// faster on the R-MAT 22 shapes; 192 is 2% slower on the mix.
constexpr uint32_t LONG_ROW = 96;
static_assert((uint64_t)WROWS * LONG_ROW < (1u << 23) && WROWS < 512, "packed scan of short spans and long flags");

// The back-edge tests of a lane's EXP_UNROLL candidates of one row (row i
// of the window, the wave-per-row pass) against the bound vertices of
// positions P.backs[bo..be): those vertices are the same for the whole
// wave, so each one's hub index is read once, and when it is a hub the
// candidates' tests are bits of its bitmap, loaded together (one load per
// candidate and edge).  Otherwise the candidates' own hub indices are read
// together and a pair with no hub falls back to has_edge's binary search.
// A candidate whose test fails skips the later ones.  oks[u] in/out.
template <bool BYTES, int U>
__device__ __forceinline__ void back_edges_of_row(const JoinArgs& a, const JoinPlan& P,
                                                  const uint32_t* __restrict__ val, uint32_t bo, uint32_t be,
                                                  uint32_t w_lo, uint32_t i, const uint32_t (&mvs)[U],
                                                  bool (&oks)[U], unsigned long long& bytes) {
  for (uint32_t b = bo; b < be; ++b) {
    const uint32_t bv = uniform(val[P.backs[b] * WROWS + i]);
    const uint32_t hb = uniform(a.hub_of[bv]);
    if (hb != ~0u) {
      const uint32_t* bm = a.hub_bits + (size_t)hb * a.W;
      uint32_t w[U];
#pragma unroll
      for (int u = 0; u < U; ++u) w[u] = oks[u] ? bm[mvs[u] >> 5] >> (mvs[u] & 31) : 0u;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (BYTES && oks[u]) bytes += 12;  // two hub indices, one bitmap word
        oks[u] = oks[u] && (w[u] & 1u);
      }
    } else {
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (oks[u]) oks[u] = has_edge<BYTES>(a.pieces, a.col, a.hub_of, a.hub_bits, a.W, mvs[u], w_lo, bv, bytes);
    }
  }
}

// Row r of a task as a row of its query's first table.
__device__ __forceinline__ uint64_t task_row(const JoinTask& t, uint64_t r) {
  return (((r >> t.shift) * t.stride + t.first) << t.shift) | (r & ((1u << t.shift) - 1u));
}

struct JoinShared {
  uint32_t pre[WROWS + 1];
  uint32_t delta[WROWS];  // list position of a row's candidate g is delta[row] + g
  unsigned long long srow[WROWS];  // product of a row's hash factors
  uint32_t tmp[8];
  uint32_t fill[MAXQ], cur_row[MAXQ], cur_cand[MAXQ];
  unsigned long long lrows[MAXQ];
  unsigned long long lwork[MAXQ];
  uint32_t task, k, abort;
  unsigned long long red[4], agg[4][3];
  // last level: the window's long rows (row, list start, candidates) and
  // the candidates they hold
  uint32_t lrow[WROWS], lst[WROWS], lub[WROWS];
  uint32_t long_cands;
  // followed by the row window: val[c * WROWS + r], c < qmax
};

// A thread's share of the work and rows of the levels counted from records
// (counted, not enumerated): examined candidates and valid rows of the level
// before the last (two levels from records only), candidates of the last.
struct AggWork {
  unsigned long long work_y, rows_y, work_w;
};

// Adds the workgroup's shares to the task's and the query's counters and
// clears them; checks the work budget.  Contains __syncthreads.
__device__ __forceinline__ void flush_agg_work(const JoinArgs& a, const JoinPlan& P, JoinShared& S, uint32_t query,
                                               AggWork& aw) {
  const uint32_t w = threadIdx.x / WAVE;
  const unsigned long long v[3] = {wave_sum64(aw.work_y), wave_sum64(aw.rows_y), wave_sum64(aw.work_w)};
  aw = {0, 0, 0};
  __syncthreads();
  if (lane_id() == 0)
    for (int i = 0; i < 3; ++i) S.agg[w][i] = v[i];
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long t[3] = {0, 0, 0};
    for (uint32_t x = 0; x < WROWS / WAVE; ++x)
      for (int i = 0; i < 3; ++i) t[i] += S.agg[x][i];
    const uint32_t wl = P.q - 1;
    if (P.agg == 2) {
      S.lwork[wl - 1] += t[0];
      S.lrows[wl - 1] += t[1];
    }
    S.lwork[wl] += t[2];
    const unsigned long long done = t[0] + t[2];
    if (done) {
      const unsigned long long before = atomicAdd(&a.out[query].work, done);
      if (a.budget && before + done > a.budget) {
        a.out[query].aborted = 1;
        S.abort = 1;
      }
    }
  }
}

__device__ __forceinline__ CetAgg agg_of(const JoinArgs& a, const CetDesc& d, uint32_t x) {
  return a.aggs[d.agg_base + rank_of(a.bitmaps + (size_t)d.x_slot * a.W, a.bprefix + (size_t)d.x_slot * a.W, x)];
}

// Whether u is in the candidate-edge list of mu in table d: u in C(w) and
// {mu, u} an edge.
template <bool BYTES>
__device__ __forceinline__ bool in_list(const JoinArgs& a, const CetDesc& d, uint32_t mu, uint32_t u,
                                        unsigned long long& bytes) {
  if (!bit_of(a.bitmaps + (size_t)d.w_slot * a.W, u)) return false;
  return has_edge<BYTES>(a.pieces, a.col, a.hub_of, a.hub_bits, a.W, u, d.w_lo, mu, bytes);
}

// The embeddings of a window of rows that bind all but the last vertex w
// (which has no back position): a row has |L| of them, and their hash is the
// row's product times the sum of the list's terms, less the bound vertices
// that sit in the list (the injectivity checks of w).  One 32-byte record
// per row stands for its whole list.
template <bool BYTES>
__device__ __forceinline__ void count_last_level(const JoinArgs& a, const JoinPlan& P, const JoinShared& S,
                                                 const uint32_t* val, uint32_t nw, unsigned long long& my_cnt,
                                                 unsigned long long& my_hash, unsigned long long& bytes,
                                                 AggWork& aw) {
  const uint32_t tid = threadIdx.x, w = P.q - 1;
  if (tid >= nw) return;
  const CetDesc& d = a.cets[P.cet[w]];
  const uint32_t qid = P.order[w];
  const uint32_t mu = val[P.par[w] * WROWS + tid];
  const CetAgg r = agg_of(a, d, mu);
  if (BYTES) bytes += 4 + 4 + sizeof(CetAgg);
  unsigned long long len = r.len, s = r.s;
  for (uint64_t m = P.inj[w]; m; m &= m - 1) {
    const uint32_t u = val[(uint32_t)(__ffsll((long long)m) - 1) * WROWS + tid];
    if (in_list<BYTES>(a, d, mu, u, bytes)) {
      --len;
      s -= tuple_term(qid, a.ids[u]);
    }
  }
  my_cnt += len;
  my_hash += S.srow[tid] * s;
  aw.work_w += r.len;
}

// The embeddings of a window of rows that bind all but the last two
// vertices y (position q - 2) and w, neither with a back position.  For a
// row, with L_y the list of y's parent and L_w(v) that of w's:
//   w's parent is y:  sum over v in L_y of |L_w(v)| (CetAgg a, b)
//   otherwise:        |L_y| * |L_w|
// less, by injectivity (vertices of one label only), exactly:
//   bound vertices in L_y (one record of the last table each in the first
//   case), bound vertices in L_w (in the first case y's parent is in every
//   L_w(v); another bound vertex u is in those of the v adjacent to u), and
//   pairs v = w of L_y and L_w (a record where the parents are the same).
// Only the v of L_y adjacent to one other vertex (u, or w's parent) have no
// record: they are enumerated from the shorter of L_y and that vertex's
// adjacency.  A row costs O(1) records instead of |L_y| * |L_w| candidates.
template <bool BYTES>
__device__ __forceinline__ void count_last_two(const JoinArgs& a, const JoinPlan& P, JoinShared& S,
                                               const uint32_t* val, uint32_t nw, unsigned long long& my_cnt,
                                               unsigned long long& my_hash, unsigned long long& bytes, AggWork& aw) {
  const uint32_t tid = threadIdx.x, lane = lane_id();
  const uint32_t w = P.q - 1, y = w - 1, py = P.par[y], pw = P.par[w];
  const CetDesc& dy = a.cets[P.cet[y]];
  const CetDesc& dw = a.cets[P.cet[w]];
  const uint32_t qy = P.order[y], qw = P.order[w];
  const uint64_t iy = P.inj[y], iw = P.inj[w];
  const bool chain = pw == y, sibling = pw == py;
  const uint32_t* bm_w = a.bitmaps + (size_t)dw.w_slot * a.W;
  uint32_t mu = 0, st_y = 0, len_y = 0;
  if (tid < nw) {
    mu = val[py * WROWS + tid];
    const CetAgg r = agg_of(a, dy, mu);
    if (BYTES) bytes += 4 + 4 + sizeof(CetAgg);
    st_y = r.off;
    len_y = r.len;
    unsigned long long n = r.len, ty = r.s, ra = r.a, rb = r.b;
    for (uint64_t m = iy; m; m &= m - 1) {
      const uint32_t u = val[(uint32_t)(__ffsll((long long)m) - 1) * WROWS + tid];
      if (!in_list<BYTES>(a, dy, mu, u, bytes)) continue;
      const unsigned long long t = tuple_term(qy, a.ids[u]);
      --n;
      ty -= t;
      if (chain) {
        const CetAgg x = agg_of(a, dw, u);
        if (BYTES) bytes += 4 + 4 + sizeof(CetAgg);
        ra -= x.len;
        rb -= t * x.s;
      } else if (sibling && bit_of(bm_w, u)) {
        --ra;
        rb -= t * tuple_term(qw, a.ids[u]);
      }
    }
    unsigned long long cnt, hash;
    if (chain) {
      aw.work_w += ra;
      cnt = ra;
      hash = rb;
      if (((iw >> py) & 1) && bit_of(bm_w, mu)) {  // y's parent is in every list
        cnt -= n;
        hash -= tuple_term(qw, a.ids[mu]) * ty;
      }
    } else {
      const uint32_t mw = val[pw * WROWS + tid];
      const CetAgg x = agg_of(a, dw, mw);
      if (BYTES) bytes += 4 + 4 + sizeof(CetAgg);
      aw.work_w += n * x.len;
      unsigned long long lw = x.len, sw = x.s;
      for (uint64_t m = iw & ~(1ull << y); m; m &= m - 1) {
        const uint32_t u = val[(uint32_t)(__ffsll((long long)m) - 1) * WROWS + tid];
        if (in_list<BYTES>(a, dw, mw, u, bytes)) {
          --lw;
          sw -= tuple_term(qw, a.ids[u]);
        }
      }
      cnt = n * lw;
      hash = ty * sw;
      if (sibling && ((iw >> y) & 1)) {
        cnt -= ra;
        hash -= rb;
      }
    }
    aw.work_y += len_y;
    aw.rows_y += n;
    my_cnt += cnt;
    my_hash += S.srow[tid] * hash;
  }
  // The v of L_y adjacent to one other vertex o per row: in the first case
  // the bound vertices of w's label except y's parent, one position at a
  // time, else w's parent (v also in C(w)) when y has w's label.
  uint64_t pos = chain ? iw & ~(1ull << py) : !sibling && ((iw >> y) & 1) ? 1ull << pw : 0ull;
  for (; pos; pos &= pos - 1) {  // uniform
    const uint32_t c = (uint32_t)(__ffsll((long long)pos) - 1);
    uint32_t o = 0, len = 0, st = 0, side = 0;
    if (tid < nw && len_y) {
      o = val[c * WROWS + tid];
      if (!chain || bit_of(bm_w, o)) {
        // the cheaper side: L_y against o's hub bitmap or adjacency, or o's
        // adjacency against C(y) and the edge to y's parent (a bit test about
        // 2, a binary search about 8 list reads)
        uint32_t o0, od;
        piece(a.pieces, o, dy.w_lo, o0, od);
        const uint64_t c0 = (uint64_t)len_y * (a.hub_of[o] != ~0u ? 2 : 8);
        const uint64_t c1 = (uint64_t)od * (a.hub_of[mu] != ~0u ? 2 : 8);
        side = c1 < c0;
        len = side ? od : len_y;
        st = side ? o0 : st_y;
        if (BYTES) bytes += 16;
      }
    }
    __syncthreads();  // the previous position's reads of S are done
    uint32_t T;
    const uint32_t ex = block_excl_scan(len, S.tmp, &T);
    S.pre[tid] = tid < nw ? ex : T;
    S.delta[tid] = st - ex;
    S.lst[tid] = o;
    S.lub[tid] = mu;
    S.lrow[tid] = side;
    __syncthreads();
    constexpr int U = 2;
    for (uint32_t f = 0; f < T; f += WROWS * U) {
      const uint32_t g0 = f + (tid / WAVE) * (WAVE * U);
      if (g0 >= T) break;  // the whole wave; no barrier below
      uint32_t is[U], v[U];
#pragma unroll
      for (int u = 0; u < U; ++u) is[u] = min(g0 + u * WAVE + lane, T - 1);
      halving_search<U>(S.pre, uniform(nw), is);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const uint32_t e = S.delta[is[u]] + min(g0 + u * WAVE + lane, T - 1);
        v[u] = S.lrow[is[u]] ? a.col[e] : a.lists[dy.list_base + e];
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const uint32_t i = is[u];
        bool ok = g0 + u * WAVE + lane < T;
        if (BYTES && ok) bytes += 4;
        for (uint64_t m = iy; m; m &= m - 1) ok &= val[(uint32_t)(__ffsll((long long)m) - 1) * WROWS + i] != v[u];
        if (ok && !chain) ok = bit_of(bm_w, v[u]);
        if (ok) {
          const bool sd = S.lrow[i] != 0;
          if (sd) ok = bit_of(a.bitmaps + (size_t)dy.w_slot * a.W, v[u]);
          if (ok) ok = has_edge<BYTES>(a.pieces, a.col, a.hub_of, a.hub_bits, a.W, v[u], dy.w_lo, sd ? S.lub[i] : S.lst[i], bytes);
        }
        if (ok) {
          --my_cnt;
          my_hash -= S.srow[i] * tuple_term(qy, a.ids[v[u]]) * tuple_term(qw, a.ids[chain ? S.lst[i] : v[u]]);
        }
      }
    }
  }
}

// BYTES: account the algorithmic bytes read and written (JoinOut::bytes);
// the kernel without it is the one timed.  KIND: the plans of the launch, each
// kind a kernel with its own register budget.  Tree plans have no back edges
// (join-mode edges) and their kernels no back-edge code: sharing the cyclic
// kernel's registers made them 1.2-1.6x slower.  The kernels that count the
// last levels from records hold no code that enumerates them: one cyclic
// kernel with both spilled 40 registers and ran R-MAT 18 cycles and cliques
// 1.2x slower than the two apart.
template <bool BYTES, JoinKind KIND>
__device__ __forceinline__ void join_body(const JoinArgs& a) {
  constexpr bool CYCLIC = KIND == JOIN_CYCLIC || KIND == JOIN_CYCLIC_ENUM;
  constexpr bool COUNTED = KIND == JOIN_TREE || KIND == JOIN_CYCLIC;  // every plan of the launch has agg > 0 (or q = 2)
  constexpr int XU = CYCLIC ? EXP_UNROLL : TREE_UNROLL;
  extern __shared__ unsigned char lds_raw[];
  JoinShared& S = *reinterpret_cast<JoinShared*>(lds_raw);
  uint32_t* val = reinterpret_cast<uint32_t*>(lds_raw + ((sizeof(JoinShared) + 15) & ~(size_t)15));
  const uint32_t tid = threadIdx.x;
  uint32_t* lvl_base = a.levels + (uint64_t)blockIdx.x * a.level_stride;

  for (;;) {
    if (tid == 0) S.task = atomicAdd(a.task_counter, 1u);
    __syncthreads();
    const uint32_t t = S.task;
    if (t >= a.ntasks) return;
    const JoinTask task = a.tasks[t];
    const JoinPlan& P = a.plans[task.query];
    const uint32_t q = P.q;
    const CetDesc d0 = a.cets[P.first_cet];
    const uint32_t* off0 = a.offsets + d0.off_base;
    const uint32_t* cl0 = a.clist + d0.clist_off;
    const uint32_t* ls0 = a.lists + d0.list_base;
    unsigned long long my_cnt = 0, my_hash = 0, my_bytes = 0;
    unsigned long long wave_cnt = 0;  // last-level embeddings of this wave (uniform)
    AggWork aw = {0, 0, 0};           // this thread's share of the levels counted from records

    if (tid < MAXQ) {
      S.lrows[tid] = 0;
      S.lwork[tid] = 0;
      S.fill[tid] = 0;
      S.cur_row[tid] = 0;
      S.cur_cand[tid] = 0;
    }
    __syncthreads();
    if (tid == 0) {
      S.fill[1] = (uint32_t)task.count;
      S.lrows[1] = task.count;
      S.lwork[1] = task.count;
      S.k = 1;
      // a query already over its work budget skips its remaining tasks
      S.abort = a.budget ? (uint32_t)__hip_atomic_load(&a.out[task.query].aborted, __ATOMIC_RELAXED,
                                                       __HIP_MEMORY_SCOPE_AGENT)
                         : 0u;
      if (S.abort) {
        S.fill[1] = S.lwork[1] = 0;
      } else {
        // first-table rows are join work too (the whole join of a 2-vertex query)
        const unsigned long long before = atomicAdd(&a.out[task.query].work, (unsigned long long)task.count);
        if (a.budget && before + task.count > a.budget) {
          a.out[task.query].aborted = 1;
          S.abort = 1;
          S.fill[1] = 0;
        }
      }
    }
    __syncthreads();

    if (q == 2) {
      // the first table is the embedding set
      for (uint64_t i = tid; i < task.count && !S.abort; i += blockDim.x) {
        const uint64_t e = task_row(task, i);
        const uint32_t j = seg_search(off0, d0.ncand + 1, (uint32_t)e);
        const uint32_t mu = cl0[j], mv = ls0[e];
        my_hash += tuple_term(P.order[0], a.ids[mu]) * tuple_term(P.order[1], a.ids[mv]);
        ++my_cnt;
        if (a.emit) {
          const unsigned long long pos = atomicAdd(a.emit_ctr, 1ULL);
          if (pos < a.emit_cap) {
            a.emit[pos * 2 + P.order[0]] = a.ids[mu];
            a.emit[pos * 2 + P.order[1]] = a.ids[mv];
          }
        }
      }
    } else {
      for (;;) {
        if (S.abort) break;  // uniform: set by thread 0 before the last barrier
        const uint32_t k = S.k;
        if (S.cur_row[k] >= S.fill[k]) {
          __syncthreads();
          if (k == 1) break;
          if (tid == 0) S.k = k - 1;
          __syncthreads();
          continue;
        }
        const uint32_t r0 = S.cur_row[k];
        const uint32_t nw = min(WROWS, S.fill[k] - r0);
        const uint32_t nk = k + 1;              // level being produced
        // this window's embeddings come from the records of the last levels
        const bool agg = COUNTED && nk + P.agg == q;
        const bool final = !COUNTED && nk == q - 1;
        const uint32_t p = P.par[nk];
        const CetDesc dn = a.cets[P.cet[nk]];
        const uint32_t* bm_x = a.bitmaps + (size_t)dn.x_slot * a.W;
        const uint32_t* bp_x = a.bprefix + (size_t)dn.x_slot * a.W;
        const uint32_t* offn = a.offsets + dn.off_base;
        const uint32_t bo = P.back_off[nk], be = CYCLIC ? P.back_off[nk + 1] : bo;  // a tree plan has none
        const uint64_t inj = P.inj[nk];
        const uint32_t wn = P.order[nk];
        const uint32_t cap = a.cap;
        // level j (j >= 2, j+1 columns) starts at cap * (j(j+1)/2 - 3)
        const uint32_t* Lk = k >= 2 ? lvl_base + (uint64_t)cap * ((k * (k + 1)) / 2 - 3) : nullptr;
        uint32_t* Ln = final ? nullptr : lvl_base + (uint64_t)cap * ((nk * (nk + 1)) / 2 - 3);

        // load the window and each row's candidate range
        uint32_t ub = 0, st = 0;
        if (tid < nw) {
          const uint32_t r = r0 + tid;
          if (k == 1) {
            const uint64_t e = task_row(task, r);
            const uint32_t j = seg_search(off0, d0.ncand + 1, (uint32_t)e);
            val[0 * WROWS + tid] = cl0[j];
            val[1 * WROWS + tid] = ls0[e];
          } else {
            for (uint32_t c = 0; c <= k; ++c) val[c * WROWS + tid] = Lk[(uint64_t)c * cap + r];
          }
          unsigned long long s = 1;
          for (uint32_t c = 0; c <= k; ++c) s *= tuple_term(P.order[c], a.ids[val[c * WROWS + tid]]);
          S.srow[tid] = s;
          if (BYTES && agg) my_bytes += k == 1 ? 8 : 4 * (k + 1);
        }
        if constexpr (COUNTED) {
          if (agg) {  // uniform
            if (P.agg == 1) count_last_level<BYTES>(a, P, S, val, nw, my_cnt, my_hash, my_bytes, aw);
            else count_last_two<BYTES>(a, P, S, val, nw, my_cnt, my_hash, my_bytes, aw);
            // with a budget every window's work is checked, without one the
            // task's work is added once at its end
            if (a.budget) flush_agg_work(a, P, S, task.query, aw);
            __syncthreads();
            if (tid == 0) {
              S.cur_row[k] = r0 + nw;
              S.cur_cand[k] = 0;
            }
            __syncthreads();
            continue;
          }
        }
        if (tid < nw) {
          // row values, rank index (prefix + words) and the offset pair
          if (BYTES) my_bytes += (k == 1 ? 8 : 4 * (k + 1)) + 4 + 4 + 8;
          const uint32_t j = rank_of(bm_x, bp_x, val[p * WROWS + tid]);
          st = offn[j];
          ub = offn[j + 1] - st;
          if (tid == 0) {
            ub -= S.cur_cand[k];
            st += S.cur_cand[k];
          }
        }
        uint32_t T, nlong = 0;
        if (!final) {
          const uint32_t ex = block_excl_scan(ub, S.tmp, &T);
          S.pre[tid] = tid < nw ? ex : T;
          S.delta[tid] = st - ex;  // wraps; delta + g is in range for g in the row's span
          if (tid == 0) S.fill[nk] = 0;
        } else {
          // last level: long rows are listed for the wave-per-row pass, the
          // others get spans of the flattened pass (T = their candidates);
          // one scan of (short candidates << 9 | long flag)
          const bool lng = tid < nw && ub >= LONG_ROW;
          uint32_t tot;
          const uint32_t ex2 = block_excl_scan(((lng ? 0u : ub) << 9) | (lng ? 1u : 0u), S.tmp, &tot);
          T = tot >> 9;
          nlong = tot & 511u;
          S.pre[tid] = tid < nw ? ex2 >> 9 : T;
          S.delta[tid] = st - (ex2 >> 9);
          if (lng) {
            S.lrow[ex2 & 511u] = tid;
            S.lst[ex2 & 511u] = st;
            S.lub[ex2 & 511u] = ub;
          }
          if (tid == 0) S.long_cands = 0;
        }
        __syncthreads();

        // expand: XU candidates per thread per step, list loads in
        // flight together; rows of the next level are appended per wave (one
        // LDS atomic per wave; row order inside a level does not matter).
        // The last level and the others are separate instantiations.
        const uint32_t* lst = a.lists + dn.list_base;
        const uint32_t lane = lane_id();
        const unsigned long long below = lane ? (~0ULL >> (WAVE - lane)) : 0ULL;
        auto expand = [&](auto fin) -> uint32_t {
          constexpr bool FINAL = decltype(fin)::value;
          const unsigned long long* trm_n = FINAL ? a.terms + dn.term_base : nullptr;
          uint32_t f = 0;
          for (; f < T; f += WROWS * XU) {
            if constexpr (!FINAL) {
              // every thread reads fill before any wave appends in this step
              const uint32_t fl = S.fill[nk];
              __syncthreads();
              if (fl + WROWS * XU > cap) break;  // uniform
            }
            uint32_t mvs[XU], is[XU];
            unsigned long long trm[XU];
            // wave w takes the step's candidates g0 .. g0 + 255 (lane l: g0 +
            // 64u + l), so one pair of searches per wave brackets the rows they
            // fall in and each candidate searches only inside the bracket
            // (T > 0 here; indices past T are clamped to T - 1 throughout, so
            // the bracket holds the row of every clamped index)
            const uint32_t g0 = f + (tid / WAVE) * (WAVE * XU);
            uint32_t rlo, rn;
            {
              const uint32_t glast = min(g0 + WAVE * XU - 1, T - 1);
              uint32_t r = lane == 0 ? min(g0, T - 1) : glast;
              halving_search<1>(S.pre, uniform(nw), &r);
              rlo = uniform(__shfl(r, 0, WAVE));
              rn = uniform(__shfl(r, 1, WAVE)) - rlo + 1;
            }
            // each candidate's row inside the bracket, the XU
            // searches of a lane stepping together
            // a candidate index past T searches for T - 1 (its loads then
            // re-read the last candidate's entry, in bounds); the candidate
            // itself is masked out (is = WROWS)
            uint32_t rb[XU];
#pragma unroll
            for (int u = 0; u < XU; ++u) rb[u] = min(g0 + u * WAVE + lane, T - 1);
            halving_search<XU>(S.pre + rlo, rn, rb);
            // LDS reads of the XU candidates are issued together
            // (row offsets, then the bound vertices the checks compare
            // with), so a lane waits once per kind rather than once per
            // candidate
            uint32_t es[XU];
#pragma unroll
            for (int u = 0; u < XU; ++u) {
              const uint32_t g = g0 + u * WAVE + lane;
              const uint32_t i = rlo + rb[u];
              is[u] = g < T ? i : WROWS;
              es[u] = S.delta[i] + min(g, T - 1);
              trm[u] = 0;
            }
#pragma unroll
            for (int u = 0; u < XU; ++u) {
              mvs[u] = lst[es[u]];
              // last level: the entry's hash term, computed once per list entry
              if constexpr (FINAL) trm[u] = trm_n[es[u]];
            }
            bool oks[XU];
#pragma unroll
            for (int u = 0; u < XU; ++u) oks[u] = is[u] != WROWS;
            // injectivity: only the positions bound to a vertex of the same
            // label that no edge test already separates
            for (uint64_t m = inj; m; m &= m - 1) {
              const uint32_t c = (uint32_t)(__ffsll((long long)m) - 1);
#pragma unroll
              for (int u = 0; u < XU; ++u) oks[u] &= val[c * WROWS + (is[u] & (WROWS - 1))] != mvs[u];
            }
            if constexpr (!FINAL) {
              // join-mode edges, then one append to the next level for the
              // lane's XU candidates together: one LDS atomic per
              // wave and step instead of one per candidate
#pragma unroll
              for (int u = 0; u < XU; ++u) {
                if (oks[u]) {
                  if (BYTES) my_bytes += 4;  // the list entry
                  for (uint32_t b = bo; b < be && oks[u]; ++b)
                    oks[u] = has_edge<BYTES>(a.pieces, a.col, a.hub_of, a.hub_bits, a.W, mvs[u], dn.w_lo,
                                             val[P.backs[b] * WROWS + is[u]], my_bytes);
                }
              }
              unsigned long long bal[XU];
              uint32_t nbal = 0;
#pragma unroll
              for (int u = 0; u < XU; ++u) {
                bal[u] = __ballot(oks[u]);
                nbal += (uint32_t)__popcll(bal[u]);
              }
              uint32_t wbase = 0;
              if (lane == 0 && nbal) wbase = atomicAdd(&S.fill[nk], nbal);
              wbase = __shfl(wbase, 0, WAVE);
#pragma unroll
              for (int u = 0; u < XU; ++u) {
                if (oks[u]) {
                  const uint64_t r = wbase + __popcll(bal[u] & below);
                  for (uint32_t c = 0; c <= k; ++c) Ln[(uint64_t)c * cap + r] = val[c * WROWS + is[u]];
                  Ln[(uint64_t)nk * cap + r] = mvs[u];
                  if (BYTES) my_bytes += 4 * (nk + 1);
                }
                wbase += (uint32_t)__popcll(bal[u]);
              }
            }
            if constexpr (FINAL) {
#pragma unroll
              for (int u = 0; u < XU; ++u) {
                const uint32_t i = is[u], mv = mvs[u];
                bool ok = oks[u];
                if (ok) {
                  if (BYTES) my_bytes += 4;  // the list entry (its hash term is a derived copy of it)
                  for (uint32_t b = bo; b < be && ok; ++b)
                    ok = has_edge<BYTES>(a.pieces, a.col, a.hub_of, a.hub_bits, a.W, mv, dn.w_lo, val[P.backs[b] * WROWS + i],
                                         my_bytes);
                }
                wave_cnt += __popcll(__ballot(ok));
                if (ok) {
                  my_hash += S.srow[i] * trm[u];
                  if (a.emit) {
                    const unsigned long long pos = atomicAdd(a.emit_ctr, 1ULL);
                    if (pos < a.emit_cap) {
                      uint32_t* t = a.emit + pos * q;
                      for (uint32_t c = 0; c <= k; ++c) t[P.order[c]] = a.ids[val[c * WROWS + i]];
                      t[wn] = a.ids[mv];
                    }
                  }
                }
              }
            }
            if constexpr (!FINAL) __syncthreads();
          }
          return f;
        };
        if (!COUNTED && final && nlong) {
          // wave-per-row pass over the window's long rows: lanes take
          // consecutive list entries of one row, whose values are uniform
          const unsigned long long* trm_n = a.terms + dn.term_base;
          for (uint32_t j = tid / WAVE; j < nlong; j += WROWS / WAVE) {
            const uint32_t i = uniform(S.lrow[j]);
            const uint32_t st_r = uniform(S.lst[j]), n_r = uniform(S.lub[j]);
            const unsigned long long srow = S.srow[i];
            unsigned long long rsum = 0;  // this lane's factors of the row's valid candidates
            if (lane == 0) atomicAdd(&S.long_cands, n_r);
            for (uint32_t g0 = 0; g0 < n_r; g0 += WAVE * XU) {
              uint32_t mvs[XU];
              unsigned long long trm[XU];
              bool oks[XU];
              // every lane loads (a lane past the row's end re-reads its
              // last entry, n_r >= LONG_ROW > 0): no branch per candidate
#pragma unroll
              for (int u = 0; u < XU; ++u) {
                const uint32_t g = g0 + u * WAVE + lane;
                oks[u] = g < n_r;
                const uint32_t e = st_r + min(g, n_r - 1);
                mvs[u] = lst[e];
                // without back edges the hash factors load beside the entries
                trm[u] = 0;
                if (!CYCLIC || bo == be) trm[u] = trm_n[e];
              }
              for (uint64_t m = inj; m; m &= m - 1) {
                const uint32_t vc = val[(uint32_t)(__ffsll((long long)m) - 1) * WROWS + i];
#pragma unroll
                for (int u = 0; u < XU; ++u) oks[u] &= mvs[u] != vc;
              }
#pragma unroll
              for (int u = 0; u < XU; ++u)
                if (BYTES && oks[u]) my_bytes += 4;  // the list entry
              if (CYCLIC && bo != be) {
                // with back edges: the tests first, then the factors of the
                // candidates that passed them
                back_edges_of_row<BYTES, XU>(a, P, val, bo, be, dn.w_lo, i, mvs, oks, my_bytes);
#pragma unroll
                for (int u = 0; u < XU; ++u)
                  if (oks[u]) trm[u] = trm_n[st_r + g0 + u * WAVE + lane];
              }
#pragma unroll
              for (int u = 0; u < XU; ++u) {
                const bool ok = oks[u];
                wave_cnt += __popcll(__ballot(ok));
                rsum += ok ? trm[u] : 0ull;
                if (ok) {
                  if (a.emit) {
                    const unsigned long long pos = atomicAdd(a.emit_ctr, 1ULL);
                    if (pos < a.emit_cap) {
                      uint32_t* t = a.emit + pos * q;
                      for (uint32_t c = 0; c <= k; ++c) t[P.order[c]] = a.ids[val[c * WROWS + i]];
                      t[wn] = a.ids[mvs[u]];
                    }
                  }
                }
              }
            }
            my_hash += srow * rsum;
          }
        }
        uint32_t f;
        if constexpr (COUNTED) f = expand(std::false_type{});
        else f = final ? expand(std::true_type{}) : expand(std::false_type{});
        if (final) __syncthreads();  // long_cands complete
        if (!final && tid == 0) S.lrows[nk] += S.fill[nk];
        // advance level k's cursor past what was expanded
        if (tid == 0) {
          // join work: candidates examined (a window cut short by a full
          // buffer is reloaded later from the cursor), and the budget on it
          const unsigned long long done = (unsigned long long)min(f, T) + (final ? S.long_cands : 0u);
          const unsigned long long before = atomicAdd(&a.out[task.query].work, done);
          S.lwork[nk] += done;
          if (a.budget && before + done > a.budget) {
            a.out[task.query].aborted = 1;
            S.abort = 1;
          }
          if (f >= T) {
            S.cur_row[k] = r0 + nw;
            S.cur_cand[k] = 0;
          } else {
            const uint32_t i = seg_search(S.pre, nw, f);
            const uint32_t extra = (i == 0) ? S.cur_cand[k] : 0u;
            S.cur_row[k] = r0 + i;
            S.cur_cand[k] = extra + (f - S.pre[i]);
          }
          if (!final && S.fill[nk] > 0) {
            S.k = nk;
            S.cur_row[nk] = 0;
            S.cur_cand[nk] = 0;
          }
        }
        __syncthreads();
      }
    }

    // flush this task's counters
    if (COUNTED && P.agg) {  // uniform
      flush_agg_work(a, P, S, task.query, aw);
      __syncthreads();
    }
    my_cnt = wave_sum64(my_cnt) + wave_cnt;
    my_hash = wave_sum64(my_hash);
    __syncthreads();
    if (lane_id() == 0) S.red[tid / WAVE] = my_cnt;
    __syncthreads();
    if (tid == 0) {
      unsigned long long c = 0;
      for (uint32_t w = 0; w < blockDim.x / WAVE; ++w) c += S.red[w];
      S.lrows[q - 1] = (q == 2) ? c : S.lrows[q - 1] + c;
      if (c) atomicAdd(&a.out[task.query].count, c);
    }
    __syncthreads();
    if (lane_id() == 0) S.red[tid / WAVE] = my_hash;
    __syncthreads();
    if (tid == 0) {
      unsigned long long h = 0;
      for (uint32_t w = 0; w < blockDim.x / WAVE; ++w) h += S.red[w];
      atomicAdd(&a.out[task.query].hash, h);
    }
    __syncthreads();
    if constexpr (BYTES) {
      my_bytes = wave_sum64(my_bytes);
      if (lane_id() == 0) S.red[tid / WAVE] = my_bytes;
      __syncthreads();
      if (tid == 0) {
        unsigned long long bsum = 0;
        for (uint32_t w = 0; w < blockDim.x / WAVE; ++w) bsum += S.red[w];
        atomicAdd(&a.out[task.query].bytes, bsum);
      }
    }
    if (tid >= 1 && tid < q && S.lrows[tid]) atomicAdd(&a.out[task.query].level_rows[tid], S.lrows[tid]);
    if (tid >= 1 && tid < q && S.lwork[tid]) atomicAdd(&a.out[task.query].level_work[tid], S.lwork[tid]);
    __syncthreads();
  }
}

// Plans counted from records: six waves per SIMD for tree plans (80 VGPRs, 10
// spilled), five for cyclic ones (no spill).
// Tree plans whose embeddings are enumerated: eight waves per SIMD, three
// candidates per thread, 64 VGPRs with 4 spilled.  Enumerating the 1M
// Chung-Lu mix (join per batch, learned order) took 438 ms, against 445 ms
// with four candidates at eight waves (7 spilled), 457 ms with four at seven
// waves (no spill), 452 ms with two at eight and 483-571 ms with six or eight
// candidates at five to seven waves: the waves in flight hide the list loads
// better than more loads per wave.
// Five waves for cyclic plans, whose batched back-edge tests spill heavily
// beyond (R-MAT 22 cycles and cliques 2.05 s per batch at five, 2.07 s at
// six, 2.33 s at eight).
template <bool BYTES>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(6))) join_tree_kernel(JoinArgs a) {
  join_body<BYTES, JOIN_TREE>(a);
}

template <bool BYTES>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(8))) join_tree_enum_kernel(JoinArgs a) {
  join_body<BYTES, JOIN_TREE_ENUM>(a);
}

template <bool BYTES>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(5))) join_cyclic_kernel(JoinArgs a) {
  join_body<BYTES, JOIN_CYCLIC>(a);
}

template <bool BYTES>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(5))) join_cyclic_enum_kernel(JoinArgs a) {
  join_body<BYTES, JOIN_CYCLIC_ENUM>(a);
}

typedef void (*JoinFn)(JoinArgs);

template <bool BYTES>
JoinFn join_fn(JoinKind kind) {
  switch (kind) {
    case JOIN_TREE: return join_tree_kernel<BYTES>;
    case JOIN_TREE_ENUM: return join_tree_enum_kernel<BYTES>;
    case JOIN_CYCLIC: return join_cyclic_kernel<BYTES>;
    default: return join_cyclic_enum_kernel<BYTES>;
  }
}

}  // namespace

uint64_t join_level_words(uint32_t qmax, uint32_t cap) {
  // levels k = 2 .. qmax-2 hold k+1 columns; level k starts at cap*(k(k+1)/2 - 3)
  if (qmax < 4) return 0;
  const uint64_t k = qmax - 1;  // one past the last materialised level
  return (uint64_t)cap * (k * (k + 1) / 2 - 3);
}

namespace {
size_t join_lds_bytes(uint32_t qmax) {
  return ((sizeof(JoinShared) + 15) & ~(size_t)15) + sizeof(uint32_t) * WROWS * qmax;
}
}  // namespace

uint32_t join_resident_per_cu(uint32_t qmax, JoinKind kind) {
  const size_t lds = join_lds_bytes(std::max<uint32_t>(qmax, 2));
  const void* fn = reinterpret_cast<const void*>(join_fn<false>(kind));
  if (lds > 65536) (void)hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  int per_cu = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, (int)WROWS, lds) != hipSuccess || per_cu < 1) {
    (void)hipGetLastError();
    per_cu = 1;
  }
  return (uint32_t)per_cu;
}

void launch_join(const JoinArgs& a, uint32_t nwg, JoinKind kind, hipStream_t s) {
  const size_t lds = join_lds_bytes(a.qmax);
  const JoinFn fn = a.count_bytes ? join_fn<true>(kind) : join_fn<false>(kind);
  if (lds > 65536)
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  hipLaunchKernelGGL(fn, dim3(nwg), dim3(WROWS), lds, s, a);
}

}  // namespace gpsm
