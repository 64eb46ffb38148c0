// Device-side data layout shared by the HIP kernels and their host launchers.
//
// Data graph (resident in HBM for the life of a gpsm_graph):
//   row[n+1], col[A]   undirected CSR, rows ascending
//   key[n]             (dense label << KEY_DEG_BITS) | min(degree, KEY_DEG_MASK):
//                      one 4-byte gather answers "label == L and degree >= d"
//                      for d <= KEY_DEG_MASK as lo <= key <= hi.
// Per batch of queries (one arena, bump-allocated):
//   bitmaps[slot][W]   candidate set C(u) of every query vertex ("slot" =
//                      batch-wide vertex index), W = ceil(n/32) words
//   bprefix[slot][W]   set bits before each word (rank index)
//   clist[coff[slot]]  ascending ids of C(u)
//   per directed query edge x->w used by a join: off[|C(x)|+1] and
//                      list[|CET|], the candidate-edge table
#pragma once
#include <cstdint>

namespace gpsm {

constexpr uint32_t KEY_DEG_BITS = 20;
constexpr uint32_t KEY_DEG_MASK = (1u << KEY_DEG_BITS) - 1;
constexpr uint32_t MAX_LABELS = (1u << (32 - KEY_DEG_BITS)) - 1;
constexpr uint32_t MAXQ = 64;

inline uint32_t words_of(uint32_t n) { return (n + 31) / 32; }

// A data graph's rows in pieces by the neighbours' label (DevGraph::lrow).
struct Pieces {
  const uint32_t* lrow;
  uint32_t n, gshift;
};

enum FilterOpType : uint32_t { OP_EXPLORE = 1, OP_REFINE = 2 };

// One filter operation of one query in a superstep.
struct FilterOp {
  uint32_t type;
  uint32_t u_slot;   // C(u) iterated
  uint32_t nv;       // neighbour entries
  uint32_t nbr_off;  // into nbr_slot / nbr_lo / nbr_hi
  // Refine rounds (match/Match.cu:863-887) after one that removed nothing
  // would remove nothing either: the state is then a fixed point of the
  // round.  mark: flag word set when this op removes a candidate (~0u: none);
  // need: flag word of the query's previous round, which must be set for
  // this op to run (~0u: always runs).
  uint32_t mark;
  uint32_t need;
  // explore: bitmap rows (nv - 1 of them) of the candidates that leave C(u)
  // but hand on matches of v_0, v_1, ...; index of the op's candidate count
  uint32_t e_slot;
  uint32_t cnt;
  // vertex ranges that hold u's label: [range0, range0 + nrange)
  uint32_t range0, nrange;
};

// One neighbour v_i of an explore op: C(v_i) receives the vertices with key in
// [lo, hi] that have a neighbour in C(u) or (e_slot != ~0) in e_slot's row.
struct FillOp {
  uint32_t u_slot, e_slot, v_slot;
  uint32_t lo, hi;
  uint32_t u_lo;              // low key of u's label
  uint32_t range0[2], nrange[2];  // vertex ranges that hold u's label, v's label
  uint32_t cnt;                   // the op's candidate count
  uint32_t nlabel;                // vertices of v_i's label
};

// Initial label/degree check of a query's start vertex.
struct InitOp {
  uint32_t slot;
  uint32_t lo, hi;  // key range
};

// One directed candidate-edge table x -> w.
struct CetDesc {
  uint32_t x_slot, w_slot;
  uint32_t ncand;      // |C(x)|
  uint32_t list_cap;   // words allocated for the list (offsets are clamped to it)
  uint64_t clist_off;  // C(x) ids in clist
  uint64_t off_base;   // offsets [ncand+1] (u32) in the offsets arena
  uint64_t list_base;  // lists in the list arena
  uint64_t total;      // |CET|
  // the last join level's table also gets the hash term of every list entry
  // (tuple_term(term_qid, list[e]) at term_base + e); ~0 for other tables
  uint64_t term_base;
  uint32_t term_qid;
  // a key of w's label (label bits at least 1): the entries walked are the
  // candidates' pieces towards that label
  uint32_t w_lo;
  // records of the last two levels' tables (CetAgg of candidate j at
  // agg_base + j); ~0 for the other tables
  uint64_t agg_base;
};

// What the join's last two levels need of one candidate's list, so that a
// row counts and hashes its embeddings without walking the list.  term_u(v)
// is tuple_term(u, v), L(j) the candidate's list.
//   last level's table (bound vertex w):   s = sum over L(j) of term_w(v)
//   the level before (bound vertex y, list L_y(j)): s the same with term_y and
//     w's parent is y:          a = sum of |L_w(v)|,  b = sum of term_y(v) * s_w(v)
//     w's parent is y's parent: a = |L_y(j) in C(w)|, b = sum of term_y(v) * term_w(v) over them
struct CetAgg {
  unsigned long long s, a, b;
  uint32_t off, len;  // the list inside its table (off: tables with lists only)
};

enum AggMode : uint32_t { AGG_SUM = 0, AGG_SIBLING = 1, AGG_CHAIN = 2 };

// One table of the level before the last: the inputs of its records.
struct AggDesc {
  uint64_t off_base, list_base, agg_base;  // the table's
  uint64_t w_agg_base;                     // the last table's records (AGG_CHAIN)
  uint32_t ncand, mode;
  uint32_t y_slot, y_qid, w_slot, w_qid;
};

// Join plan of one query: vertex order and, per level, how to extend.
struct JoinPlan {
  uint32_t q;
  uint32_t vbase;             // slot of query vertex 0
  uint32_t first_cet;         // CetDesc index of the first table (pi0 -> pi1)
  uint32_t nback_total;
  // levels the join counts from CetAgg records instead of enumerating them:
  // the last agg levels (0, 1 or 2), none of which has a back position
  uint32_t agg;
  uint32_t out;  // index of the query's JoinOut
  // injectivity checks of level k: positions c < k whose query vertex has
  // the label of position k's, other than the parent and the back
  // positions.  A candidate of another label cannot equal the vertex bound
  // there, and one adjacent to the vertex at c cannot equal it (no self-loops).
  uint64_t inj[MAXQ];
  uint32_t order[MAXQ];       // position -> query id
  uint32_t par[MAXQ];         // parent position of level k (k >= 2)
  uint32_t cet[MAXQ];         // CetDesc index used to extend level k (k >= 2)
  uint32_t back_off[MAXQ + 1];  // back positions of level k in backs[]
  uint8_t backs[MAXQ * MAXQ / 2];  // back positions (excluding the parent)
};

// A slice of one query's first table: chunks first, first + stride, ... of
// 2^shift consecutive rows, count rows in all.  A query's tasks interleave
// its chunks, so the rows of hub candidates (the table's first rows on a
// power-law graph) are spread over all of its tasks instead of making the
// first task the longest.  Row r of the task is row task_row(t, r) of the
// table.
struct JoinTask {
  uint32_t query;
  uint32_t stride;
  uint32_t shift, pad;
  uint64_t first, count;
};

// Per-query accumulators written by the join.
struct JoinOut {
  unsigned long long count;
  unsigned long long hash;
  unsigned long long level_rows[MAXQ];
  unsigned long long bytes;  // algorithmic bytes the join read and wrote for this query
  unsigned long long work;   // candidate rows examined (checked against the work budget)
  unsigned long long aborted;
  unsigned long long level_work[MAXQ];  // [1]: first-table rows; [k]: candidates examined for level k
};

}  // namespace gpsm
