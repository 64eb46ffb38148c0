// Host launchers of the device kernels (one translation unit per phase).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <vector>

#include "bfs_sizes.h"
#include "gpsm_dev.h"

namespace gpsm {

struct DevGraph {
  uint32_t n = 0;
  uint64_t adj = 0;
  uint32_t W = 0;   // bitmap words per query vertex
  // The vertices are numbered by (label, id) on the device, so that a
  // candidate set, all of one label, is one dense piece of every bitmap and of
  // every hub's: ids[i] is the id of vertex i, pos its inverse.  row / col and
  // everything below are in this numbering; what leaves the device (hashes,
  // tuples, lists, bitmaps) is in ids.  row0 / col0: the CSR in ids (the same
  // arrays where the numbering is the ids' own).
  uint32_t* row0 = nullptr;
  uint32_t* col0 = nullptr;
  uint32_t* ids = nullptr;
  uint32_t* pos = nullptr;
  // The adjacency in pieces by the neighbours' label, the pieces of one label
  // side by side: the entries of vertex v whose neighbours have a label of
  // group g (1 << gshift consecutive dense labels) are col[lrow[g * n + v]] ..
  // col[lrow[g * n + v + 1] - 1], ascending.  A step that looks for one label
  // among the neighbours of a candidate set (vertices of one label) streams
  // what it needs and nothing else.  One group: lrow is row.  row: degrees
  // (row[v + 1] - row[v]).
  uint32_t* row = nullptr;
  uint32_t* col = nullptr;
  uint32_t* lrow = nullptr;
  uint32_t ngroup = 1, gshift = 0;
  uint32_t* key = nullptr;
  // ckey[e] = key[col[e]]: the filter's label/degree tests stream the keys
  // of a row's neighbours beside the row instead of gathering them
  uint32_t* ckey = nullptr;
  // filter work items: vertex ranges [fchunk[i], fchunk[i+1]) of at most
  // FCHUNK_VERTS vertices and FCHUNK_ENTRIES adjacency entries (a vertex
  // with more entries is a range of its own), so that no wave of the filter
  // walks far more adjacency than the others (power-law hubs)
  uint32_t* fchunk = nullptr;
  uint32_t nfchunk = 0;
  // the vertices with more than FCHUNK_ENTRIES entries in parts of HUB_PART:
  // (vertex, part) pairs
  uint2* hparts = nullptr;
  uint32_t nhparts = 0;
  // wrange[w]: the vertex range holding vertex 32w (one per bitmap word)
  uint32_t* wrange = nullptr;
  // hubs (degree above hub_degree): hub_of[v] = index of v's adjacency
  // bitmap (W words each, in hub_bits) or ~0u, so an edge test touching a
  // hub is one bit; other edge tests search the shorter adjacency list
  uint32_t* hub_of = nullptr;
  uint32_t* hub_bits = nullptr;
  uint32_t nhub = 0;
  uint32_t hub_degree = 0;
};

inline Pieces pieces_of(const DevGraph& g) { return Pieces{g.lrow, g.n, g.gshift}; }

// Vertices per range: fewer where the graph is small, whose candidate sets
// (one label's vertices, next to each other) otherwise fill too few waves.
// 64 against 256 vertices a range on Chung-Lu graphs of 8 n edges and 4 labels,
// an 8-vertex walk by itself (filter and counts) and 64 walks of 6 to 8 in a
// batch: n = 30k 393 / 490 us and 3.1 / 3.1 ms, 200k 608 / 708 us and 8.6 / 7.7
// ms, 400k 820 / 855 us and 15.2 / 13.6 ms, 600k 1165 / 1127 us and 21.2 / 18.4
// ms, 1M 1570 / 1430 us and 39.7 / 34.6 ms.  With 16 labels the single walk is
// even at 1M (682 / 672 us), a batch at 100k (2.75 / 2.65 ms).  The line is
// where single queries of few labels are even.
constexpr uint32_t FCHUNK_VERTS = 256, FCHUNK_VERTS_SMALL = 64;
inline uint32_t range_verts(uint32_t n) { return n < 1u << 19 ? FCHUNK_VERTS_SMALL : FCHUNK_VERTS; }
constexpr uint32_t FCHUNK_ENTRIES = 4096;
constexpr uint32_t HUB_PART = 2048;

// graph.hip: what a resident graph holds besides its CSR, built from it.
constexpr uint32_t LABEL_HIST = 4096, HUB_STEPS = 34;
// hist (LABEL_HIST + 1 words) and hubs (HUB_STEPS), zeroed by the caller: the
// labels' counts and the vertices by how often min_degree doubles below their
// degree (vertex_stats_kernel).
void launch_vertex_stats(const uint32_t* row, const uint32_t* label, uint32_t n, uint32_t min_degree, uint32_t* hist,
                         uint32_t* hubs, hipStream_t s);
// Sets *bad (zeroed by the caller) if a row of the CSR (offsets monotone, the
// last one the length of col) is not strictly ascending, holds its own vertex
// or one >= n.
void launch_check_rows(const uint32_t* row, const uint32_t* col, uint32_t n, uint64_t adj, uint32_t* bad,
                       hipStream_t s);
// From row0 / col0, the vertices' labels (by id) and the nl distinct label
// values, ascending: ids, pos, row, col and lrow (unless they are row0 / col0:
// the vertices then keep their ids) and key.  scratch: relabel_words(n, adj)
// words, 8-byte aligned; relabel_words(n, 0) where the ids are kept.
uint64_t relabel_words(uint32_t n, uint64_t adj);
void launch_relabel(const DevGraph& g, const uint32_t* label, const uint32_t* value, uint32_t nl, uint32_t* scratch,
                    hipStream_t s);
// The groups of g.lrow for nl labels: at most PIECE_GROUPS, a table of at most
// four words per adjacency entry, and entries that sort as 64-bit keys.
constexpr uint32_t PIECE_GROUPS = 64;
void choose_pieces(DevGraph& g, uint32_t nl);
// range[2 l], range[2 l + 1]: the first vertex range with a vertex of label l
// and the one after the last; start[l]: vertices of the labels before l (nl + 1
// words, device).
void launch_label_ranges(const DevGraph& g, const uint32_t* start, uint32_t nl, uint32_t* range, hipStream_t s);
// Bitmap rows of vertices to bitmap rows of ids.
void launch_id_bitmaps(const DevGraph& g, const uint32_t* bitmaps, uint32_t nrows, uint32_t* out, hipStream_t s);
// Vertices to ids in place.
void launch_to_ids(const DevGraph& g, uint32_t* v, uint64_t n, hipStream_t s);
// The filter's vertex ranges: their ends and their number (*total), then, with
// g.fchunk and g.wrange allocated, those.  scratch: range_words(n) words.
// *parts (zeroed by the caller): the parts of all vertices with more than
// FCHUNK_ENTRIES entries; launch_ranges also writes g.hparts (in any order,
// *next zeroed by the caller).
uint64_t range_words(uint32_t n);
void launch_range_ends(const uint32_t* row, uint32_t n, uint32_t* scratch, unsigned long long* total, uint32_t* parts,
                       hipStream_t s);
void launch_ranges(const DevGraph& g, const uint32_t* scratch, uint32_t* next, hipStream_t s);
// g.hub_of and, with nhub of them above hub_degree and hub_bits zeroed, their
// bitmaps.  scratch: hub_words(n) words, 8-byte aligned.
uint64_t hub_words(uint32_t n);
void launch_hubs(const DevGraph& g, uint32_t* scratch, hipStream_t s);

// build.hip: the undirected CSR of an edge list (host arrays src/dst of m
// edges, either orientation; duplicates and self-loops dropped), built on
// the device.  *row (n+1) and *col (*adj) are taken from pool, as is what the
// build itself needs.  GPSM_EINVAL if an endpoint is >= n.
class BlockPool;
class Stager;
int build_csr_from_edges(uint32_t n, uint64_t m, const uint32_t* src, const uint32_t* dst, BlockPool& pool,
                         Stager& stager, hipStream_t s, uint32_t** row, uint32_t** col, uint64_t* adj);

void launch_neighbour_keys(const DevGraph& g, hipStream_t s);

// filter.hip ------------------------------------------------------------------
// Start-vertex candidates: C(slot) = {v : lo <= key[v] <= hi} (check_kernel).
void launch_init(const DevGraph& g, const InitOp* ops, uint32_t nops, uint32_t* bitmaps, hipStream_t s);
// One superstep: every op (one per query) explores or refines its C(u); the
// explore ops' neighbours are filled by a second launch (fills, one per
// neighbour).  stats (optional, STAT_COPIES x STAT_STRIDE u64, zeroed by the
// caller): copy c, entries 0..4 = pieces looked up (one per candidate and
// neighbour), adjacency entries read, vertex and second entry keys read, bitmap
// probes, bits set, added by the workgroups with blockIdx %
// copies == c (the sum over copies is the launch's total).
// Of more than FILTER_DIRECT (op, vertex range) pairs the superstep visits
// only those whose range holds a candidate of C(u): a first kernel lists them
// in items (nops x max_ranges capacity) and counts them in *nitems (zeroed by
// the caller), the second processes the list.  Fewer are all visited by one
// launch, whose waves leave an empty range after reading its bitmap words:
// listing the pairs of one op on a 1M-vertex graph took 35 us (four
// workgroups), more than the pass over its 5,000 ranges.
// max_ranges: the most ranges any of the ops' or fills' labels has.
// resident: filter_resident(block).  rflags: the refine rounds' change flags
// (FilterOp::mark / need), zeroed by the caller once per batch; an op whose
// need flag is clear is left out.  counts: the explore ops' candidates
// (FilterOp::cnt), zeroed by the caller.
constexpr uint32_t STAT_COPIES = 32, STAT_STRIDE = 8;
constexpr uint32_t FILTER_OVERSUB = 8;
constexpr uint64_t FILTER_DIRECT = 1u << 17;
// A fill is pulled when FILL_PULL times the op's candidates are at least the
// vertices of the neighbour's label.  With 8 / 32 / 256 / 1024 here and all
// pulled: 245 queries on the 1M Chung-Lu graph 22.3 / 19.6 / 19.0 / 19.0 / 19.0
// ms, a 14-vertex filter on it 1.38 / 1.28 / 1.11 / 1.13 / 1.14 ms, the filter
// and tables of an 8-vertex query on a 100k graph 1.19 / 1.14 / 1.18 / 1.19 /
// 1.18 ms (run to run +-0.03).
constexpr uint32_t FILL_PULL = 256;
void launch_filter_step(const DevGraph& g, const FilterOp* ops, uint32_t nops, const uint32_t* nbr_slot,
                        const uint32_t* nbr_lo, const uint32_t* nbr_hi, const FillOp* fills, uint32_t nfill,
                        uint32_t* bitmaps, uint32_t max_ranges, uint32_t block, uint32_t resident, uint2* items,
                        uint32_t* nitems, uint32_t* rflags, uint32_t* counts, unsigned long long* stats,
                        hipStream_t s);
// Workgroups of `block` threads of the superstep's kernel that are resident at once.
uint32_t filter_resident(uint32_t block);

// scan.hip ---------------------------------------------------------------------
// Bitmap rows are compacted in segments of SEG_WORDS words, one workgroup
// per (row, segment).
constexpr uint32_t SEG_WORDS = 2048;
inline uint32_t segs_of(uint32_t W) { return (W + SEG_WORDS - 1) / SEG_WORDS; }
// segc[r * segs_of(W) + i] = set bits of bitmap row r before segment i
// (exclusive prefix of the segments' popcounts); counts[r] = popcount of row r.
void launch_row_popcount(const DevGraph& g, const uint32_t* bitmaps, uint32_t nrows, uint32_t* segc,
                         uint32_t* counts, hipStream_t s);
// Compaction of bitmap rows to ascending id lists (row r at clist + coff[r])
// plus the rank index, from the segment counts of launch_row_popcount.
void launch_compact_rows(const DevGraph& g, const uint32_t* bitmaps, uint32_t nrows, const uint32_t* segc,
                         const uint64_t* coff, uint32_t* clist, uint32_t* bprefix, hipStream_t s);
void launch_fill_u32(uint32_t* p, uint32_t v, uint64_t n, hipStream_t s);
// Exclusive scan of n u32 values; out may alias in.  total (device, u64) optional.
void launch_exclusive_scan(const uint32_t* in, uint32_t* out, uint64_t n, unsigned long long* total,
                           uint32_t* scratch, uint64_t scratch_words, hipStream_t s);
uint64_t scan_scratch_words(uint64_t n);
// Ascending ids of set bits of one bitmap; count written to *count (device
// u64).  scratch: compact_scratch_words(nbits) words, 8-byte aligned.
uint64_t compact_scratch_words(uint64_t nbits);
void launch_compact_bitmap(const uint32_t* bits, uint64_t nbits, uint32_t* ids, unsigned long long* count,
                           uint32_t* scratch, hipStream_t s);

// radix.hip --------------------------------------------------------------------
// One stable pass over the 8 bits of the keys at shift: in to out, with values
// vin to vout unless null.  hist, hstart: radix_hist_words(n) words each;
// scratch: scan_scratch_words of that many.  n < 2^32.
uint64_t radix_hist_words(uint64_t n);
void launch_radix_pass(const unsigned long long* in, unsigned long long* out, const uint32_t* vin, uint32_t* vout,
                       uint64_t n, uint32_t shift, uint32_t* hist, uint32_t* hstart, uint32_t* scratch,
                       uint64_t scratch_words, hipStream_t s);

// tuples.hip -------------------------------------------------------------------
// Lexicographic order of rows of q u32 values below 2^bits, all distinct.
// Up to cap <= TUPLE_RANK rows: one launch, the number of rows read from
// *count on the device (more than cap: nothing is written); out may be host
// memory the device can write.
constexpr uint32_t TUPLE_RANK = 8192;
void launch_rank_tuples(const uint32_t* tuples, uint32_t q, uint32_t bits, const unsigned long long* count,
                        uint32_t cap, uint32_t* out, hipStream_t s);
// Any number below 2^32: radix passes over the rows' packed bits, the rows
// themselves moved once.  scratch: tuple_sort_words(n) words, 8-byte aligned.
uint64_t tuple_sort_words(uint64_t n);
void launch_sort_tuples(const uint32_t* tuples, uint64_t n, uint32_t q, uint32_t bits, uint32_t* scratch,
                        uint32_t* out, hipStream_t s);

// text.hip ---------------------------------------------------------------------
// Embedding lines "(j, k) ... \n" of IO::output.  R = text_rows_per_wg(q)
// rows per workgroup; wg_len / wg_off: ceil(rows / R) words.
constexpr uint32_t TEXT_STAGE_BYTES = 61440;
uint32_t text_fixed_length(uint32_t q);
uint32_t text_rows_per_wg(uint32_t q);
void launch_text_len(const uint32_t* tuples, uint64_t rows, uint32_t q, const uint8_t* keep, uint32_t* wg_len,
                     hipStream_t s);
void launch_text_write(const uint32_t* tuples, uint64_t rows, uint32_t q, const uint8_t* keep,
                       const uint32_t* wg_off, char* out, hipStream_t s);

// cet.hip ----------------------------------------------------------------------
// Per CetDesc: |CET| into desc.total (atomic); per-candidate counts into
// offsets at desc.off_base.
// chunk_base[d]: chunks of 64 candidates in the tables before d (ndesc + 1
// entries); grid: workgroups (persistent).
// stats (optional, STAT_COPIES x STAT_STRIDE u64, zeroed by the caller):
// entries 0..3 = candidates (cet_count, cet_write), adjacency entries examined,
// bitmap probes, list entries written, 4 = cet_sum's candidates, 5..7 = cet_agg's
// candidates, list entries and records read, summed over the copies.
void launch_cet_count(const DevGraph& g, const uint32_t* bitmaps, const uint32_t* clist, CetDesc* descs,
                      uint32_t ndesc, uint32_t* offsets, const uint32_t* chunk_base, uint32_t grid, hipStream_t s,
                      unsigned long long* stats = nullptr);
// Segmented exclusive scan of the per-candidate counts of every desc.
void launch_cet_offsets(CetDesc* descs, uint32_t ndesc, uint32_t* offsets, hipStream_t s);
// Records of the last join levels' tables (CetAgg::s and len of every
// candidate): one pass over the adjacency, no lists written.
void launch_cet_sums(const DevGraph& g, const uint32_t* bitmaps, const uint32_t* clist, const CetDesc* descs,
                     uint32_t ndesc, const uint32_t* chunk_base, CetAgg* aggs, uint32_t grid, hipStream_t s,
                     unsigned long long* stats = nullptr);
// Records of the tables of the level before the last, from their lists and
// the last tables' records.
void launch_cet_aggs(const DevGraph& g, const uint32_t* bitmaps, const uint32_t* bprefix, const AggDesc* descs,
                     uint32_t ndesc, const uint32_t* chunk_base, const uint32_t* offsets, const uint32_t* lists,
                     CetAgg* aggs, uint32_t grid, hipStream_t s, unsigned long long* stats = nullptr);
// Hash terms of the last join levels' lists: for table term_desc[i] (terms
// [term_start[i], term_start[i+1]) of terms), tuple_term(term_qid, id of list[e]).
void launch_cet_terms(const DevGraph& g, const uint32_t* lists, const CetDesc* descs, const uint32_t* term_desc,
                      const uint64_t* term_start, uint32_t nterm_desc, uint64_t nterms, unsigned long long* terms,
                      hipStream_t s);
// Writes the lists.
void launch_cet_write(const DevGraph& g, const uint32_t* bitmaps, const uint32_t* clist, const CetDesc* descs,
                      uint32_t ndesc, const uint32_t* offsets, uint32_t* lists, const uint32_t* chunk_base, uint32_t grid,
                      hipStream_t s, unsigned long long* stats = nullptr);

// join.hip ---------------------------------------------------------------------
struct JoinArgs {
  const uint32_t* col;
  const uint32_t* ids;       // DevGraph::ids
  Pieces pieces;
  const uint32_t* hub_of;    // DevGraph::hub_of / hub_bits
  const uint32_t* hub_bits;
  const uint32_t* bitmaps;
  const uint32_t* bprefix;
  const uint32_t* clist;
  const uint32_t* offsets;
  const uint32_t* lists;
  const unsigned long long* terms;  // hash terms of the last level's lists (CetDesc::term_base)
  const CetAgg* aggs;  // records of the last two levels' tables (CetDesc::agg_base)
  const CetDesc* cets;
  const JoinPlan* plans;
  const JoinTask* tasks;
  uint32_t ntasks;
  uint32_t W;
  uint32_t cap;       // rows per level buffer
  uint32_t qmax;      // widest query of the batch
  uint32_t* levels;   // per workgroup: (qmax-2) buffers of cap rows, column-major
  uint64_t level_stride;  // words per workgroup
  unsigned int* task_counter;
  JoinOut* out;
  // optional tuple output (query-id order), emit_cap tuples of q words
  uint32_t* emit;
  unsigned long long* emit_ctr;
  uint64_t emit_cap;
  // 0 or the candidate rows a query may examine before it is abandoned
  unsigned long long budget;
  // nonzero: account algorithmic bytes in JoinOut::bytes (a slower variant)
  uint32_t count_bytes;
};
// Kernel of a join launch: tree plans (no back edges) whose last levels are
// counted from records, tree plans whose embeddings are enumerated (tuples
// wanted), plans with back edges whose last levels are counted from records,
// plans with back edges at the last position (or tuples wanted).
enum JoinKind { JOIN_TREE = 0, JOIN_TREE_ENUM = 1, JOIN_CYCLIC = 2, JOIN_CYCLIC_ENUM = 3 };
// One persistent join launch over tasks [0, ntasks) of a.tasks, all of them
// of plans of that kind.
void launch_join(const JoinArgs& a, uint32_t nwg, JoinKind kind, hipStream_t s);
uint64_t join_level_words(uint32_t qmax, uint32_t cap);

// join_bfs.hip -------------------------------------------------------------------
// Breadth-first join of up to BFS_PLANS plans with back edges and at most
// BFS_MAXQ positions: launch_bfs_first writes the level-1 rows, launch_bfs_expand
// takes level to level + 1: all its rows, or (resume) those that an earlier
// launch left when the next level's buffer was full.  j: plans (nplans of them, JoinPlan::out their
// results), cets, lists, budget and out as for launch_join.
constexpr uint32_t BFS_PLANS = 256;
struct BfsCursor {
  uint32_t idx, pos, skip;
  uint32_t rows;  // a quad's rows with candidates in the step that skip counts in, a bit each
};
struct BfsArgs {
  JoinArgs j;
  uint32_t nplans, level;
  uint32_t block;             // row slots a wave reserves at a time
  uint32_t any_source;        // a row's candidates may come from any of its bound neighbours (finish_rows)
  const uint64_t* first_row;  // first-table rows of the plans before each (nplans + 1)
  // rows of `level` and `level + 1`: records of stride_* words; short lists,
  // long lists, and their counts (2 words each, zeroed by the caller)
  const uint32_t *rows_in, *long_in;
  uint32_t cap_in, long_cap_in, stride_in;
  const uint32_t* cin;
  uint32_t *rows_out, *long_out;  // null at the last level
  uint32_t cap, long_cap, stride_out;
  uint32_t* cout;
  BfsCursor* cursors;  // two per wave of the level's launches (the same grid each time)
  uint32_t resume;
  uint32_t* pending;   // waves that stopped at a full buffer (zeroed by the caller)
};
void launch_bfs_first(const BfsArgs& a, uint32_t nwg, hipStream_t s);
void launch_bfs_expand(const BfsArgs& a, uint32_t nwg, hipStream_t s);
uint32_t bfs_resident_per_cu(uint32_t nplans);
// Join workgroups (of the timed variant of the kind's kernel) that are
// resident on one CU at once for a batch whose widest query has qmax
// vertices (LDS and registers); a persistent grid gains nothing from more.
uint32_t join_resident_per_cu(uint32_t qmax, JoinKind kind);

}  // namespace gpsm
