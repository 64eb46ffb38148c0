// Sizes of the breadth-first join's level buffers (kernels/join_bfs.hip), and
// how they shrink where the device has no room for them.
#pragma once
#include <algorithm>
#include <cstdint>

namespace gpsm {

constexpr uint32_t BFS_MAXQ = 8;  // positions of the widest plan joined breadth-first

// Words of a row of `level`: six of its header, level + 1 vertices, even.
constexpr uint32_t bfs_row_words(uint32_t level) { return (6 + level + 1 + 1) & ~1u; }

// The buffers of levels 1 .. widest - 2: short rows of level l at word at[l],
// cap[l] of them, long_cap[l] long ones behind them; words in all.
struct BfsSizes {
  uint64_t at[BFS_MAXQ] = {0}, cap[BFS_MAXQ] = {0}, long_cap[BFS_MAXQ] = {0};
  uint64_t words = 0;
};

// first: rows of level 1, which is written whole, short or long; slack: slots
// of blocks that waves reserve and do not fill; rows: of every later level.
inline BfsSizes bfs_sizes(uint32_t widest, uint64_t first, uint64_t slack, uint64_t rows) {
  BfsSizes s;
  for (uint32_t l = 1; l + 1 < widest; ++l) {
    s.cap[l] = slack + (l == 1 ? first : rows);
    s.long_cap[l] = l == 1 ? first : s.cap[l] / 16;
    s.at[l] = s.words;
    s.words += (s.cap[l] + s.long_cap[l]) * bfs_row_words(l);
  }
  return s;
}

// Rows per level: at most 2^24, and no more than fit `bytes` together with
// level 1 and the quarter that a growing buffer adds; at least BFS_MIN_ROWS (a
// level that does not fit its buffer is joined in several passes).
constexpr uint64_t BFS_MIN_ROWS = 1ull << 18, BFS_MAX_ROWS = 1ull << 24;

inline uint64_t bfs_rows(uint32_t widest, uint64_t first, uint64_t slack, double expected, double bytes) {
  uint64_t rows = (uint64_t)std::min(std::max(16.0 * expected, (double)BFS_MIN_ROWS), (double)BFS_MAX_ROWS);
  while (rows > BFS_MIN_ROWS && 5.0 * bfs_sizes(widest, first, slack, rows).words > bytes) rows /= 2;
  return std::max(rows, BFS_MIN_ROWS);
}

// Asks alloc(bytes) for the buffers, with half the rows each time it has no
// room.  False when not even BFS_MIN_ROWS fit: the plans are joined
// depth-first then, which needs a few hundred KB per workgroup.
template <typename Alloc>
bool bfs_fit(uint32_t widest, uint64_t first, uint64_t slack, uint64_t rows, BfsSizes& s, Alloc alloc) {
  for (;;) {
    s = bfs_sizes(widest, first, slack, rows);
    if (alloc(sizeof(uint32_t) * s.words)) return true;
    if (rows <= BFS_MIN_ROWS) return false;
    rows = std::max(rows / 2, BFS_MIN_ROWS);
  }
}

}  // namespace gpsm
