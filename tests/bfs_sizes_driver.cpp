// One line per "widest first slack expected bytes room" line: whether the
// breadth-first join's buffers fit `room` bytes, the requests made, and what
// the last one lays out.
#include <cstdio>
#include <vector>

#include "bfs_sizes.h"

int main() {
  unsigned widest;
  unsigned long long first, slack, room;
  double expected, bytes;
  while (std::scanf("%u %llu %llu %lf %lf %llu", &widest, &first, &slack, &expected, &bytes, &room) == 6) {
    gpsm::BfsSizes s;
    std::vector<unsigned long long> asked;
    const bool ok = gpsm::bfs_fit(widest, first, slack, gpsm::bfs_rows(widest, first, slack, expected, bytes), s,
                                  [&](size_t n) {
                                    asked.push_back(n);
                                    return n + n / 4 <= room;
                                  });
    std::printf("%d %zu", (int)ok, asked.size());
    for (auto n : asked) std::printf(" %llu", n);
    std::printf(" |");
    for (unsigned l = 1; l + 1 < widest; ++l)
      std::printf(" %llu %llu %llu %u", (unsigned long long)s.at[l], (unsigned long long)s.cap[l],
                  (unsigned long long)s.long_cap[l], gpsm::bfs_row_words(l));
    std::printf("\n");
  }
}
