// Prints, for each "lo hi" line, the number of for_steps' indices, the first
// and the last, and whether they rise by 64; "endless" if they do not end.
#include <cstdio>

#include "kernels/steps.h"

int main() {
  unsigned long long lo, hi;
  while (std::scanf("%llu %llu", &lo, &hi) == 2) {
    unsigned long long n = 0, first = 0, last = 0;
    bool even = true;
    struct Endless {};
    try {
      gpsm::for_steps(lo, hi, [&](uint64_t x) {
        if (n > (hi - lo) / 64 + 1) throw Endless();
        if (!n) first = x;
        even = even && (!n || x == last + 64);
        last = x;
        ++n;
      });
      std::printf("%llu %llu %llu %d\n", n, first, last, (int)even);
    } catch (Endless&) {
      std::printf("endless\n");
    }
  }
}
