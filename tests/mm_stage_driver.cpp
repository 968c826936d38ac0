// reads "rows cols values bytes slab waves row_tiles" a line (a block's values and bytes, the K split, the rows' tiles a workgroup)
// and prints the matrix's bytes, the end of the furthest read of any thread of mm.hip's staged kernel, and that end under an earlier
// rule: the step back taken from the thread's own place, also for threads past the round's words
#include <cstdio>

#include "../libosmos_amd/csrc/mmstage.h"

int main() {
  unsigned rows, cols, values, bytes, slab, waves, row_tiles;
  while (scanf("%u %u %u %u %u %u %u", &rows, &cols, &values, &bytes, &slab, &waves, &row_tiles) == 7) {
    const uint32_t rb = cols / values * bytes, rv = slab * waves, rrb = rv / values * bytes, wb = rb % 4 || rrb % 4 ? 2 : 4;
    const uint32_t threads = waves * 64, words = 16 * row_tiles * rrb / wb, per = (words + threads - 1) / threads, wr = rrb / wb;
    uint64_t end = 0, old_end = 0;
    for (uint32_t row0 = 0; row0 < rows; row0 += 16 * row_tiles)
      for (uint32_t r = 0; r * rv < cols; r++) {
        const uint32_t left = (cols - r * rv) / values * bytes, lim = left;
        for (uint32_t u = 0; u < per; u++)
          for (uint32_t t = 0; t < threads; t++) {
            const uint32_t i = osm::mm::stage_word(u, threads, t, words), row = row0 + i / wr < rows ? row0 + i / wr : rows - 1;
            const uint64_t at = (uint64_t) r * rrb + (uint64_t) row * rb + i % wr * wb;
            const uint64_t e = at - osm::mm::stage_back(i, wr, wb, lim) + wb;
            const uint64_t f = at - osm::mm::stage_back(u * threads + t, wr, wb, lim) + wb;
            if (e > end) end = e;
            if (f > old_end) old_end = f;
          }
      }
    printf("%llu %llu %llu\n", (unsigned long long) rows * rb, (unsigned long long) end, (unsigned long long) old_end);
  }
  return 0;
}
