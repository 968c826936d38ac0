// libosmos MI355X - which word of a round the threads of the f16 matmul's staged kernel (mm.hip) load: plain arithmetic, so that the
// host can check every thread's reads against the matrix.
#pragma once
#include <stdint.h>

#ifdef __HIPCC__
#define OSM_HD __host__ __device__
#else
#define OSM_HD
#endif

namespace osm {
namespace mm {

// a thread's u-th word of a round of `words` (past them: the last again, not stored)
OSM_HD constexpr uint32_t stage_word(uint32_t u, uint32_t threads, uint32_t thread, uint32_t words) {
  return u * threads + thread < words ? u * threads + thread : words - 1;
}
// word i lies at byte i % row_words wb of its row's round. in a round of only `lim` bytes a row, the bytes to step back so that a
// word past them is the last one again
OSM_HD constexpr uint32_t stage_back(uint32_t i, uint32_t row_words, uint32_t wb, uint32_t lim) {
  return i % row_words * wb < lim ? 0 : i % row_words * wb - (lim - wb);
}

}  // namespace mm
}  // namespace osm
