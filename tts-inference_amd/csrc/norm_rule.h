// Which RMSNorm kernel a call takes (w8a16_fused.hip).
#pragma once

#include <stdint.h>

namespace qtts {

// vectors > 0: the row in registers, threads a row, vectors of 8 elements a thread.  vectors == 0, threads > 0: one wave a
// row, read twice in vectors.  threads == 0: one wave a row, element by element.
struct NormForm { int threads, vectors; };

// vec: 16-bit rows, 16-byte aligned, k % 8 == 0.  In registers up to 8192 columns (the fewest threads, 64 to 256, that hold the
// row in one vector each, then up to four vectors a thread) and up to 2^22 rows (one workgroup a row: the grid's
// threads stay within 2^30).
inline NormForm norm_form(bool vec, int64_t m, int64_t k) {
  const int64_t nv = k / 8;
  if (!vec || k <= 0) return {0, 0};
  if (nv > 1024 || m > (1 << 22)) return {64, 0};
  if (nv <= 64) return {64, 1};
  if (nv <= 128) return {128, 1};
  if (nv <= 256) return {256, 1};
  return {256, nv <= 512 ? 2 : 4};
}

}  // namespace qtts
