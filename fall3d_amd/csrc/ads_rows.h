// ads_rows.h -- iterations and row offsets of the streaming sweeps (plain C++).
#pragma once

#include <cstdint>

namespace f3d {

// Iterations of a line of n cells and nst stages: blocks of 16 that end with
// the final update of cell n and start at or before 2 - pf, pf the prefetch
// distance; with half, the first block runs its second half only where that
// still starts there.
struct StreamSpan {
  int first_block, first, last;
};
constexpr StreamSpan stream_span(int n, int nst, int pf, bool half) {
  const int last = n + 2 * nst + 1;
  const int start = last + 1 - 16 * ((last + pf - 1 + 15) / 16);
  return {start, half && start + 8 <= 2 - pf ? start + 8 : start, last};
}

// Byte offset of row r of a line whose rows (r = 0: cell -1) lie pitch bytes
// apart. The first iterations finish rows before the line, up to 25 of them:
// they take row 0, and it is the row that is clamped, since that many pitches
// need not fit 32 bits (a plane of a z line may take 2 GiB / (nz + 4)). The
// offsets are tabulated with the iterations' factors (ads_internal.h).
constexpr uint32_t row_offset(int r, uint32_t pitch) { return r > 0 ? (uint32_t)r * pitch : 0u; }

}  // namespace f3d
