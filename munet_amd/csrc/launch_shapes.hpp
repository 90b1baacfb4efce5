// Launch shapes and row walks that must hold for every row count that the
// calls admit (just below 2^31, far past what a test can allocate).  Kept free
// of device code, so that the host compiler can run them over those counts
// (tests/cxx/launch_shapes_check.cpp).
#pragma once

#include <algorithm>

namespace mh {

// f(r) for r = first, first + step, ... below rows.  64 bits: a step of 2^23
// past a row count near 2^31 leaves the range of int.
template <class F>
__host__ __device__ __forceinline__ void walk_rows(long first, long step, long rows, F f) {
  for (long r = first; r < rows; r += step) f(r);
}

// f(row0, n) for the launches that cover rows with one workgroup of `threads`
// per row: a launch's work-items must fit in 32 bits.
template <class F> inline void split_rows(long rows, int threads, F f) {
  const long cap = 0xffffffffL / threads;
  for (long r = 0; r < rows; r += cap) f(r, int(std::min(cap, rows - r)));
}

// Row-broadcast kernel: tpr threads per row, rpb rows per 256-thread
// workgroup, gx x gy workgroups for rows of cpr 16-byte chunks; up to 8192
// workgroups, a thread with kRowsInFlight rows in flight.
constexpr int kRowsInFlight = 4;
struct RowBcastShape {
  int tpr, rpb, gx, gy;
};
inline RowBcastShape row_bcast_shape(long rows, int cpr) {
  RowBcastShape s;
  s.tpr = std::min(cpr, 256);
  s.rpb = 256 / s.tpr;
  s.gy = (cpr + s.tpr - 1) / s.tpr;
  const long per = long(kRowsInFlight) * s.rpb;
  s.gx = int(std::max(1L, std::min((rows + per - 1) / per, long(8192 / s.gy))));
  return s;
}

}  // namespace mh
