// msx_rows.h - the rows of a run of stored positions, for kernels that split
// the matrix by values instead of by rows (a row of any length is then shared
// by as many waves as its values need).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "msx_device.h"

namespace msx {

// The last row r in [0, n_rows) with indptr[r] <= p (0 when there is none),
// the same in every lane: 64 probes a step, so three or four dependent loads
// where a bisection needs about twenty.
template <class I>
__device__ inline int64_t wave_row_of(const I *__restrict__ indptr, int64_t n_rows, int64_t p,
                                      int lane) {
  int64_t lo = 0, hi = n_rows;  // indptr[lo] <= p (or lo == 0), indptr[hi] > p (or hi == n_rows)
  while (hi - lo > 1) {
    const int64_t step = (hi - lo + kWave - 1) / kWave;
    const int64_t at = lo + step * (lane + 1);
    const bool below = at < hi && static_cast<int64_t>(indptr[at < hi ? at : lo]) <= p;
    const int n = __popcll(__ballot(below));
    lo += step * n;
    hi = lo + step < hi ? lo + step : hi;
  }
  return lo;
}

// The row of each lane's position p = b + lane, for the 64 positions from b
// on, and in `row` (in: a row at or before b's; out: lane 63's, where the
// next 64 positions go on).  The row ends that follow are loaded one per lane
// and counted by a bisection over the lanes; only where more than 64 rows end
// inside the 64 positions (runs of empty rows) each lane searches indptr.
// Always in [0, n_rows), whatever indptr holds.
template <class I>
__device__ inline int64_t lane_rows(const I *__restrict__ indptr, int64_t n_rows, int64_t b,
                                    int lane, int64_t &row) {
  const int64_t at = row + 1 + lane;
  const int64_t end = static_cast<int64_t>(indptr[at < n_rows ? at : n_rows]);
  // the row ends before position b + rel; rows past the last one never end
  const int64_t d = end - b;
  const int rel = at >= n_rows || d > kWave ? kWave : (d < 0 ? 0 : static_cast<int>(d));
  int n = 0;  // row ends at or before the lane's position
#pragma unroll
  for (int s = kWave / 2; s >= 1; s >>= 1)
    if (__shfl(rel, n + s - 1, kWave) <= lane) n += s;
  int64_t r = row + n;
  if (__shfl(rel, kWave - 1, kWave) < kWave) {  // wave-uniform: 64 rows end here
    int64_t lo = row, hi = n_rows;
    while (hi - lo > 1) {
      const int64_t mid = lo + (hi - lo) / 2;
      if (static_cast<int64_t>(indptr[mid]) <= b + lane) lo = mid; else hi = mid;
    }
    r = lo;
  }
  if (r > n_rows - 1) r = n_rows - 1;
  row = __shfl(r, kWave - 1, kWave);
  return r;
}

}  // namespace msx
