// runs.h - the maximal runs of plasma cells in one row of the medium, for
// the tiler (which tiles hold plasma, which are plasma through and through).
// Free of HIP so that the host tests compile it alone.
#ifndef FDTD2D_RUNS_H
#define FDTD2D_RUNS_H

#include <algorithm>

namespace fdtd2d {

// Calls emit(first, end) for each maximal run [first, end) of cells i < n
// with positive(i) != 0, in order. Blocks of 64 cells with no change of
// state are passed over after one counting pass (the plasma of a row is one
// or a few long runs).
template <class Positive, class Emit>
inline void scan_runs(int n, Positive positive, Emit emit) {
  constexpr int kBlock = 64;
  int run = -1;  // first column of the open run
  for (int i = 0; i < n; i += kBlock) {
    const int m = std::min(kBlock, n - i);
    int count = 0;
    for (int k = 0; k < m; ++k) count += positive(i + k) != 0;
    if (count == (run >= 0 ? m : 0)) continue;
    for (int k = 0; k < m; ++k) {
      const bool pos = positive(i + k) != 0;
      if (pos && run < 0) {
        run = i + k;
      } else if (!pos && run >= 0) {
        emit(run, i + k);
        run = -1;
      }
    }
  }
  if (run >= 0) emit(run, n);
}

// Whether one of a row's runs r[first] .. r[end - 1], in order as scan_runs
// emits them, covers [c0, c1): the last that starts at or before c0 does, or
// none. (Tiles ask this of every row they load, and a medium of single plasma
// cells has thousands of runs a row: looked through one by one, the tiles of a
// 3800^2 checkerboard took 33 of 73 ms of plan creation.)
template <class Run>
inline bool run_covers(const Run *r, int first, int end, int c0, int c1) {
  int lo = first, hi = end;  // runs before lo start at or before c0, runs from hi on after it
  while (hi - lo > 4) {
    const int mid = lo + (hi - lo) / 2;
    if (r[mid].x <= c0) lo = mid + 1;
    else hi = mid;
  }
  while (lo < hi && r[lo].x <= c0) ++lo;  // (most rows hold one run)
  return lo > first && r[lo - 1].y >= c1;
}

}  // namespace fdtd2d

#endif
