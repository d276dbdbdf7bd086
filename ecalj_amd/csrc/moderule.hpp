// moderule.hpp -- sizes of the Sigma_c mode form (sigmodes.hip): how many
// groups the columns of a k are cut into, how many planes are kept for their
// modes.  Plain C++, checked on the host.
#pragma once
#include <algorithm>
#include <cmath>
#include <cstdint>

namespace ecalj {

constexpr int kModeGroups = 16;
constexpr int kModeSort = 16384;  // columns of one sort (128 KB of LDS)

// Planes kept per k: the mean rank times the groups (C3: 12 groups of 6 modes;
// FP64 at C2: 13 of 11), with room to spare
constexpr int mode_planes(bool f64, int nw1) { return (f64 ? 11 : 6) * nw1; }

// Sorts of a k of T column tiles of BN columns
inline int mode_sorts(int T, int BN) { return (T + kModeSort / BN - 1) / (kModeSort / BN); }

// Column tiles of the groups of one sort of T tiles, of which the k has `sorts`:
// sqrt(f T) equal groups, about the least of rank sum x tiles + the modes' cost.
// bf16x3, f = 1.6: a mode costs about 1.5 tiles at one rank (23 tiles: 6 groups,
// 90 tiles: 12); FP64 / FP32 on 64-column tiles, f = 2.2: about 0.5 (45 tiles: 10
// groups).  No more groups than the planes hold: the ranks of G groups of
// physical weights sum up to 5 G + 16 in the mixed forms, 10.3 G + 22 in FP64
// (and nw1 each), for 8 to 24 frequencies and 500 to 11 000 columns.  A pool that
// overflows means the plain contraction with the modes' overhead on top: at 9
// frequencies and 6150 columns 14 groups of 5.5 did not fit their 54 planes.
inline double mode_rank_sum(bool f64, int G, int nw1) {
  return std::min((double)G * nw1, f64 ? 10.3 * G + 22.0 : 5.0 * G + 16.0);
}
inline int mode_group_tiles(int T, int sorts, bool f64, bool bf3, int nw1) {
  int G = std::max(1, std::min(kModeGroups, (int)(std::sqrt((bf3 ? 1.6 : 2.2) * T) + 0.5)));
  const double room = (double)mode_planes(f64, nw1) / sorts;
  while (G > 1 && mode_rank_sum(f64, G, nw1) > room) --G;
  return (T + G - 1) / G;
}

}  // namespace ecalj
