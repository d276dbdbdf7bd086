// moderule.hpp -- sizes of the Sigma_c mode form (sigmodes.hip): how many
// groups the columns of a k are cut into, how many planes are kept for their
// modes, and when the form is taken.  Plain C++, checked on the host.
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

// Whether the mode form is taken, for nk k-points of nm[step k] ntq columns:
// where its time, modeled, is below the plain contraction's by 5% (10% in FP64).
// The models (us) are least squares over 447 measured calls of each FP64 and
// FP32 and 534 of bf16x3, of 1.5e10 to 2.5e12 flop (n 60 to 1200, 520 to 19 360
// columns, 1 to 8 k, 8 to 21 frequencies), physical weights; they are within 5 to
// 10% (rms) of the times.  Terms of the modes: launches; the sort (one block per
// sort); the steps of the bases; planes written; W read; the products, by rounds
// of blocks; zmel in sorted order.  Of the plain form: launches; products; W
// unpacked or split; columns.
// Of the calls that the rule takes, 7 of 218, 2 of 302 and 1 of 216 (FP64, FP32,
// bf16x3) were slower than the plain form by more than 3%, at worst 11, 5 and 5%;
// of those it leaves, the modes would have gained at most 40, 25 and 16%.  A rule
// on the flops alone (4e10, 4e10 and 2e11) took 70, 29 and 132 slower ones, at
// worst 42, 21 and 32%: below some 500 tiles a launch of the modes leaves the
// chip part idle, and a few frequencies with many columns give little to save.
// Fewer flops than measured: the plain form.
inline bool mode_pays(bool f64, bool bf3, int n, int64_t nk, const int* nm, int step, int ntq, int nw1) {
  const int BN = bf3 ? 128 : 64, BM = f64 || bf3 ? 128 : 64, BP = bf3 ? 128 : 64;
  double cols = 0, mb = 0, pb = 0, mbk = 0, planes = 0, sorts = 0, rank = 0, sort = 0;
  for (int64_t k = 0; k < (step ? nk : 1); ++k) {
    const double mult = step ? 1.0 : (double)nk;
    const int64_t c = (int64_t)nm[step * k] * ntq;
    if (c == 0) continue;
    if (c > 0x3fffffff) return false;
    const int T = (int)((c + BN - 1) / BN), so = mode_sorts(T, BN), tn = (T + so - 1) / so;
    const int gt = mode_group_tiles(tn, so, f64, bf3, nw1), G = (tn + gt - 1) / gt;
    const double S = mode_rank_sum(f64, G, nw1);
    if (S * so > mode_planes(f64, nw1)) return false;  // the plain contraction in the end
    double M = 128;
    while (M < (double)tn * BN) M *= 2;
    const double b = (double)((n + BM - 1) / BM) * T * mult;
    cols += c * mult;
    mb += b;
    mbk += b * S / G;
    pb += (double)((n + BP - 1) / BP) * T * mult;
    planes += S * so * mult;
    sorts += so * mult;
    rank = std::max(rank, S / G);
    sort = std::max(sort, M * std::log2(M) * std::log2(M) * 1e-6);
  }
  const double flop = 8.0 * n * n * nw1 * cols, nn = 1e-9 * n * n;
  if (cols == 0 || flop < (bf3 ? 8e10 : 1.5e10)) return false;
  sort *= std::max(1.0, sorts / 256);
  const double mr = bf3 ? mb / 256 + 0.5 : 0.3 * std::ceil(mb / 256) + 0.7 * std::max(mb / 256, 0.5);
  const double rest = pb - 512 * std::floor(pb / 512);
  const double pr = bf3 ? 0.5 * std::ceil(pb / 256) + pb / 512
                        : std::floor(pb / 512) + (rest == 0 ? 0 : rest <= 256 ? 0.7 : 1.0);
  const double steps = 0.01 * nw1 * rank, w = (double)nk * nw1 * nn, mg = 1e-3 * n * mr * mbk / mb, pg = 1e-3 * n * pr * nw1;
  const double io = 1e-9 * n * cols;
  if (f64) return 410 + 330 * pg + 9300 * w + 43000 * io > 1.1 * (400 + 190 * sort + 150 * steps + 6400 * planes * nn + 9500 * w + 250 * mg);
  if (!bf3) return 510 + 170 * pg + 12000 * w > 1.05 * (360 + 110 * sort + 250 * steps + 6100 * planes * nn + 940 * w + 78 * mg);
  return 32 + 62 * pg + 4100 * w + 12000 * io > 1.05 * (73 * sort + 130 * steps + 570 * planes * nn + 6100 * w + 56 * mg + 16000 * io);
}

}  // namespace ecalj
