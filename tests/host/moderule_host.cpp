// C entries to the sizes of the Sigma_c mode form for tests/test_moderule_host.py.
#include "moderule.hpp"

extern "C" {
int moderule_pays(int f64, int bf3, int n, int nk, const int* nm, int step, int ntq, int nw1) {
  return ecalj::mode_pays(f64, bf3, n, nk, nm, step, ntq, nw1);
}
int moderule_planes(int f64, int nw1) { return ecalj::mode_planes(f64, nw1); }
int moderule_sorts(int tiles, int bn) { return ecalj::mode_sorts(tiles, bn); }
int moderule_group_tiles(int tiles, int sorts, int f64, int bf3, int nw1) {
  return ecalj::mode_group_tiles(tiles, sorts, f64, bf3, nw1);
}
}
