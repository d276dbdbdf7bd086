// gemm64.hip -- batched FP64 complex GEMM on the tile of gemm64.hpp: the
// large products of the FP64 engine (Gauss-Jordan trailing updates, M <-> E
// transforms, zmel).
#include "gemm64.hpp"

namespace ecalj {

template <bool AT, bool BT>
__global__ __launch_bounds__(D6T, 4) void zgemm64_kernel(GemmArgs g) {
  __shared__ D6Smem s;
  int b, mt, nt;
  if (g.xt == 0) {
    b = blockIdx.z;
    mt = blockIdx.x;
    nt = blockIdx.y;
  } else {
    const int p = blockIdx.x, j = p >> 3, t = j % g.xt;
    b = (j / g.xt) * 8 + (p & 7);
    if (b >= g.batch) return;
    mt = t % g.xg;
    nt = t / g.xg;
  }
  const int m0 = mt * D6M, n0 = nt * D6N;
  if (g.epi == EPI_GJ && m0 >= g.gj_k0 && min(m0 + D6M, g.M) <= g.gj_k1) return;  // rows that are not updated
  const cd* A = static_cast<const cd*>(g.A) + g.bA.off(b, g.div);
  const cd* B = static_cast<const cd*>(g.B) + g.bB.off(b, g.div);
  cd* C = static_cast<cd*>(g.C) + g.bC.off(b, g.div);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  typedef D6Ld<D6M, AT> LA;
  typedef D6Ld<D6N, !BT> LB;
  LA la;
  LB lb;
  la.init(A, g.lda, m0, g.M, wave, lane);
  lb.init(B, g.ldb, n0, g.N, wave, lane);
  constexpr int PER = LA::NI + LB::NI;
  const int nst = (g.K + D6K - 1) / D6K;
  auto issue = [&](int st, int buf) {
    la.issue(s.a[buf], wave, st * D6K, g.K);
    lb.issue(s.b[buf], wave, st * D6K, g.K);
  };
  D6Acc c;
  c.zero();
  const double w[2] = {1.0, 1.0};
  // every step issues one stage (past the last one again the last, into a free
  // buffer), so one wait count covers the current stage throughout
  issue(0, 0);
  issue(min(1, nst - 1), 1);
  const int nfull = g.K / D6K;
  int buf = 0;
  for (int st = 0; st < nfull; ++st) {
    d6_wait<PER>();
    const int nb = buf == 0 ? 2 : buf - 1;  // (st + 2) % 3
    issue(min(st + 2, nst - 1), nb);
    d6_stage<LA, LB, false, false>(c, s.a[buf], s.b[buf], wm, wn, lane, g.csA, g.csB, w, D6K);
    buf = buf == 2 ? 0 : buf + 1;
  }
  if (nfull < nst) {
    d6_wait<0>();
    d6_stage<LA, LB, true, false>(c, s.a[buf], s.b[buf], wm, wn, lane, g.csA, g.csB, w, g.K - nfull * D6K);
  }
  ECALJ_WAIT_VMCNT(0);  // the repeated stages have landed before the block's LDS is released
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        __builtin_amdgcn_sched_barrier(0);
        gemm_store(g, C, m0 + wm * 32 + i * 16 + acc_row_f64(lane, e), n0 + wn * 32 + j * 16 + (lane & 15),
                   c.cr[i][j][e], c.ci[i][j][e]);
      }
}

// Whether a product goes to this kernel: enough rows and columns to fill its
// tile, enough k to fill the ring, 16-byte aligned operands (the loads move
// whole elements), and a block for every CU (below that the 64 x 64 tile
// spreads over twice the blocks).
bool gemm64_pays(const ecalj_ctx* h, const GemmArgs& g) {
  const int64_t blocks = (int64_t)((g.M + D6M - 1) / D6M) * ((g.N + D6N - 1) / D6N) * g.batch;
  return g.M > 64 && g.N > 32 && g.K >= 3 * D6K && blocks >= h->ncu && ((uintptr_t)g.A | (uintptr_t)g.B) % 16 == 0;
}

ecalj_status gemm64(ecalj_ctx* h, const GemmArgs& g0, bool at, bool bt) {
  GemmArgs g = g0;
  dim3 grid((g.M + D6M - 1) / D6M, (g.N + D6N - 1) / D6N, g.batch);
  g.xg = g.xt = 0;
  if (g.batch >= 8 && (g.batch % 8 == 0 || g.batch >= 128)) {  // XCD order, as in launch_gemm
    const int64_t xt = (int64_t)grid.x * grid.y, p = 8 * xt * ((g.batch + 7) / 8);
    if (p <= 0x7fffffff) {
      g.xg = (int)grid.x;
      g.xt = (int)xt;
      grid = dim3((unsigned)p, 1, 1);
    }
  }
  if (grid.y > 65535 || grid.z > 65535) return ECALJ_ERR_DIM;
  auto go = [&](auto kern) { hipLaunchKernelGGL(kern, grid, dim3(D6T), 0, h->stream, g); };
  if (at) {
    if (bt) go(zgemm64_kernel<true, true>);
    else go(zgemm64_kernel<true, false>);
  } else {
    if (bt) go(zgemm64_kernel<false, true>);
    else go(zgemm64_kernel<false, false>);
  }
  ECALJ_HIP(hipGetLastError());
  return ECALJ_OK;
}

}  // namespace ecalj
