// gemm64.hpp -- FP64 complex block tile for large products: 128 x 64 outputs,
// 8 waves (4 x 2, 32 x 32 each), complex128 operands moved global -> LDS
// directly (no registers, no address arithmetic per element), three stages of
// 8 k in a ring, two of them in flight, one barrier per stage.
//
// What bounded the 64 x 64 tile of gemm.hpp (C2 Sigma_c: matrix cores busy 62%
// of the time): every stage passed through registers, with two barriers
// around its LDS writes (split into re and im planes, a third of the LDS
// cycles in bank conflicts) and index arithmetic per element.  Here 72 KB of
// LDS leave two blocks on a CU, four waves on a SIMD.
//
// LDS layout: complex elements (16 bytes: one read gives re and im).
//   x contiguous in memory: [k][x], 64 consecutive x per load instruction;
//   k contiguous: [x][slot], slot = k ^ (x & 7): 8 rows per load instruction,
//   and the 8 lanes of one LDS pass read 8 different slots.
// Rows / columns beyond the operand are clamped to its last one (their
// outputs are not stored), k beyond K is clamped and masked when read.
#pragma once
#include "sigtile.hpp"

namespace ecalj {

constexpr int D6M = 128, D6N = 64, D6K = 8, D6R = 3, D6T = 512;

typedef double d2 __attribute__((ext_vector_type(2)));

struct alignas(16) D6Smem {
  d2 a[D6R][D6K * D6M];  // 16 KB per stage
  d2 b[D6R][D6K * D6N];  // 8 KB per stage
};

// Load addresses of one lane: NI instructions of 1 KB per wave and stage.
template <int BX, bool KC>
struct D6Ld {
  static constexpr int NI = BX * D6K / (D6T / 64) / 64;
  const cd* p[NI];   // KC: the lane's row at k = 0; else the lane's x at k = 0
  int64_t ld;        // !KC: element step per k
  int kk[NI];        // k within the stage
  __device__ void init(const cd* base, int64_t ld_, int x0, int X, int wave, int lane) {
    ld = ld_;
#pragma unroll
    for (int q = 0; q < NI; ++q) {
      const int r = wave * NI + q;  // run of 64 elements in the stage
      if (KC) {
        const int x = r * 8 + (lane >> 3);
        p[q] = base + ld * min(x0 + x, X - 1);
        kk[q] = (lane & 7) ^ (x & 7);
      } else {
        constexpr int XR = BX / 64;
        p[q] = base + min(x0 + (r % XR) * 64 + lane, X - 1);
        kk[q] = r / XR;
      }
    }
  }
  // stage at k0 of K (k clamped): element (x, k) of the operand
  __device__ void issue(d2* dst, int wave, int k0, int K) const {
#pragma unroll
    for (int q = 0; q < NI; ++q) {
      const int k = min(k0 + kk[q], K - 1);
      const cd* s = p[q] + (KC ? (int64_t)k : ld * k);
      __builtin_amdgcn_global_load_lds((gbl_ptr_t)s, (lds_ptr_t)(dst + (wave * NI + q) * 64), 16, 0, 0);
    }
  }
  __device__ static int slot(int x, int k) { return KC ? x * D6K + (k ^ (x & 7)) : k * BX + x; }
};

// Accumulators of one wave: 2 x 2 tiles of 16 x 16.
struct D6Acc {
  d4 cr[2][2], ci[2][2];
  __device__ void zero() {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) cr[i][j] = ci[i][j] = d4{0, 0, 0, 0};
  }
};

// One stage: C += (conj when CA)(A) (conj when CB)(B); w: real factor of the
// lane's two columns; klim < D6K masks the tail.
template <class LA, class LB, bool TAIL, bool WT>
__device__ __forceinline__ void d6_stage(D6Acc& c, const d2* a, const d2* b, int wm, int wn, int lane, double csA,
                                         double csB, const double (&w)[2], int klim) {
  const int l = lane & 15, g = lane >> 4;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    __builtin_amdgcn_sched_barrier(0);  // one half's fragments at a time: 128 registers hold four waves per SIMD
    d2 fa[2], fb[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      fa[i] = a[LA::slot(wm * 32 + i * 16 + l, 4 * h + g)];
      fb[i] = b[LB::slot(wn * 32 + i * 16 + l, 4 * h + g)];
    }
    if (TAIL && 4 * h + g >= klim) {
#pragma unroll
      for (int i = 0; i < 2; ++i) fa[i] = fb[i] = d2{0, 0};
    }
    double an[2], ai[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      ai[i] = csA * fa[i][1];
      an[i] = -ai[i];
      if (WT) {
        fb[i][0] *= w[i];
        fb[i][1] *= w[i];
      } else {
        fb[i][1] *= csB;
      }
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
        c.cr[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(fa[i][0], fb[j][0], c.cr[i][j], 0, 0, 0);
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
        c.ci[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(fa[i][0], fb[j][1], c.ci[i][j], 0, 0, 0);
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
        c.cr[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(an[i], fb[j][1], c.cr[i][j], 0, 0, 0);
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
        c.ci[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(ai[i], fb[j][0], c.ci[i][j], 0, 0, 0);
  }
}

// The stage wait and barrier: every load but the `left` newest has landed in
// every wave, and every wave has left the stage before: its LDS reads have
// returned (lgkmcnt 0) before the barrier, after which that stage's buffer is
// loaded anew.  (The reads' values are there anyway when their products run,
// so this costs nothing; without it only the compiler's order of the products
// would keep the reads ahead of the barrier.)
template <int LEFT>
__device__ __forceinline__ void d6_wait() {
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt((LEFT & 0xF) | ((LEFT >> 4) << 14) | (0x7 << 4));  // vmcnt(LEFT) lgkmcnt(0)
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __builtin_amdgcn_s_barrier();
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

}  // namespace ecalj
