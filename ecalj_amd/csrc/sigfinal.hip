// sigfinal.hip -- the final product of the bf16x3 Sigma_c,
//   zsec(m,m') += sum_{I,n} conj(czmelwc(I,n,m)) zmel(I,n,m')
// (S/m_sxcf_gemm.f90:599): ntq x ntq outputs over R = ngb nm rows, a tall
// product bound by reading both operands once.
#include <algorithm>

#include "bf16split.hpp"
#include "sigtile.hpp"

namespace ecalj {

// 16-byte loads of 8-byte aligned pairs (a column starts at any element)
typedef float f4a8 __attribute__((ext_vector_type(4), aligned(8)));

// One block per chunk of KC rows of one internal k, four waves with a quarter
// of the rows each; every wave forms all TT x TT 16x16 tiles, so each operand
// element is read once, straight from memory to the MFMA lane that uses it
// (lane (c, g): rows 8g..8g+7 of column c, 64 contiguous bytes; no LDS stage).
// The hi/lo split keeps all four products, lo*lo included (the kernel is bound
// by memory): the error of Sigma_c against 64 bits falls from 1.8e-7 to 0.8e-7
// (C2) and 1.1e-7 to 0.4e-7 (C3).  The GEMM tile it replaces padded ntq to 64
// and staged through LDS.  Sigma_c, before and after: C1-like (ntq = 8, 8 k)
// 0.180 -> 0.095 ms, C4-like windows (ntq = 16, 9 k, two launches per k) 21.8 ->
// 20.6 ms, C3 (ntq = 36, 12 k) 67.2 -> 66.6 ms.
template <int TT>
__global__ __launch_bounds__(256, 2) void sig_final_bf3_kernel(const cf* __restrict__ cz, const cf* __restrict__ z,
                                                               int64_t R, int64_t zs, int chunks,
                                                               const SigFinalK* __restrict__ tab, int nk, int KC,
                                                               int ntq, cf* __restrict__ part) {
  __shared__ float red[2][TT * 16][TT * 16 + 1];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int64_t q = blockIdx.x, base, row0;
  if (tab) {  // last k whose first chunk is at or before q
    int lo = 0, hi = nk - 1;
    const int q0 = tab[0].p0;
    while (lo < hi) {
      const int mid = (lo + hi + 1) / 2;
      if (tab[mid].p0 - q0 <= q) lo = mid;
      else hi = mid - 1;
    }
    R = tab[lo].R;
    base = tab[lo].off - tab[0].off;
    row0 = (q - (tab[lo].p0 - q0)) * KC;
  } else {
    base = zs * (q / chunks);
    row0 = (q % chunks) * KC;
  }
  const int64_t rend = min(R, row0 + KC), r1 = min(rend, row0 + (int64_t)(wave + 1) * (KC / 4));
  const int g8 = 8 * (lane >> 4), col = lane & 15;
  f4 cr[TT][TT], ci[TT][TT];
#pragma unroll
  for (int i = 0; i < TT; ++i)
#pragma unroll
    for (int j = 0; j < TT; ++j) cr[i][j] = ci[i][j] = f4{0, 0, 0, 0};
  struct Frag {
    u4q rh, rl, ih, il;
  };
  auto load = [&](const cf* x, int t, int64_t r, Frag& f) {
    const int m = 16 * t + col;
    f4 v[4] = {};
    if (m < ntq) {
      const cf* p = x + base + R * m + r;
      if (r + 8 <= r1) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = reinterpret_cast<const f4a8*>(p)[e];
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (r + e < r1) {
            v[e >> 1][2 * (e & 1)] = p[e].re;
            v[e >> 1][2 * (e & 1) + 1] = p[e].im;
          }
      }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const HiLo2 a = split2_bf16_alu(v[e][0], v[e][2]), b = split2_bf16_alu(v[e][1], v[e][3]);
      f.rh[e] = a.hi;
      f.rl[e] = a.lo;
      f.ih[e] = b.hi;
      f.il[e] = b.lo;
    }
  };
  for (int64_t rr = row0 + (int64_t)wave * (KC / 4); rr < r1; rr += 32) {
    Frag a[TT];
#pragma unroll
    for (int i = 0; i < TT; ++i) load(cz, i, rr + g8, a[i]);
#pragma unroll
    for (int j = 0; j < TT; ++j) {
      Frag b;
      load(z, j, rr + g8, b);
      const u4q nh = b.rh ^ 0x80008000u, nl = b.rl ^ 0x80008000u;
#define ECALJ_F_TERM(ACC, AF, BF)                                                                          \
  _Pragma("unroll") for (int i = 0; i < TT; ++i) ACC[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(      \
      __builtin_bit_cast(bf8, a[i].AF), __builtin_bit_cast(bf8, BF), ACC[i][j], 0, 0, 0);
      // conj(a) b: re = ar br + ai bi, im = ar bi - ai br
      ECALJ_F_TERM(cr, rl, b.rl)
      ECALJ_F_TERM(ci, rl, b.il)
      ECALJ_F_TERM(cr, il, b.il)
      ECALJ_F_TERM(ci, il, nl)
      ECALJ_F_TERM(cr, rl, b.rh)
      ECALJ_F_TERM(ci, rl, b.ih)
      ECALJ_F_TERM(cr, il, b.ih)
      ECALJ_F_TERM(ci, il, nh)
      ECALJ_F_TERM(cr, rh, b.rl)
      ECALJ_F_TERM(ci, rh, b.il)
      ECALJ_F_TERM(cr, ih, b.il)
      ECALJ_F_TERM(ci, ih, nl)
      ECALJ_F_TERM(cr, rh, b.rh)
      ECALJ_F_TERM(ci, rh, b.ih)
      ECALJ_F_TERM(cr, ih, b.ih)
      ECALJ_F_TERM(ci, ih, nh)
#undef ECALJ_F_TERM
    }
  }
  // the four waves' sums, in a fixed order
  for (int w = 1; w < 4; ++w) {
    if (wave == w) {
#pragma unroll
      for (int i = 0; i < TT; ++i)
#pragma unroll
        for (int j = 0; j < TT; ++j)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            red[0][16 * i + acc_row_f32(lane, e)][16 * j + col] = cr[i][j][e];
            red[1][16 * i + acc_row_f32(lane, e)][16 * j + col] = ci[i][j][e];
          }
    }
    __syncthreads();
    if (wave == 0) {
#pragma unroll
      for (int i = 0; i < TT; ++i)
#pragma unroll
        for (int j = 0; j < TT; ++j)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            cr[i][j][e] += red[0][16 * i + acc_row_f32(lane, e)][16 * j + col];
            ci[i][j][e] += red[1][16 * i + acc_row_f32(lane, e)][16 * j + col];
          }
    }
    __syncthreads();
  }
  if (wave == 0) {
    cf* P = part + (int64_t)ntq * ntq * q;
#pragma unroll
    for (int i = 0; i < TT; ++i)
#pragma unroll
      for (int j = 0; j < TT; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int m = 16 * i + acc_row_f32(lane, e), mp = 16 * j + col;
          if (m < ntq && mp < ntq) P[m + (int64_t)ntq * mp] = cf{cr[i][j][e], ci[i][j][e]};
        }
  }
}

// Rows of one chunk: 2048, fewer (down to 256) while the call has under 1024
// chunks (one block each, two on a CU); rows = all rows of the call.
int sig_final_chunk(int64_t rows) {
  int kc = 2048;
  while (kc > 256 && rows / kc < 1024) kc /= 2;
  return kc;
}

// Partials of nblk chunks: uniform k-points (R rows each, stride zs, chunks
// per k) when tab is null, else the nk k-points of tab (device), whose first
// offset and first chunk are the origin of cz, z and part.
ecalj_status sig_final_bf3(ecalj_ctx* h, const cf* cz, const cf* z, int64_t R, int64_t zs, int chunks,
                           const SigFinalK* tab, int nk, int64_t nblk, int KC, int ntq, cf* part) {
  if (nblk == 0) return ECALJ_OK;
  if (nblk > 0x7fffffff || ntq > kSigFinalMax) return ECALJ_ERR_DIM;
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3((unsigned)nblk), dim3(256), 0, h->stream, cz, z, R, zs, chunks, tab, nk, KC, ntq,
                       part);
  };
  if (ntq <= 16) go(sig_final_bf3_kernel<1>);
  else if (ntq <= 32) go(sig_final_bf3_kernel<2>);
  else if (ntq <= 48) go(sig_final_bf3_kernel<3>);
  else go(sig_final_bf3_kernel<4>);
  ECALJ_HIP(hipGetLastError());
  return ECALJ_OK;
}

}  // namespace ecalj
