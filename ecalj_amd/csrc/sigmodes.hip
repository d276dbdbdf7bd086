// sigmodes.hip -- the Sigma_c frequency contraction in frequency modes.
//
//   czmelwc(I,c) = sum_v sum_J Wt_v(I,J) wgt(v,c) zmel(J,c)
//
// costs one product of a W with zmel per frequency.  The weights of a range
// of middle states are smooth in the energy difference to the end state, so
// their vectors over the frequencies span far fewer dimensions than there
// are frequencies: with an orthonormal basis Q (nw1 x R) of the weights of a
// group of columns,
//   wgt(v,c) = sum_r (Q_vr / s_v) g_r(c),  g_r(c) = sum_v Q_vr s_v wgt(v,c),
//   czmelwc(I,c) = sum_r sum_J [sum_v Q_vr / s_v Wt_v](I,J) g_r(c) zmel(J,c),
// R products instead of nw1.  s_v is the Frobenius norm of W_v, so that a
// column's error is weighed as it enters the product.  R is the number of
// steps of a pivoted Gram-Schmidt after which the residual of EVERY column of
// the group is at most the rounding of its weights (2^-25 of their norm in the
// mixed forms, which take them in FP32, 2^-51 in FP64); weights
// that span all frequencies give R = nw1 and the plain contraction.
// R is found and used on the device: no host wait, and a captured graph
// replays with the ranks of its present inputs.
//
// Grouping: a column's weights depend on the distance |e_n - omega_m| of its
// middle and end states, and columns of like distance span few dimensions, so
// the columns of a k are sorted by it (by the weight at the highest frequency,
// which grows with it; whatever the weights are, the order only decides how
// low the ranks get) and taken in groups of whole column tiles.  C3, 21
// frequencies: mean rank 17 for one group, 8.8 for 4, 6.8 for 8, 6.0 for 12;
// groups of consecutive middle states instead of sorted columns: 10.6 for 8.
// More groups mean more modes to form and write; one mode costs about as much
// as 1.5 column tiles at one rank.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <vector>

#include "gemm64.hpp"
#include "moderule.hpp"
#include "sig3mtile.hpp"

namespace ecalj {

constexpr int kModeMax = Q3NW;    // frequencies, and therefore modes, of one launch
constexpr int kModeChunks = 16;   // partial sums of one W norm
template <class WT>
__host__ __device__ constexpr int mode_pool_planes(int nw1) { return mode_planes(sizeof(WT) == 8, nw1); }
// Largest residual of a column's weights, relative: 2^-25, the rounding of a
// weight to FP32; FP64: 2^-51, the weights' own rounding with that of the steps.
template <class G>
__host__ __device__ constexpr double mode_tol() { return sizeof(G) == 4 ? 0x1p-25 : 0x1p-51; }

// Columns c0 .. c0+cnt-1 of one internal k, sorted together.
struct SigModeSort {
  int64_t gsrc;   // weights of the k (elements of wgtim)
  int64_t cbase;  // first position in the sorted order of all k
  int c0, cnt, ncp, pad;
};
// One group: positions cbase .. cbase+ncp-1 of the sorted order, the first
// ncol of them columns, the rest padding (perm = -1).
struct SigMode {
  int64_t cbase;
  int64_t gsrc;   // weights of the k
  int64_t zsrc;   // zmel and czmelwc of the k (elements)
  int64_t wbase;  // plane pool of the k (16-bit elements)
  int k, ncol, ncp, pad;
};
struct SigModeTile {
  int grp, ct0, cnt, pad;  // up to 32 consecutive column tiles of one group
};
// What the device finds for a group: its modes, the first of them in the pool, the basis' size
struct SigModeRank {
  int rank, poff, raw, pad;
};

// ---------------------------------------------------------------- order of the columns
// Bitonic sort in LDS, one block per entry; keys (|weight at the highest
// frequency| as bits, column), so the order is unique.
__global__ __launch_bounds__(1024) void mode_sort_kernel(const SigModeSort* __restrict__ so,
                                                         const double* __restrict__ wgt, int nw1,
                                                         int* __restrict__ perm) {
  __shared__ unsigned long long key[kModeSort];
  const SigModeSort s = so[blockIdx.x];
  const int t = threadIdx.x;
  int M = 128;
  while (M < s.cnt) M *= 2;
  for (int i = t; i < M; i += 1024) {
    unsigned long long x = ~0ull;
    if (i < s.cnt) {
      const float g = fabsf((float)wgt[s.gsrc + (int64_t)nw1 * (s.c0 + i) + nw1 - 1]);
      x = ((unsigned long long)__float_as_uint(g) << 32) | (unsigned)i;
    }
    key[i] = x;
  }
  __syncthreads();
  for (int k = 2; k <= M; k *= 2)
    for (int j = k / 2; j > 0; j /= 2) {
      for (int q = t; q < M / 2; q += 1024) {
        const int i = 2 * q - (q & (j - 1)), l = i + j;  // bit j of i clear
        const unsigned long long x = key[i], y = key[l];
        if ((x > y) == ((i & k) == 0)) {
          key[i] = y;
          key[l] = x;
        }
      }
      __syncthreads();
    }
  for (int i = t; i < s.ncp; i += 1024)
    perm[s.cbase + i] = i < s.cnt ? s.c0 + (int)(unsigned)(key[i] & 0xffffffffu) : -1;
}

// ---------------------------------------------------------------- norms of W
// part[(k*nw1 + v)*kModeChunks + ch]: sum |W_v(I,J)|^2, I <= J, over every
// kModeChunks-th column: one pass over the upper triangles, bound by HBM.
__global__ __launch_bounds__(256) void mode_norm_kernel(const cd* __restrict__ w, int64_t ldw, int64_t w_stride,
                                                        int n, int nw1, double* __restrict__ part) {
  __shared__ double red[4];
  const int kv = blockIdx.y, k = kv / nw1, v = kv % nw1;
  const cd* W = w + w_stride * k + ldw * n * v;
  double s = 0.0;
  for (int J = blockIdx.x; J < n; J += kModeChunks) {
    const cd* col = W + ldw * J;
    for (int I = threadIdx.x; I <= J; I += 256) {
      const cd x = col[I];
      s += x.re * x.re + x.im * x.im;
    }
  }
  for (int o = 32; o > 0; o >>= 1) s += __shfl_down(s, o);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) part[(int64_t)kv * kModeChunks + blockIdx.x] = red[0] + red[1] + red[2] + red[3];
}

// ---------------------------------------------------------------- modes of one group
// One block per group.  X (nw1 x ncp, scratch) holds the residuals of the
// normalised columns, nrm their norms.  Each step takes the column of largest
// residual as the next basis vector and removes it from every column; the
// coefficients are those of the Gram-Schmidt, so the representation holds to
// the residual whatever rounding does to the basis' orthogonality.
// gm: mode weights (mode-major, ncp each); coef: kModeMax x kModeMax per group,
// coef[m*kModeMax + v] = Q_vr / s_v; rank >= 1.  Step r's mode is m = nw1-1-r: the
// contraction takes the modes from the smallest weights to the largest, so that
// its running sum is small until the last mode.  (Largest first, every later
// product is rounded at the size of the whole sum: czmelwc's error against
// extended precision was 1.5 to 2.2 times the plain contraction's in FP64 and
// 1.1 to 1.8 in FP32; smallest first it is 0.35 to 0.65 of it.)
// Latency-bound: 8-15 steps, each one pass over X in L2.
template <class WT>
__global__ __launch_bounds__(512) void mode_basis_kernel(const SigMode* __restrict__ grp, const int* __restrict__ perm,
                                                         const double* __restrict__ wgt,
                                                         const double* __restrict__ part, int nw1,
                                                         double* __restrict__ xs, double* __restrict__ nrms,
                                                         WT* __restrict__ gms, WT* __restrict__ coef,
                                                         SigModeRank* __restrict__ rank) {
  constexpr double kTol2 = mode_tol<WT>() * mode_tol<WT>();
  __shared__ double sv[kModeMax], q[kModeMax];
  __shared__ double bval[8];
  __shared__ int bcol[8];
  const SigMode g = grp[blockIdx.x];
  const int t = threadIdx.x, ncp = g.ncp;
  const int64_t cbase = g.cbase;
  double* X = xs + cbase * nw1;
  double* nrm = nrms + cbase;
  WT* gm = gms + cbase * nw1;
  WT* cf_ = coef + (int64_t)blockIdx.x * kModeMax * kModeMax;
  if (t < 64) {  // the first wave
    double s = 0.0;
    if (t < nw1)
      for (int c = 0; c < kModeChunks; ++c) s += part[((int64_t)g.k * nw1 + t) * kModeChunks + c];
    s = sqrt(s);
    // Only the ratios of the s_v matter (any positive s_v gives the product; they
    // weigh its error), so they are taken relative to the largest, by a power of
    // two: W of any scale gives the same digits.  A W at or near zero beside the
    // others takes a floor; one whose norm is infinite or NaN, and all of them
    // where every norm is zero, go unscaled, so that infinities and NaN reach
    // every mode and the result.
    double m = (s < 1e300) ? s : 0.0;
    for (int o = 32; o > 0; o >>= 1) m = fmax(m, __shfl_xor(m, o));
    int e = 0;
    if (m > 0.0) (void)frexp(m, &e);
    if (t < kModeMax) sv[t] = (m > 0.0 && s < 1e300) ? fmax(ldexp(s, -e), 1e-30) : 1.0;
  }
  for (int e = t; e < kModeMax * kModeMax; e += 512) cf_[e] = 0;
  __syncthreads();
  double best = 0.0;
  int bc = 0;
  for (int c = t; c < ncp; c += 512) {
    double x[kModeMax], m = 0.0;
    bool bad = false;
    if (c < g.ncol) {
      const double* src = wgt + g.gsrc + (int64_t)nw1 * perm[cbase + c];
#pragma unroll
      for (int v = 0; v < kModeMax; ++v) {
        x[v] = v < nw1 ? sv[v] * src[v] : 0.0;
        m = fmax(m, fabs(x[v]));
        bad |= !(fabs(x[v]) < __builtin_inf());
      }
    } else {
#pragma unroll
      for (int v = 0; v < kModeMax; ++v) x[v] = 0.0;
    }
    // the norm of x / 2^e (its squares in range), inv = 1 / that norm
    int e = 0;
    if (m > 0.0 && !bad) (void)frexp(m, &e);
    double n2 = 0.0;
#pragma unroll
    for (int v = 0; v < kModeMax; ++v) {
      x[v] = bad ? __builtin_nan("") : ldexp(x[v], -e);
      n2 += x[v] * x[v];
    }
    const double nr = sqrt(n2), inv = n2 > 0.0 ? 1.0 / nr : 0.0;
    double r2 = 0.0;
#pragma unroll
    for (int v = 0; v < kModeMax; ++v)
      if (v < nw1) {
        const double y = x[v] * inv;
        X[(int64_t)v * ncp + c] = y;
        r2 += y * y;
      }
    nrm[c] = ldexp(nr, e);
    gm[(int64_t)(nw1 - 1) * ncp + c] = bad ? (WT)__builtin_nanf("") : (WT)0;  // (stays where no mode is found)
    if (r2 > best) {
      best = r2;
      bc = c;
    }
  }
  int r = 0;
  for (; r < nw1; ++r) {
    // column of the largest residual (the lower index on a tie)
    for (int o = 32; o > 0; o >>= 1) {
      const double ov = __shfl_xor(best, o);
      const int oc = __shfl_xor(bc, o);
      if (ov > best || (ov == best && oc < bc)) {
        best = ov;
        bc = oc;
      }
    }
    if ((t & 63) == 0) {
      bval[t >> 6] = best;
      bcol[t >> 6] = bc;
    }
    __syncthreads();
    best = bval[0];
    bc = bcol[0];
#pragma unroll
    for (int w = 1; w < 8; ++w)
      if (bval[w] > best || (bval[w] == best && bcol[w] < bc)) {
        best = bval[w];
        bc = bcol[w];
      }
    if (!(best > kTol2)) break;
    if (t < nw1) {
      const double x = X[(int64_t)t * ncp + bc] / sqrt(best);
      q[t] = x;
      cf_[(nw1 - 1 - r) * kModeMax + t] = sv[t] > 0.0 ? (WT)(x / sv[t]) : (WT)0;
    }
    __syncthreads();
    best = 0.0;
    bc = 0;
    for (int c = t; c < ncp; c += 512) {
      double x[kModeMax], d = 0.0, r2 = 0.0;
#pragma unroll
      for (int v = 0; v < kModeMax; ++v) {
        x[v] = 0.0;
        if (v < nw1) {
          x[v] = X[(int64_t)v * ncp + c];
          d += q[v] * x[v];
        }
      }
#pragma unroll
      for (int v = 0; v < kModeMax; ++v)
        if (v < nw1) {
          const double y = x[v] - d * q[v];
          X[(int64_t)v * ncp + c] = y;
          r2 += y * y;
        }
      gm[(int64_t)(nw1 - 1 - r) * ncp + c] = (WT)(d * nrm[c]);
      if (r2 > best) {
        best = r2;
        bc = c;
      }
    }
  }
  if (t == 0) rank[blockIdx.x].raw = max(r, 1);  // all weights zero: one mode of weight 0
}

// Places of the groups' modes in the plane pool of their k (one block per
// group): coefp[(k pool planes + p) kModeMax + v] for plane p, nplane[k]
// planes.  When they do not fit, every group of the k takes the W planes of
// the frequencies themselves with the weights as they are: the plain contraction.
template <class WT>
__global__ __launch_bounds__(256) void mode_pack_kernel(const SigMode* __restrict__ grp, const int* __restrict__ kgrp,
                                                        const int* __restrict__ perm, const double* __restrict__ wgt,
                                                        int nw1, WT* __restrict__ gms,
                                                        const WT* __restrict__ coef, WT* __restrict__ coefp,
                                                        int* __restrict__ nplane, SigModeRank* __restrict__ rank) {
  const SigMode g = grp[blockIdx.x];
  const int g0 = kgrp[g.k], g1 = kgrp[g.k + 1];
  int tot = 0, before = 0;
  for (int i = g0; i < g1; ++i) {
    if (i == (int)blockIdx.x) before = tot;
    tot += rank[i].raw;
  }
  const bool fits = tot <= mode_pool_planes<WT>(nw1);
  SigModeRank* r = rank + blockIdx.x;
  const int R = fits ? r->raw : nw1;
  WT* cp = coefp + ((int64_t)g.k * mode_pool_planes<WT>(nw1) + (fits ? before : 0)) * kModeMax;
  if (threadIdx.x == 0) {
    r->rank = R;
    r->poff = fits ? before : 0;
    if ((int)blockIdx.x == g0) nplane[g.k] = fits ? tot : nw1;
  }
  if (fits || (int)blockIdx.x == g0)
    for (int e = threadIdx.x; e < R * kModeMax; e += 256)
      cp[e] = fits ? coef[((int64_t)blockIdx.x * kModeMax + nw1 - R) * kModeMax + e] : (e / kModeMax == e % kModeMax ? (WT)1 : (WT)0);
  if (!fits)
    for (int e = threadIdx.x; e < g.ncp * nw1; e += 256) {
      const int c = e % g.ncp, v = e / g.ncp;
      gms[g.cbase * nw1 + e] = c < g.ncol ? (WT)wgt[g.gsrc + (int64_t)nw1 * perm[g.cbase + c] + v] : (WT)0;
    }
}

// ---------------------------------------------------------------- W planes of the modes
// Per internal k and tile pair (a, b), a <= b, of W's upper triangle: the nw1
// frequencies of a 32 x 32 tile are read from HBM once and held in registers
// (FP32), then every mode of the k is formed and, through LDS, split and
// written as the two output tiles it feeds, (row tile a, k slice b) and (row
// tile b, k slice a), in the layout of split_w6_kernel.  Two modes per
// barrier: 512 threads are then 2 modes x 2 tiles x 32 rows x 4 chunks, one
// 16-byte store per plane each.  Rows beyond the last tile of n are not
// written: they only reach output rows that do not exist.  Bound by the writes
// of the planes (12 bytes per element and mode).
template <int NV>
__global__ __launch_bounds__(512, 4) void mode_planes_kernel(const cd* __restrict__ w, int64_t ldw, int64_t w_stride,
                                                             int n, int nw1, int MP, int NS, int64_t pool,
                                                             const int* __restrict__ kpool,
                                                             const float* __restrict__ coefp,
                                                             const int* __restrict__ nplane,
                                                             unsigned short* __restrict__ as) {
  __shared__ __align__(16) float2 tr[2][2][32][34];
  const int64_t tri = blockIdx.x;
  int b = (int)((sqrt(8.0 * (double)tri + 1.0) - 1.0) * 0.5);
  while ((int64_t)(b + 1) * (b + 2) / 2 <= tri) ++b;
  while ((int64_t)b * (b + 1) / 2 > tri) --b;
  const int a = (int)(tri - (int64_t)b * (b + 1) / 2);
  const int k = blockIdx.y;
  if (kpool[k] < 0) return;  // no columns
  const int I0 = a * 32, J0 = b * 32;
  // thread: row r of the tile, k values 2 kp and 2 kp + 1 of its slice
  const int r = threadIdx.x >> 4, kp = threadIdx.x & 15;
  const cd* W = w + w_stride * k;
  float xr[NV][2], xi[NV][2];
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const int I = I0 + r, J = J0 + 2 * kp + e;
    const bool low = I > J;  // below the diagonal (diagonal tiles only): conj(W(J, I))
    const int64_t o = low ? J + ldw * I : I + ldw * J;
    const bool in = I < n && J < n;
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      const cd x = (in && v < nw1) ? W[o + ldw * n * v] : cd{0.0, 0.0};
      xr[v][e] = (float)x.re;
      xi[v][e] = low ? -(float)x.im : (float)x.im;
    }
  }
  // writing: mode wm of the pair, tile wo (0: row tile a, 1: row tile b), row wr, chunk wc
  const int wc = threadIdx.x & 3, wr = (threadIdx.x >> 2) & 31, wo = (threadIdx.x >> 7) & 1, wm = threadIdx.x >> 8;
  const int64_t pst = (int64_t)MP * QBK, plane = (int64_t)NS * Q3PL * pst;
  const int row = (wo ? J0 : I0) + wr;
  unsigned short* A = as + pool * kpool[k] + (int64_t)(wo ? a : b) * Q3PL * pst + (int64_t)row * QBK +
                      8 * chunk_slot(row, wc);
  const bool put = wo == 0 || a < b;
  const int P = nplane[k];
  const float* c0 = coefp + (int64_t)k * mode_pool_planes<float>(nw1) * kModeMax;
  for (int p = 0; p < P; p += 2) {
    float2(*T)[32][34] = tr[(p >> 1) & 1];
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      const float* c = c0 + min(p + m, P - 1) * kModeMax;
      float ar[2] = {0.f, 0.f}, ai[2] = {0.f, 0.f};
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        const float f = c[v];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          ar[e] = fmaf(f, xr[v][e], ar[e]);
          ai[e] = fmaf(f, xi[v][e], ai[e]);
        }
      }
      *reinterpret_cast<f4*>(&T[m][r][2 * kp]) = f4{ar[0], ai[0], ar[1], ai[1]};
    }
    __syncthreads();  // the other buffer was last read before the previous barrier
    if (put && p + wm < P) {
      u4q h[Q3PL];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        f4 x;
        if (wo) {
          const float2 u = T[wm][8 * wc + 2 * q][wr], v = T[wm][8 * wc + 2 * q + 1][wr];
          x = f4{u.x, -u.y, v.x, -v.y};
        } else {
          x = *reinterpret_cast<const f4*>(&T[wm][wr][8 * wc + 2 * q]);
        }
        const HiLo2 s0 = split2_bf16_alu(x[0], x[2]), s1 = split2_bf16_alu(x[1], x[3]),
                    s2 = split2_bf16_alu(x[0] + x[1], x[2] + x[3]);
        h[0][q] = s0.hi;
        h[1][q] = s0.lo;
        h[2][q] = s1.hi;
        h[3][q] = s1.lo;
        h[4][q] = s2.hi;
        h[5][q] = s2.lo;
      }
      unsigned short* d = A + (p + wm) * plane;
#pragma unroll
      for (int q = 0; q < Q3PL; ++q) *reinterpret_cast<u4q*>(d + q * pst) = h[q];
    }
  }
}

// zp[p * NP + J] = zmel(J, column perm[p]), zero beyond n and for padding columns
__global__ __launch_bounds__(256) void mode_pad_kernel(const SigMode* __restrict__ grp, const int* __restrict__ perm,
                                                       const cf* __restrict__ z, int n, int NP, cf* __restrict__ zp) {
  const SigMode g = grp[blockIdx.y];
  for (int p = blockIdx.x; p < g.ncp; p += gridDim.x) {
    const int c = perm[g.cbase + p];
    const cf* src = z + g.zsrc + (int64_t)n * max(c, 0);
    cf* dst = zp + (g.cbase + p) * NP;
    for (int J = threadIdx.x; J < NP; J += 256) dst[J] = (c >= 0 && J < n) ? src[J] : cf{0.f, 0.f};
  }
}

// ---------------------------------------------------------------- contraction
// 1-D grid, block p on XCD p % 8: XCD x's j-th block belongs to super-tile
// (j / G)*8 + x, a (run of up to G column tiles of one group, row tile), so
// the blocks that read the same planes run together on one XCD and share them
// through its L2.  The runs come in the order of the groups within their k,
// the nearest columns (the highest ranks) first, so the short blocks end the launch.
__global__ __launch_bounds__(512, 1) void sig3m_modes_kernel(const SigMode* __restrict__ grp,
                                                             const SigModeTile* __restrict__ runs, int nrun, int G,
                                                             const SigModeRank* __restrict__ rank,
                                                             const int* __restrict__ perm,
                                                             const unsigned short* __restrict__ as,
                                                             const cf* __restrict__ zp, const float* __restrict__ gms,
                                                             int n, int nw1, int MP, int NS, int NP,
                                                             cf* __restrict__ cz) {
  __shared__ Sig3Smem s;
  const int p = blockIdx.x, x = p & 7, j = p >> 3, R = MP / QBM;
  const int sigma = (j / G) * 8 + x, loc = j % G;
  if (sigma >= nrun * R) return;
  const SigModeTile t = runs[sigma / R];
  if (loc >= t.cnt) return;
  const SigMode g = grp[t.grp];
  const int c0 = (t.ct0 + loc) * Q3BN, nwg = __builtin_amdgcn_readfirstlane(rank[t.grp].rank);
  const int64_t poff = __builtin_amdgcn_readfirstlane(rank[t.grp].poff);
  const float* gm = gms + g.cbase * nw1 + (int64_t)(nw1 - nwg) * g.ncp + c0;
  const int* pm = perm + g.cbase + c0;
  sig3m_tile<2>(
      s, as + g.wbase + poff * NS * Q3PL * MP * QBK, zp + g.cbase * NP,
      [&](int v, int e) { return gm[(int64_t)v * g.ncp + e]; }, [&](int e) { return pm[e]; }, n, 0, nwg, MP, NS, NP,
      (sigma % R) * QBM, c0, 0, cz + g.zsrc, (int64_t)n);
}

// ---------------------------------------------------------------- FP64 and FP32 forms
// Planes of the modes for the planar GEMM: mode p of the k as a full matrix
// W'(I,J), I < n, J < NK = n rounded up to 8 (zero beyond n), in the
// contraction's type, from the upper triangle (tile pair (a, b) written as
// (I, J) and, through LDS, as its conjugate transpose).
template <class T, int NV>
__global__ __launch_bounds__(512) void mode_full_kernel(const cd* __restrict__ w, int64_t ldw, int64_t w_stride,
                                                        int n, int nw1, int64_t pool, const int* __restrict__ kpool,
                                                        const typename ElemT<T>::V* __restrict__ coefp,
                                                        const int* __restrict__ nplane, T* __restrict__ as) {
  typedef typename ElemT<T>::V V;
  __shared__ T tr[2][32][33];
  const int64_t tri = blockIdx.x;
  int b = (int)((sqrt(8.0 * (double)tri + 1.0) - 1.0) * 0.5);
  while ((int64_t)(b + 1) * (b + 2) / 2 <= tri) ++b;
  while ((int64_t)b * (b + 1) / 2 > tri) --b;
  const int a = (int)(tri - (int64_t)b * (b + 1) / 2);
  const int k = blockIdx.y;
  if (kpool[k] < 0) return;  // no columns
  // thread: elements (I0 + i, J0 + j + 16 e)
  const int i = threadIdx.x & 31, j = threadIdx.x >> 5;
  const int I = a * 32 + i, I2 = b * 32 + i;
  const cd* W = w + w_stride * k;
  V xr[NV][2], xi[NV][2];
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const int J = b * 32 + j + 16 * e;
    const bool low = I > J;
    const int64_t o = low ? J + ldw * I : I + ldw * J;
    const bool in = I < n && J < n;
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      const cd x = (in && v < nw1) ? W[o + ldw * n * v] : cd{0.0, 0.0};
      xr[v][e] = (V)x.re;
      xi[v][e] = low ? -(V)x.im : (V)x.im;
    }
  }
  const int P = nplane[k];
  const int NK = (n + 7) / 8 * 8;
  const int64_t nn = (int64_t)n * NK;
  T* A = as + pool * kpool[k];
  const V* c0 = coefp + (int64_t)k * mode_pool_planes<V>(nw1) * kModeMax;
  for (int p = 0; p < P; ++p) {
    T(*L)[33] = tr[p & 1];
    const V* c = c0 + p * kModeMax;
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      V ar = 0, ai = 0;
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        ar += c[v] * xr[v][e];
        ai += c[v] * xi[v][e];
      }
      const int J = b * 32 + j + 16 * e;
      if (I < n && J < NK) A[nn * p + I + (int64_t)n * J] = T{ar, ai};
      L[j + 16 * e][i] = T{ar, -ai};
    }
    if (a == b) continue;  // uniform
    __syncthreads();
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int J2 = a * 32 + j + 16 * e;
      if (I2 < n && J2 < NK) A[nn * p + I2 + (int64_t)n * J2] = L[i][j + 16 * e];
    }
  }
}

// B operand of the planar GEMM: B(kk, c') = gm_r(c') zmel(J, perm[c']), kk = r NK + J.
// A thread's columns stay the same over the stages, so their addresses are kept.
template <class T, int BN, int BK>
struct LdMode {
  typedef typename ElemT<T>::V V;
  static constexpr int R = BN * BK / kThreads, XS = kThreads / BK;
  const T* z[R];   // column base (null: padding)
  const V* gm;     // weights of the thread's first column
  int n, NK, ncp, K;
  unsigned inv;    // ceil(2^32 / NK): kk / NK = umulhi(kk, inv) while kk NK < 2^32, n >= 2
  struct Regs { V re[R]; V im[R]; };
  __device__ void init(const T* zk, const V* gms, const int* pm, int n_, int ncp_, int K_) {
    n = n_;
    ncp = ncp_;
    K = K_;
    NK = (n + 7) / 8 * 8;
    inv = (unsigned)((0x100000000ull + NK - 1) / NK);
    const int x = threadIdx.x / BK;
    gm = gms + x;
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const int c = pm[x + q * XS];
      z[q] = c >= 0 ? zk + (int64_t)n * c : nullptr;
    }
  }
  __device__ void fetch(int, int k0, Regs& r) const {
    const int kk = k0 + threadIdx.x % BK;
    const int v = (int)__umulhi((unsigned)kk, inv), J = kk - v * NK;
    const bool in = kk < K && J < n;
#pragma unroll
    for (int q = 0; q < R; ++q) {
      r.re[q] = 0;
      r.im[q] = 0;
      if (in && z[q]) {
        const V g = gm[(int64_t)v * ncp + q * XS];
        const T x = z[q][J];
        r.re[q] = g * x.re;
        r.im[q] = g * x.im;
      }
    }
  }
  template <class S>
  __device__ void store(S& s, const Regs& r) const {
#pragma unroll
    for (int q = 0; q < R; ++q) s.putB(threadIdx.x % BK, threadIdx.x / BK + q * XS, r.re[q], r.im[q]);
  }
};

// czmelwc of the FP32 form on the planar GEMM core, 64 x 64 tiles, K = rank x
// NK; block order as sig3m_modes_kernel.
template <int MODE, class T>
__global__ __launch_bounds__(kThreads) void mode_gemm_kernel(const SigMode* __restrict__ grp,
                                                             const SigModeTile* __restrict__ runs, int nrun, int G,
                                                             const SigModeRank* __restrict__ rank,
                                                             const int* __restrict__ perm, const T* __restrict__ as,
                                                             const T* __restrict__ zmel,
                                                             const typename ElemT<T>::V* __restrict__ gms, int n,
                                                             int nw1, T* __restrict__ cz) {
  constexpr int BK = ModeBK<MODE>::value;
  typedef typename ElemT<T>::V V;
  __shared__ typename StageOf<MODE, 64, 64, BK>::type s;
  const int p = blockIdx.x, x = p & 7, j = p >> 3, R = (n + 63) / 64;
  const int sigma = (j / G) * 8 + x, loc = j % G;
  if (sigma >= nrun * R) return;
  const SigModeTile t = runs[sigma / R];
  if (loc >= t.cnt) return;
  const SigMode g = grp[t.grp];
  const int NK = (n + 7) / 8 * 8, c0 = (t.ct0 + loc) * 64, m0 = (sigma % R) * 64, K = rank[t.grp].rank * NK;
  const V* gm = gms + g.cbase * nw1 + (int64_t)(nw1 - rank[t.grp].rank) * g.ncp + c0;
  const int* pm = perm + g.cbase + c0;
  Ld<AccN<T, false>, 64, BK, true, 1> la{
      AccN<T, false>{as + g.wbase + (int64_t)rank[t.grp].poff * n * NK, (int64_t)n, n, K, (V)1}};
  LdMode<T, 64, BK> lb;
  lb.init(zmel + g.zsrc, gm, pm, n, g.ncp, K);
  Core<MODE, 64, 64, BK, false> core;
  gemm_mainloop<MODE, 64, 64, BK, false>(la, lb, m0, 0, K, s, core);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  core.for_each(wave >> 1, wave & 1, lane, [&](int rr, int cc, double xr, double xi) {
    const int i = m0 + rr, c = pm[cc];
    if (i < n && c >= 0) st_c(cz + g.zsrc + i + (int64_t)n * c, xr, xi);
  });
}

// czmelwc of the FP64 form on the 128 x 64 tile of gemm64.hpp: a lane moves 8 k
// of one column per stage, so the gather costs one pointer per lane, and the
// mode's weight multiplies the fragments of the lane's two columns after the
// LDS read.  Block order as sig3m_modes_kernel.
__global__ __launch_bounds__(D6T, 4) void mode_gemm64_kernel(const SigMode* __restrict__ grp,
                                                             const SigModeTile* __restrict__ runs, int nrun, int G,
                                                             const SigModeRank* __restrict__ rank,
                                                             const int* __restrict__ perm, const cd* __restrict__ as,
                                                             const cd* __restrict__ zmel,
                                                             const double* __restrict__ gms, int n, int nw1,
                                                             cd* __restrict__ cz) {
  __shared__ D6Smem s;
  const int p = blockIdx.x, x = p & 7, j = p >> 3, NR = (n + D6M - 1) / D6M;
  const int sigma = (j / G) * 8 + x, loc = j % G;
  if (sigma >= nrun * NR) return;
  const SigModeTile t = runs[sigma / NR];
  if (loc >= t.cnt) return;
  const SigMode g = grp[t.grp];
  const int NS = (n + D6K - 1) / D6K, NK = NS * D6K;
  const int c0 = (t.ct0 + loc) * D6N, m0 = (sigma % NR) * D6M;
  const int R = __builtin_amdgcn_readfirstlane(rank[t.grp].rank);
  const int* pm = perm + g.cbase + c0;
  const double* gm = gms + g.cbase * nw1 + (int64_t)(nw1 - R) * g.ncp + c0;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  typedef D6Ld<D6M, false> LA;
  typedef D6Ld<D6N, true> LB;
  static_assert(D6M == QBM, "row tiles are counted in QBM");
  static_assert(LB::NI == 1, "one load of B per wave and stage");
  LA la;
  la.init(as + g.wbase + (int64_t)rank[t.grp].poff * n * NK, n, m0, n, wave, lane);
  // B: the lane's column (padding columns take column 0 with weight 0) and k
  const int bx = wave * 8 + (lane >> 3), bk = (lane & 7) ^ (bx & 7);
  const cd* bp = zmel + g.zsrc + (int64_t)n * max(pm[bx], 0);
  int ir = 0, iks = 0;  // the next stage to issue
  auto issue = [&](int buf) {
    la.issue(s.a[buf], wave, (ir * NS + iks) * D6K, R * NK);
    __builtin_amdgcn_global_load_lds((gbl_ptr_t)(bp + min(iks * D6K + bk, n - 1)), (lds_ptr_t)(s.b[buf] + wave * 64),
                                     16, 0, 0);
    if (iks + 1 < NS) ++iks;
    else if (ir + 1 < R) iks = 0, ++ir;
  };
  D6Acc c;
  c.zero();
  issue(0);
  issue(1);
  int buf = 0;
  for (int r = 0; r < R; ++r) {
    double w[2];
#pragma unroll
    for (int q = 0; q < 2; ++q) w[q] = gm[(int64_t)r * g.ncp + wn * 32 + q * 16 + (lane & 15)];
    for (int ks = 0; ks < NS; ++ks) {
      d6_wait<LA::NI + 1>();
      issue(buf == 0 ? 2 : buf - 1);
      d6_stage<LA, LB, false, true>(c, s.a[buf], s.b[buf], wm, wn, lane, 1.0, 1.0, w, D6K);
      buf = buf == 2 ? 0 : buf + 1;
    }
  }
  ECALJ_WAIT_VMCNT(0);  // the repeated stages have landed before the block's LDS is released
#pragma unroll
  for (int jj = 0; jj < 2; ++jj) {
    const int col = pm[wn * 32 + jj * 16 + (lane & 15)];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        __builtin_amdgcn_sched_barrier(0);  // (one address at a time)
        const int I = m0 + wm * 32 + i * 16 + acc_row_f64(lane, e);
        if (I < n && col >= 0) cz[g.zsrc + I + (int64_t)n * col] = cd{c.cr[i][jj][e], c.ci[i][jj][e]};
      }
  }
}

// ---------------------------------------------------------------- host
// Whether the mode form is taken, for nk k-points of nm[step k] ntq columns:
// 8 frequencies (fewer leave too little to save) to kModeMax (one launch holds
// no more), and where it pays (moderule.hpp).  n: what LdMode divides by (beyond
// it the planes pass the scratch limit in every form).
// Tuner mode kTuneModes asks for it at any size, any other forced variant for
// the plain contraction, in every form.
bool sig_modes_pays(const ecalj_ctx* h, int mode, int n, int64_t nk, const int* nm, int step, int ntq, int nw1) {
  if (nw1 > kModeMax || n < 2 || n > 13000) return false;
  if (mode == MBF3 && h->sigc_fp8) return false;
  if (h->tune_mode == kTuneModes) return true;
  if (h->tune_mode != 0) return false;
  return nw1 >= 8 && mode_pays(mode == M64, mode == MBF3, n, nk, nm, step, ntq, nw1);
}

static size_t al256(size_t b) { return (b + 255) & ~(size_t)255; }

// What one k of a call takes: elements of its plane pool, and whether its
// zmel is copied in sorted order (bf16x3).
static int64_t mode_planes_max(int mode, int nw1) {
  return mode_planes(mode == M64, nw1);
}
static int64_t mode_pool(int mode, int n, int nw1) {
  return mode_planes_max(mode, nw1) * (mode == MBF3 ? (int64_t)sig3m_a_elems_per_k(n, 1) : (int64_t)n * ((n + 7) / 8 * 8));
}
static size_t mode_pool_elem(int mode) { return mode == MBF3 ? 2 : mode == M64 ? sizeof(cd) : sizeof(cf); }

// Scratch of one k: plane pool, padded zmel, order, residuals, weights
size_t sig_modes_bytes(int mode, int n, int nm, int ntq, int nw1) {
  const size_t wt = mode == M64 ? 8 : 4;
  // norms, coefficients and counts of a k, also of one without columns
  const size_t per_k = (size_t)nw1 * kModeChunks * 8 + mode_planes_max(mode, nw1) * kModeMax * wt + 4;
  if (nm == 0) return al256(per_k);
  const int64_t NP = pad_to(n, QBK), ncol = (int64_t)nm * ntq, ncp = (ncol + Q3BN - 1) / Q3BN * Q3BN;
  const int64_t groups = kModeGroups * (ncol / kModeSort + 1);
  return al256(mode_pool(mode, n, nw1) * mode_pool_elem(mode) +
               (size_t)ncp * ((mode == MBF3 ? sizeof(cf) * NP : 0) + (8 + wt) * nw1 + 12) +
               (kModeMax * kModeMax * wt + sizeof(SigModeRank)) * groups + per_k + 4096);
}

// k-points whose (k, frequency) and (k, group) pairs fit one grid's y.
int sig_modes_max_k(int nw1, int64_t ncol) {
  return (int)std::max<int64_t>(1, 65535 / std::max<int64_t>(nw1, kModeGroups * (ncol / kModeSort + 1)));
}

// czmelwc of nk internal k-points (zmel, wgt, cz packed per k: n x nm[k] x ntq
// and nw1 x nm[k] x ntq) in the storage type of the mode; scratch: the sum of
// sig_modes_bytes.
template <int MODE, class T, class WT>
static ecalj_status sig_modes_t(ecalj_ctx* h, int nk, const int* nm, int ntq, const T* zmel, int n, int nw1,
                                const cd* wc, int64_t ldw, int64_t w_stride, const double* wgt, T* cz,
                                unsigned char* scratch) {
  constexpr int BN = MODE == MBF3 ? Q3BN : 64;
  const int MP = pad_to(n, QBM), NP = pad_to(n, QBK), NS = NP / QBK, R = MODE == M32 ? (n + 63) / 64 : MP / QBM;
  const int64_t pool = mode_pool(MODE, n, nw1);
  std::vector<SigModeSort> sorts;
  std::vector<SigMode> grp;
  std::vector<int> kgrp(2 * nk + 1, 0);  // first group of each k, then its pool (-1: no columns)
  int64_t cols = 0, co = 0;
  int pools = 0;
  int maxg = 0;
  for (int k = 0; k < nk; ++k) {
    const int64_t N = (int64_t)nm[k] * ntq;
    if (N > 0x7fffffff / 2) return ECALJ_ERR_DIM;
    const int TT = (int)((N + BN - 1) / BN), parts = mode_sorts(TT, BN);
    const int tp = parts ? (TT + parts - 1) / parts : 0;  // column tiles of one sort
    for (int t0 = 0; t0 < TT; t0 += tp) {
      const int tn = std::min(tp, TT - t0), cnt = (int)std::min<int64_t>(N - (int64_t)t0 * BN, (int64_t)tn * BN);
      sorts.push_back({co * nw1, cols, t0 * BN, cnt, tn * BN, 0});
      const int gt = mode_group_tiles(tn, parts, MODE == M64, MODE == MBF3, nw1);
      for (int g0 = 0; g0 < tn; g0 += gt) {
        const int gn = std::min(gt, tn - g0);
        grp.push_back({cols + g0 * BN, co * nw1, co * n, pools * pool, k, std::min(gn * BN, cnt - g0 * BN), gn * BN,
                       0});
      }
      cols += (int64_t)tn * BN;
    }
    co += N;
    kgrp[nk + 1 + k] = N > 0 ? pools++ : -1;
    kgrp[k + 1] = (int)grp.size();
    maxg = std::max(maxg, kgrp[k + 1] - kgrp[k]);
  }
  const int ng = (int)grp.size();
  if (ng == 0) return ECALJ_OK;
  // runs of column tiles, group index within the k outermost
  std::vector<SigModeTile> runs;
  int G = 1, ncpmax = 0;
  for (int gi = 0; gi < maxg; ++gi)
    for (int k = 0; k < nk; ++k) {
      if (kgrp[k] + gi >= kgrp[k + 1]) continue;
      const SigMode& m = grp[kgrp[k] + gi];
      const int ct = m.ncp / BN, parts = (ct + 31) / 32, per = (ct + parts - 1) / parts;
      for (int c = 0; c < ct; c += per) runs.push_back({kgrp[k] + gi, c, std::min(per, ct - c), 0});
      G = std::max(G, per);
      ncpmax = std::max(ncpmax, m.ncp);
    }
  const TuneKey key{TUNE_SIGC_MODES, n, cols, nw1, nk};  // one line of the report per shape
  int seen;
  if (!tune_lookup(h, key, &seen)) {
    h->tuned[key] = 0;
    char line[128];
    snprintf(line, sizeof line, "sigc_modes [%d %lld %d %d]: frequency modes\n", n, (long long)cols, nw1, nk);
    h->tune_log += line;
  }
  const int64_t npair = (int64_t)NS * (NS + 1) / 2;
  const int64_t blocks = 8LL * G * (((int64_t)runs.size() * R + 7) / 8);
  if (blocks > 0x7fffffff || npair > 0x7fffffff || nk > 65535 || (int64_t)nw1 * nk > 65535 || ng > 65535)
    return ECALJ_ERR_DIM;
  unsigned char* q = scratch;
  auto take = [&](size_t bytes) {
    unsigned char* r = q;
    q += al256(bytes);
    return r;
  };
  unsigned char* as = take((size_t)(pool * pools) * mode_pool_elem(MODE));
  cf* zp = (cf*)take(MODE == MBF3 ? sizeof(cf) * (size_t)cols * NP : 0);
  double* xs = (double*)take(sizeof(double) * (size_t)cols * nw1);
  double* nrm = (double*)take(sizeof(double) * (size_t)cols);
  WT* gm = (WT*)take(sizeof(WT) * (size_t)cols * nw1);
  int* perm = (int*)take(sizeof(int) * (size_t)cols);
  WT* coef = (WT*)take(sizeof(WT) * kModeMax * kModeMax * (size_t)ng);
  double* part = (double*)take(sizeof(double) * kModeChunks * (size_t)nw1 * nk);
  SigModeRank* rank = (SigModeRank*)take(sizeof(SigModeRank) * (size_t)ng);
  WT* coefp = (WT*)take(sizeof(WT) * kModeMax * (size_t)mode_planes_max(MODE, nw1) * nk);
  int* nplane = (int*)take(sizeof(int) * (size_t)nk);
  // tables
  const size_t b0 = sizeof(SigModeSort) * sorts.size(), b1 = sizeof(SigMode) * grp.size();
  const size_t b2 = sizeof(SigModeTile) * runs.size(), b3 = sizeof(int) * kgrp.size();
  std::vector<unsigned char> blob(b0 + b1 + b2 + b3);
  std::memcpy(blob.data(), sorts.data(), b0);
  std::memcpy(blob.data() + b0, grp.data(), b1);
  std::memcpy(blob.data() + b0 + b1, runs.data(), b2);
  std::memcpy(blob.data() + b0 + b1 + b2, kgrp.data(), b3);
  unsigned char* d;
  ECALJ_TRY(upload_blob(h, ecalj_ctx::S_GTAB, blob, &d));
  const SigModeSort* ds = (const SigModeSort*)d;
  const SigMode* dg = (const SigMode*)(d + b0);
  const SigModeTile* dr = (const SigModeTile*)(d + b0 + b1);
  const int* dk = (const int*)(d + b0 + b1 + b2);

  hipLaunchKernelGGL(mode_sort_kernel, dim3((unsigned)sorts.size()), dim3(1024), 0, h->stream, ds, wgt, nw1, perm);
  ECALJ_HIP(hipGetLastError());
  hipLaunchKernelGGL(mode_norm_kernel, dim3(kModeChunks, nw1 * nk), dim3(256), 0, h->stream, wc, ldw, w_stride, n, nw1,
                     part);
  ECALJ_HIP(hipGetLastError());
  hipLaunchKernelGGL(mode_basis_kernel<WT>, dim3(ng), dim3(512), 0, h->stream, dg, perm, wgt, part, nw1, xs, nrm, gm,
                     coef, rank);
  ECALJ_HIP(hipGetLastError());
  hipLaunchKernelGGL(mode_pack_kernel<WT>, dim3(ng), dim3(256), 0, h->stream, dg, dk, perm, wgt, nw1, gm, coef, coefp,
                     nplane, rank);
  ECALJ_HIP(hipGetLastError());
  const dim3 pgrid((unsigned)npair, nk);
  if constexpr (MODE == MBF3) {
    auto planes = [&](auto kern) {
      hipLaunchKernelGGL(kern, pgrid, dim3(512), 0, h->stream, wc, ldw, w_stride, n, nw1, MP, NS, pool, dk + nk + 1,
                         coefp, nplane, (unsigned short*)as);
    };
    if (nw1 <= 13) planes(mode_planes_kernel<13>);
    else if (nw1 <= 17) planes(mode_planes_kernel<17>);
    else if (nw1 <= 21) planes(mode_planes_kernel<21>);
    else planes(mode_planes_kernel<24>);
    ECALJ_HIP(hipGetLastError());
    hipLaunchKernelGGL(mode_pad_kernel, dim3(std::min(ncpmax, 4096), ng), dim3(256), 0, h->stream, dg, perm, zmel, n,
                       NP, zp);
    ECALJ_HIP(hipGetLastError());
  } else {
    auto planes = [&](auto kern) {
      hipLaunchKernelGGL(kern, pgrid, dim3(512), 0, h->stream, wc, ldw, w_stride, n, nw1, pool, dk + nk + 1, coefp,
                         nplane, (T*)as);
    };
    if (nw1 <= 13) planes(mode_full_kernel<T, 13>);
    else if (nw1 <= 17) planes(mode_full_kernel<T, 17>);
    else planes(mode_full_kernel<T, 24>);
    ECALJ_HIP(hipGetLastError());
  }
  int tev = -1;
  ECALJ_TRY(timing_begin(h, 0, &tev));
  if constexpr (MODE == MBF3)
    hipLaunchKernelGGL(sig3m_modes_kernel, dim3((unsigned)blocks), dim3(512), 0, h->stream, dg, dr, (int)runs.size(), G,
                       rank, perm, (const unsigned short*)as, zp, gm, n, nw1, MP, NS, NP, cz);
  else if constexpr (MODE == M64)
    hipLaunchKernelGGL(mode_gemm64_kernel, dim3((unsigned)blocks), dim3(D6T), 0, h->stream, dg, dr, (int)runs.size(),
                       G, rank, perm, (const cd*)as, zmel, gm, n, nw1, cz);
  else
    hipLaunchKernelGGL((mode_gemm_kernel<MODE, T>), dim3((unsigned)blocks), dim3(kThreads), 0, h->stream, dg, dr,
                       (int)runs.size(), G, rank, perm, (const T*)as, zmel, gm, n, nw1, cz);
  ECALJ_HIP(hipGetLastError());
  ECALJ_TRY(timing_end(h, 0, tev));
  return ECALJ_OK;
}

ecalj_status sig_modes(ecalj_ctx* h, int mode, int nk, const int* nm, int ntq, const void* zmel, int n, int nw1,
                       const cd* wc, int64_t ldw, int64_t w_stride, const double* wgt, void* cz,
                       unsigned char* scratch) {
  if (mode == M64)
    return sig_modes_t<M64, cd, double>(h, nk, nm, ntq, (const cd*)zmel, n, nw1, wc, ldw, w_stride, wgt, (cd*)cz,
                                        scratch);
  if (mode == M32)
    return sig_modes_t<M32, cf, float>(h, nk, nm, ntq, (const cf*)zmel, n, nw1, wc, ldw, w_stride, wgt, (cf*)cz,
                                       scratch);
  return sig_modes_t<MBF3, cf, float>(h, nk, nm, ntq, (const cf*)zmel, n, nw1, wc, ldw, w_stride, wgt, (cf*)cz,
                                      scratch);
}

}  // namespace ecalj
