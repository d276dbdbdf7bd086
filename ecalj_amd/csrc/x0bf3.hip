// x0bf3.hip -- x0gemm (S/x0gemm.f90:2-97) in the bf16x3 form on the block tile of sigtile.hpp.
#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "bf16split.hpp"
#include "sigtile.hpp"

namespace ecalj {

// ================================================================ x0gemm on the bf16x3 core
// rcxq(:,:,slice(bin)) += sum_{t in bin} conj(z_t(i)) w_t z_t(ipr_col-1+j)
// (S/x0gemm.f90:51-97) as one grouped GEMM per histogram bin: the bin's
// columns are gathered once into pre-split bf16 planes (A = z_t, B = w_t z_t,
// K = the bin's entries padded to 32 with zeros), and every (bin, row tile,
// column tile) is one block.  A square output (ipr_col = 1, npr_col = npr) is
// Hermitian: only the tiles that reach the upper triangle run, and each
// element I < c also adds its conjugate.  If no weight is negative, that
// output needs one set of planes, A = B = sqrt(w_t) z_t, which halves the
// gather's writes and the tiles' plane reads.

constexpr int X0T = 64;  // tile rows and columns

// One block per (K slice of 32 entries, 64 rows), four lanes per row (its four
// chunks): a wave writes 16 whole rows of each plane.  Weight of entry t: 1, w,
// sqrt(w).  Memory-bound; at C2 with 32 k-points 235 us for one set of planes,
// where two sets, four lanes per row over all rows of a slice, took 474.
enum { X0_Z = 0, X0_WZ = 1, X0_RZ = 2 };
__global__ __launch_bounds__(256) void x0_split_kernel(const cf* __restrict__ z, const int64_t* __restrict__ colp,
                                                       const double* __restrict__ wp, int mode, int64_t off,
                                                       int nrow, int RP, unsigned short* __restrict__ out,
                                                       float* __restrict__ res) {
  __shared__ int64_t c[QBK];
  __shared__ float w[QBK];
  const int nr = RP / X0T, rb = (int)(blockIdx.x % nr);
  const int64_t sl = blockIdx.x / nr;
  if (threadIdx.x < QBK) {
    const int64_t t = sl * QBK + threadIdx.x;
    c[threadIdx.x] = colp[t];
    w[threadIdx.x] = mode == X0_Z ? 1.f : (float)(mode == X0_WZ ? wp[t] : sqrt(wp[t]));
  }
  __syncthreads();
  const int ch = threadIdx.x & 3, r = rb * X0T + (threadIdx.x >> 2);
  const SplitMasks mk = split_masks();
  u4q rh, rl, ih, il;
  float d = 0.f;  // sum of x^2 - (hi^2 + 2 hi lo) over both parts
  auto rest = [&](float x, unsigned h, unsigned l) {  // h, l: bf16 in the upper half
    const float a = __uint_as_float(h), b = __uint_as_float(l), r = x - a;  // exact
    d = fmaf(r, r, fmaf(a + a, r - b, d));
  };
  auto split = [&](float x0, float x1, u4q& hi, u4q& lo, int q) {
    const HiLo2 s = split2_bf16(x0, x1, mk);
    hi[q] = s.hi;
    lo[q] = s.lo;
    if (res) {
      rest(x0, s.hi << 16, s.lo << 16);
      rest(x1, s.hi & 0xffff0000u, s.lo & 0xffff0000u);
    }
  };
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    float xr[2], xi[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int64_t cc = c[8 * ch + 2 * q + u];
      const float f = w[8 * ch + 2 * q + u];
      xr[u] = xi[u] = 0.f;
      if (cc >= 0 && r < nrow) {
        const cf x = z[cc + off + r];
        xr[u] = f * x.re;
        xi[u] = f * x.im;
      }
    }
    split(xr[0], xr[1], rh, rl, q);
    split(xi[0], xi[1], ih, il, q);
  }
  if (res) {
    d += __shfl_xor(d, 1);
    d += __shfl_xor(d, 2);
    if (ch == 0) res[sl * RP + r] = d;
  }
  const int64_t pst = (int64_t)RP * QBK;
  unsigned short* P = out + sl * 4 * pst + (int64_t)r * QBK + 8 * chunk_slot(r, ch);
  *reinterpret_cast<u4q*>(P) = rh;
  *reinterpret_cast<u4q*>(P + pst) = rl;
  *reinterpret_cast<u4q*>(P + 2 * pst) = ih;
  *reinterpret_cast<u4q*>(P + 3 * pst) = il;
}

struct X0Bin {
  int64_t aoff, boff;  // plane offsets (elements) of the bin's first K slice
  int ns, slice;       // K slices, output slice
};

// One 64 x 64 tile of one bin per block, 4 waves of 32 x 32, one K slice of 32
// in LDS; C += conj(A) B.  MFMA-bound, with the output (read and written once
// per bin) beside it: four blocks per CU in different phases overlap the stage
// loads, the products and the updates.  At C2 with 32 k-points (some 100 000
// entries in 135 bins) 580 us, 0.93 PFLOP/s of bf16 products; one 128 x 128
// block per CU with two slices in LDS, where nothing ran beside the updates,
// took 780, this tile with two slices and two blocks per CU 10% more than with one.
__global__ __launch_bounds__(256, 4) void x0_bf3_kernel(const X0Bin* __restrict__ bins, int nbin,
                                                        const unsigned short* __restrict__ as,
                                                        const unsigned short* __restrict__ bs, int npr, int npr_col,
                                                        int MP, int NCP, const float* __restrict__ res, int mirror,
                                                        cf* __restrict__ rcxq, int64_t slice_elems) {
  typedef float f4a8 __attribute__((ext_vector_type(4), aligned(8)));
  __shared__ alignas(16) unsigned short sa[4][X0T * QBK], sb[4][X0T * QBK];
  // blocks 8 y' + x in a row of the grid run on XCD x: all tiles of a bin on one
  // XCD, whose L2 then holds the bin's planes once for all of them
  const int bin = 8 * blockIdx.y + (blockIdx.x & 7);
  if (bin >= nbin) return;
  int ti = 0, tj = blockIdx.x >> 3;  // the tile's number in the bin, row by row
  for (int len = NCP / X0T; tj >= len; len -= mirror) {
    tj -= len;
    ++ti;
  }
  const int I0 = ti * X0T, c0 = (tj + (mirror ? ti : 0)) * X0T;
  const X0Bin bb = bins[bin];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int64_t apst = (int64_t)MP * QBK, bpst = (int64_t)NCP * QBK;
  const unsigned short* A = as + bb.aoff + (int64_t)I0 * QBK;
  const unsigned short* B = bs + bb.boff + (int64_t)c0 * QBK;
  auto issue = [&](int ks) {  // wave p loads plane p of both
    const unsigned short* a = A + (ks * 4 + wave) * apst + lane * 8;
    const unsigned short* b = B + (ks * 4 + wave) * bpst + lane * 8;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      __builtin_amdgcn_global_load_lds((gbl_ptr_t)(a + 512 * q), (lds_ptr_t)(&sa[wave][512 * q]), 16, 0, 0);
      __builtin_amdgcn_global_load_lds((gbl_ptr_t)(b + 512 * q), (lds_ptr_t)(&sb[wave][512 * q]), 16, 0, 0);
    }
  };
  // One set of planes: the two factors of a diagonal element have the same
  // rounding errors, which do not average out: the dropped lo*lo is a square
  // (-2.7e-6 of the element on average), the lo planes' own errors count twice.
  // What the three products leave out there, x^2 - (hi^2 + 2 hi lo), comes in
  // FP32 from the gather.  (As a fourth product it is lost below half an ulp of
  // the accumulator once a bin has some 20 slices.)
  const bool diag = res && I0 == c0;
  float rest = 0.f;  // thread t: diagonal element c0 + t
  f4 cr[2][2], ci[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) cr[i][j] = ci[i][j] = f4{0, 0, 0, 0};
  const int slot = chunk_slot(lane & 15, lane >> 4);
  const int aoff = (wm * 32 + (lane & 15)) * QBK + 8 * slot, boff = (wn * 32 + (lane & 15)) * QBK + 8 * slot;
  for (int ks = 0; ks < bb.ns; ++ks) {
    __syncthreads();  // the last slice's reads are done
    issue(ks);
    if (diag && threadIdx.x < X0T) rest += res[bb.aoff / (4 * QBK) + (int64_t)ks * MP + c0 + threadIdx.x];
    ECALJ_WAIT_VMCNT(0);
    __syncthreads();
    u4q b[2][4];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int p = 0; p < 4; ++p) b[j][p] = *reinterpret_cast<const u4q*>(&sb[p][boff + j * 16 * QBK]);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      u4q a[4], n[2];
#pragma unroll
      for (int p = 0; p < 4; ++p) a[p] = *reinterpret_cast<const u4q*>(&sa[p][aoff + i * 16 * QBK]);
#pragma unroll
      for (int p = 0; p < 2; ++p) n[p] = a[2 + p] ^ 0x80008000u;  // -im
#define ECALJ_X0_TERM(ACC, AF, P)                                                                               \
  _Pragma("unroll") for (int j = 0; j < 2; ++j) ACC[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(            \
      __builtin_bit_cast(bf8, AF), __builtin_bit_cast(bf8, b[j][P]), ACC[i][j], 0, 0, 0);
      // re = ar br + ai bi, im = ar bi - ai br; hi*hi + hi*lo + lo*hi of each
      ECALJ_X0_TERM(cr, a[0], 0)
      ECALJ_X0_TERM(ci, a[0], 2)
      ECALJ_X0_TERM(cr, a[0], 1)
      ECALJ_X0_TERM(ci, a[0], 3)
      ECALJ_X0_TERM(cr, a[1], 0)
      ECALJ_X0_TERM(ci, a[1], 2)
      ECALJ_X0_TERM(cr, a[2], 2)
      ECALJ_X0_TERM(ci, n[0], 0)
      ECALJ_X0_TERM(cr, a[2], 3)
      ECALJ_X0_TERM(ci, n[0], 1)
      ECALJ_X0_TERM(cr, a[3], 2)
      ECALJ_X0_TERM(ci, n[1], 0)
#undef ECALJ_X0_TERM
    }
  }
  __shared__ float srest[X0T];
  if (diag) {
    if (threadIdx.x < X0T) srest[threadIdx.x] = rest;
    __syncthreads();
  }
  cf* C = rcxq + slice_elems * bb.slice;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      // the lane's four rows I..I+3 of column c: 32 contiguous bytes
      const int I = I0 + wm * 32 + i * 16 + 4 * (lane >> 4), c = c0 + wn * 32 + j * 16 + (lane & 15);
      if (I >= npr || c >= npr_col || (mirror && I > c)) continue;
      cf* p = C + I + (int64_t)npr * c;
      f4 x = cr[i][j];
      const f4 y = ci[i][j];
      if (diag && c - I < 4)
#pragma unroll
        for (int q = 0; q < 4; ++q) x[q] += (I + q == c) ? srest[c - c0] : 0.f;
      if (I + 3 < npr && (!mirror || I + 3 <= c)) {
        f4a8* v = reinterpret_cast<f4a8*>(p);
        const f4a8 o0 = v[0], o1 = v[1];
        v[0] = f4a8{o0[0] + x[0], o0[1] + y[0], o0[2] + x[1], o0[3] + y[1]};
        v[1] = f4a8{o1[0] + x[2], o1[1] + y[2], o1[2] + x[3], o1[3] + y[3]};
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (I + e < npr && (!mirror || I + e <= c)) {
            const cf o = p[e];
            p[e] = cf{o.re + x[e], o.im + y[e]};
          }
      }
      if (mirror)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (I + e < c) {  // C(c, I) += conj
            cf* q = C + c + (int64_t)npr * (I + e);
            const cf o = *q;
            *q = cf{o.re + x[e], o.im - y[e]};
          }
    }
}

// Scratch for the gathered planes of one group of bins (A and B planes):
// larger entry lists run as several groups, each accumulating into rcxq.
constexpr size_t X0_SCRATCH = (size_t)4 << 30;

ecalj_status x0_bf3(ecalj_ctx* h, const cf* z, int npr, int npr_col, int ipr_col, int nbin, const int64_t* cnt,
                    const int64_t* col, const double* wt, const int* slice, cf* rcxq, int64_t slice_elems,
                    int mirror) {
  const int MP = pad_to(std::max(npr, 1), X0T), NCP = pad_to(std::max(npr_col, 1), X0T);
  const int R = MP / X0T, Ct = NCP / X0T;
  // one set of planes when the weights have real square roots (a NaN keeps its own)
  const bool one = mirror && std::none_of(wt, wt + cnt[nbin], [](double w) { return w < 0.0; });
  // entries per group (multiple of 32): the group's planes fit X0_SCRATCH;
  // ECALJ_X0_GROUP_ENTRIES sets a smaller group (tests of the grouping)
  int64_t kcap = std::max<int64_t>(QBK, (int64_t)(X0_SCRATCH / (8 * (size_t)(MP + NCP))) / QBK * QBK);
  if (const char* e = std::getenv("ECALJ_X0_GROUP_ENTRIES")) {
    const long long v = std::atoll(e);
    if (v > 0) kcap = std::min<int64_t>(kcap, std::max<int64_t>(QBK, (int64_t)v / QBK * QBK));
  }
  // pieces: (bin, first entry, entries) with at most kcap entries; groups of consecutive pieces
  struct Piece { int bin; int64_t t0, k; };
  std::vector<std::vector<Piece>> groups(1);
  int64_t gk = 0;
  for (int b = 0; b < nbin; ++b) {
    const int64_t K = cnt[b + 1] - cnt[b];
    for (int64_t t0 = 0; t0 < K; t0 += kcap) {
      const int64_t k = std::min(kcap, K - t0), k32 = (k + QBK - 1) / QBK * QBK;
      if (gk + k32 > kcap) {
        groups.emplace_back();
        gk = 0;
      }
      groups.back().push_back({b, cnt[b] + t0, k});
      gk += k32;
    }
  }
  if (groups.back().empty()) groups.pop_back();
  if (groups.empty()) return ECALJ_OK;
  // blobs of every group first: the list slot and the planes are sized once (no growth between groups)
  struct Blob { std::vector<unsigned char> v; size_t o_w, o_bin; int64_t kp; int nbin; };
  std::vector<Blob> blobs(groups.size());
  size_t maxblob = 0;
  int64_t maxkp = 0;
  for (size_t gi = 0; gi < groups.size(); ++gi) {
    const std::vector<Piece>& g = groups[gi];
    std::vector<X0Bin> bins;
    int64_t kp = 0;
    for (const Piece& pc : g) {
      const int64_t k32 = (pc.k + QBK - 1) / QBK * QBK;
      if (k32 / QBK > 0x7fffffff) return ECALJ_ERR_DIM;
      bins.push_back({kp / QBK * 4 * (int64_t)MP * QBK, kp / QBK * 4 * (int64_t)NCP * QBK, (int)(k32 / QBK),
                      slice[pc.bin]});
      kp += k32;
    }
    std::vector<int64_t> colp(kp, -1);
    std::vector<double> wp(kp, 0.0);
    int64_t o = 0;
    for (const Piece& pc : g) {
      for (int64_t t = 0; t < pc.k; ++t) {
        colp[o + t] = col[pc.t0 + t];
        wp[o + t] = wt[pc.t0 + t];
      }
      o += (pc.k + QBK - 1) / QBK * QBK;
    }
    // longest K first
    std::stable_sort(bins.begin(), bins.end(), [](const X0Bin& x, const X0Bin& y) { return x.ns > y.ns; });
    // blob: [colp | wp | bins]
    Blob& B = blobs[gi];
    B.kp = kp;
    B.nbin = (int)bins.size();
    B.o_w = sizeof(int64_t) * kp;
    B.o_bin = B.o_w + sizeof(double) * kp;
    B.v.resize(B.o_bin + sizeof(X0Bin) * bins.size());
    memcpy(B.v.data(), colp.data(), B.o_w);
    memcpy(B.v.data() + B.o_w, wp.data(), B.o_bin - B.o_w);
    memcpy(B.v.data() + B.o_bin, bins.data(), sizeof(X0Bin) * bins.size());
    maxblob = std::max(maxblob, B.v.size());
    maxkp = std::max(maxkp, kp);
  }
  unsigned char* d;
  unsigned short *as, *bs;
  ECALJ_TRY(slot_ensure(h, ecalj_ctx::S_LIST, maxblob, (void**)&d));
  ECALJ_TRY(slot_ensure(h, ecalj_ctx::S_X0A, sizeof(unsigned short) * 4 * (size_t)MP * maxkp, (void**)&as));
  float* res = nullptr;
  if (one) {
    bs = as;
    ECALJ_TRY(slot_ensure(h, ecalj_ctx::S_X0B, sizeof(float) * (size_t)(maxkp / QBK) * MP, (void**)&res));
  } else ECALJ_TRY(slot_ensure(h, ecalj_ctx::S_X0B, sizeof(unsigned short) * 4 * (size_t)NCP * maxkp, (void**)&bs));
  const int64_t per = mirror ? (int64_t)R * (R + 1) / 2 : (int64_t)R * Ct;  // tiles per bin
  int tev = -1;
  ECALJ_TRY(timing_begin(h, 1, &tev));
  for (const Blob& B : blobs) {
    ECALJ_TRY(upload_blob(h, ecalj_ctx::S_LIST, B.v, &d));
    const int64_t nslice = B.kp / QBK;
    auto split = [&](int mode, int64_t off, int nrow, int RP, unsigned short* out) {
      hipLaunchKernelGGL(x0_split_kernel, dim3((unsigned)(nslice * (RP / X0T))), dim3(256), 0, h->stream, z,
                         (const int64_t*)d, (const double*)(d + B.o_w), mode, off, nrow, RP, out, res);
    };
    split(one ? X0_RZ : X0_Z, 0, npr, MP, as);
    if (!one) split(X0_WZ, ipr_col - 1, npr_col, NCP, bs);
    ECALJ_HIP(hipGetLastError());
    hipLaunchKernelGGL(x0_bf3_kernel, dim3(8 * (unsigned)per, (B.nbin + 7) / 8), dim3(256), 0,
                       h->stream, (const X0Bin*)(d + B.o_bin), B.nbin, as, bs, npr, npr_col, MP, NCP, res, mirror, rcxq,
                       slice_elems);
    ECALJ_HIP(hipGetLastError());
  }
  ECALJ_TRY(timing_end(h, 1, tev));
  return ECALJ_OK;
}

}  // namespace ecalj
