// sig3mtile.hpp -- the block tile of the frequency-inner three-product bf16x3
// Sigma_c contraction: W planes of a few frequencies (sig3m.hip) or of a few
// frequency modes (sigmodes.hip) against FP32 zmel columns.
#pragma once
#include <type_traits>

#include "bf16split.hpp"
#include "sigtile.hpp"

namespace ecalj {

constexpr int Q3PL = 6;    // W planes: re hi, re lo, im hi, im lo, (re+im) hi, (re+im) lo
constexpr int Q3R = 3;     // W stages in the LDS ring (two in flight)
constexpr int Q3NW = 24;   // frequencies per launch (weight table in LDS)
constexpr int Q3BN = 128;  // block columns

struct alignas(16) Sig3Smem {
  unsigned short a[Q3R][Q3PL][QBM * QBK];  // 8 KB per plane, 48 KB per stage
  float wt[Q3NW][Q3BN];                    // per-frequency weights of the block's columns
  unsigned pf[512];                        // landing area of the 32x32 form's L2 prefetch (never read)
};

// ---------------------------------------------------------------- block tile
// Rows I0..I0+128 of one internal k, columns c0..c0+128; 8 waves in 2 x 4,
// wave tile 64 x 32 (4 x 2 MFMA tiles).  Ak: the k's W planes; zp: its padded
// zmel (column c at zp + c*NP).  Stage st = ks*nwg + vl carries the W tile of
// frequency v0+vl and k slice ks.
// WM: wave rows; the 8 waves form WM x 8/WM, each (128/WM) rows x 16*WM columns
// (WM = 2: 4 x 2 MFMA tiles per wave; WM = 1: 8 x 1, so one split of the
// weighted columns feeds twice the MFMAs and each wave reads all 128 rows).
// wgt(v, e): weight of frequency v (0..nwg-1) for block column e; col(e): the
// output column of block column e, or -1 (padding).
template <int WM, class WF, class CF>
__device__ __forceinline__ void sig3m_tile(Sig3Smem& s, const unsigned short* __restrict__ Ak,
                                           const cf* __restrict__ zp, WF&& wgt, CF&& col, int n, int v0, int nwg,
                                           int MP, int NS, int NP, int I0, int c0, int accumulate,
                                           cf* __restrict__ C, int64_t ldc) {
  static_assert(WM == 1 || WM == 2, "one or two wave rows");
  constexpr int NT = 512, WN = 8 / WM, TM = 8 / WM, TN = WM;
  constexpr int APP = QBM * QBK / 512;        // 1 KB runs per plane
  constexpr int ARW = Q3PL * APP / 8;         // runs per wave and stage
  static_assert(ARW * 8 == Q3PL * APP, "runs split evenly over the waves");
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6), wm = wave / WN, wn = wave % WN;
  const int64_t apst = (int64_t)MP * QBK;
  // uniform base (scalar registers) + the lane's 16 bytes of each 1 KB run, so
  // the stage loads take the scalar-base form with no per-load address VALU
  const unsigned short* A = Ak + (int64_t)I0 * QBK;
  const int lane8 = lane * 8;
  const int nst = NS * nwg;

  for (int e = t; e < nwg * Q3BN; e += NT) s.wt[e / Q3BN][e % Q3BN] = wgt(e / Q3BN, e % Q3BN);
  __syncthreads();

  auto issue = [&](int st, int buf) {
    const int ks = st / nwg, v = v0 + st % nwg;
    const unsigned short* a = A + ((int64_t)v * NS + ks) * Q3PL * apst;
#pragma unroll
    for (int q = 0; q < ARW; ++q) {
      const int run = ARW * wave + q, p = run / APP, sub = run % APP;
      __builtin_amdgcn_global_load_lds((gbl_ptr_t)(a + (p * apst + sub * 512) + lane8),
                                       (lds_ptr_t)(&s.a[buf][p][sub * 512]), 16, 0, 0);
    }
  };

  // the lane's zmel: column c0 + 32 wn + 16 j + (lane & 15), k values 8 (lane >> 4) .. +7 of the slice,
  // as (re, im) pairs: zv[j][q] = (re, im) of k = 2q and 2q+1
  f4 zv[TN][4];
  const cf* zcol[TN];
#pragma unroll
  for (int j = 0; j < TN; ++j)
    zcol[j] = zp + (int64_t)(c0 + wn * 16 * TN + j * 16 + (lane & 15)) * NP + 8 * (lane >> 4);
  auto zload = [&](int ks) {
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) zv[j][q] = *reinterpret_cast<const f4*>(zcol[j] + (int64_t)ks * QBK + 2 * q);
  };

  f4 p1[TM][TN], p2[TM][TN], p3[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) p1[i][j] = p2[i][j] = p3[i][j] = f4{0, 0, 0, 0};
  const int slot = chunk_slot(lane & 15, lane >> 4);
  const int aoff = (wm * TM * 16 + (lane & 15)) * QBK + 8 * slot;

  // issue order: zmel of slice 0, then stages 0 .. Q3R-2; in the loop the zmel of
  // slice ks+1 is loaded in the last frequency of slice ks, before that
  // iteration's stage.  Every iteration issues one stage: past the last one it
  // loads the last stage again into the free buffer, so that exactly the ARW
  // loads of one stage follow any other load, and waiting for all but ARW
  // loads covers the current stage and the current slice's zmel.
  zload(0);
  __builtin_amdgcn_sched_barrier(0);
  for (int q = 0; q < Q3R - 1; ++q) issue(min(q, nst - 1), q);
  // weighted zmel columns of frequency vl, split into bf16 hi/lo: re, im, re + im
  u4q brh[TN], brl[TN], bih[TN], bil[TN], bsh[TN], bsl[TN];
  // the residual of the split: v_dot2c in the 1 x 8 layout (fewest VALU
  // instructions); unpack and subtract in the 2 x 4 layout, where the split of
  // one wave then overlaps the MFMAs of the other wave on the SIMD, which
  // v_dot2c does not (C3 step: 422 against 435 ms)
  const SplitMasks mk = split_masks();
  auto split2 = [&](float x0, float x1) { return WM == 1 ? split2_bf16(x0, x1, mk) : split2_bf16_alu(x0, x1); };
  auto make_b = [&](int vl) {
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const float w = s.wt[vl][wn * 16 * TN + j * 16 + (lane & 15)];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const f4 z = zv[j][q];
        const float r0 = w * z[0], i0 = w * z[1], r1 = w * z[2], i1 = w * z[3];
        const float s0 = r0 + i0, s1 = r1 + i1;
        {
          const HiLo2 t = split2(r0, r1);
          brh[j][q] = t.hi;
          brl[j][q] = t.lo;
        }
        {
          const HiLo2 t = split2(i0, i1);
          bih[j][q] = t.hi;
          bil[j][q] = t.lo;
        }
        {
          const HiLo2 t = split2(s0, s1);
          bsh[j][q] = t.hi;
          bsl[j][q] = t.lo;
        }
      }
    }
  };

  // One frequency of one k slice.  TOP: form this frequency's weighted columns
  // after the barrier; END: form the next frequency's after the MFMAs (then
  // the next step has them already).  ZL: the last frequency of the slice,
  // which also loads the next slice's zmel (the last slice's again at the end,
  // so the step is straight-line code; scheduling barriers keep the loads
  // after the last read of zv and before the stage's loads).  Waves 0-3 form
  // every frequency's columns at the top; waves 4-7 form those of the slice's
  // first frequency at the top and every later one at the end of the step
  // before.  Wave w runs on SIMD w % 4, so between two barriers one wave of a
  // SIMD splits operands on the VALU while the other issues MFMAs.
  auto substep = [&](int ks, int vl, int st, auto top, auto end, auto zl) {
    constexpr bool TOP = decltype(top)::value, END = decltype(end)::value, ZL = decltype(zl)::value;
    const int buf = st % Q3R;
    ECALJ_WAIT_VMCNT(ARW);
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_barrier();
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    // W fragments of row tile i (planes: re hi, re lo, im hi, im lo,
    // (re + im) hi, (re + im) lo).  The LDS stage loads in flight make the
    // compiler drain every outstanding LDS read (lgkmcnt(0)) before the first
    // use of any of them, so each group of reads is issued just after the
    // MFMA that waits for the previous group, and the rest of the group's
    // MFMAs cover it.  Tile 0's first reads go before the stage's global loads.
    //  WM = 1 (TN = 1, registers to spare): two register sets; tile i+1's six
    //    planes are read after tile i's first MFMA.
    //  WM = 2: one set; the lo planes of tile i after its first MFMA, the hi
    //    planes of tile i+1 (in the registers just released) after its first
    //    lo MFMA.
    us8q fa[WM == 1 ? 2 : 1][Q3PL];
    auto read = [&](int i, int set, int p0, int dp) {
      const int o = aoff + i * 16 * QBK;
#pragma unroll
      for (int p = p0; p < Q3PL; p += dp) fa[set][p] = *reinterpret_cast<const us8q*>(&s.a[buf][p][o]);
    };
    if constexpr (TOP) make_b(vl);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (WM == 1)
      read(0, 0, 0, 1);
    else
      read(0, 0, 0, 2);
    if constexpr (ZL) {
      __builtin_amdgcn_sched_barrier(0);
      zload(min(ks + 1, NS - 1));
      __builtin_amdgcn_sched_barrier(0);
    }
    // the buffer of stage st+Q3R-1 was last read in iteration st-1, which every wave has left
    issue(min(st + Q3R - 1, nst - 1), (st + Q3R - 1) % Q3R);

    auto mma = [&](f4& acc, const us8q& a, const u4q& b) {
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8, a), __builtin_bit_cast(bf8, b), acc, 0,
                                                    0, 0);
    };
    if constexpr (WM == 1) {
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const int c = i & 1;
        const us8q* a = fa[c];
        __builtin_amdgcn_sched_barrier(0);
        mma(p1[i][0], a[0], brh[0]);
        __builtin_amdgcn_sched_barrier(0);
        if (i + 1 < TM) read(i + 1, c ^ 1, 0, 1);
        __builtin_amdgcn_sched_barrier(0);
        mma(p2[i][0], a[2], bih[0]);
        mma(p3[i][0], a[4], bsh[0]);
        mma(p1[i][0], a[0], brl[0]);
        mma(p2[i][0], a[2], bil[0]);
        mma(p3[i][0], a[4], bsl[0]);
        mma(p1[i][0], a[1], brh[0]);
        mma(p2[i][0], a[3], bih[0]);
        mma(p3[i][0], a[5], bsh[0]);
      }
    } else {
      us8q* a = fa[0];
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        __builtin_amdgcn_sched_barrier(0);
        mma(p1[i][0], a[0], brh[0]);
        __builtin_amdgcn_sched_barrier(0);
        read(i, 0, 1, 2);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 1; j < TN; ++j) mma(p1[i][j], a[0], brh[j]);
#pragma unroll
        for (int j = 0; j < TN; ++j) mma(p2[i][j], a[2], bih[j]);
#pragma unroll
        for (int j = 0; j < TN; ++j) mma(p3[i][j], a[4], bsh[j]);
#pragma unroll
        for (int j = 0; j < TN; ++j) mma(p1[i][j], a[0], brl[j]);
#pragma unroll
        for (int j = 0; j < TN; ++j) mma(p2[i][j], a[2], bil[j]);
#pragma unroll
        for (int j = 0; j < TN; ++j) mma(p3[i][j], a[4], bsl[j]);
        __builtin_amdgcn_sched_barrier(0);
        mma(p1[i][0], a[1], brh[0]);
        __builtin_amdgcn_sched_barrier(0);
        if (i + 1 < TM) read(i + 1, 0, 0, 2);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 1; j < TN; ++j) mma(p1[i][j], a[1], brh[j]);
#pragma unroll
        for (int j = 0; j < TN; ++j) mma(p2[i][j], a[3], bih[j]);
#pragma unroll
        for (int j = 0; j < TN; ++j) mma(p3[i][j], a[5], bsh[j]);
      }
    }
    if constexpr (END) {  // after the MFMAs in program order too: one set of operand registers
      __builtin_amdgcn_sched_barrier(0);
      make_b(vl + 1);
    }
  };
  using T_ = std::true_type;
  using F_ = std::false_type;
  int st = 0, ks = 0;
  if (wave < 4 || nwg == 1) {
    do {  // do-while (NS, nwg >= 1): the prologue's loads stay in the block that precedes the loop
      for (int vl = 0; vl < nwg - 1; ++vl, ++st) substep(ks, vl, st, T_{}, F_{}, F_{});
      substep(ks, nwg - 1, st, T_{}, F_{}, T_{});
      ++st;
    } while (++ks < NS);
  } else {
    do {
      substep(ks, 0, st++, T_{}, T_{}, F_{});
      for (int vl = 1; vl < nwg - 1; ++vl, ++st) substep(ks, vl, st, F_{}, T_{}, F_{});
      substep(ks, nwg - 1, st++, F_{}, F_{}, T_{});
    } while (++ks < NS);
  }
  ECALJ_WAIT_VMCNT(0);  // the repeated last stages have landed before the block's LDS is released
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int c = col(wn * TN * 16 + j * 16 + (lane & 15));
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int I = I0 + wm * TM * 16 + i * 16 + acc_row_f32(lane, e);
        if (I < n && c >= 0) {
          const float re = p1[i][j][e] - p2[i][j][e];
          const float im = p3[i][j][e] - p1[i][j][e] - p2[i][j][e];
          cf* p = C + I + ldc * c;
          if (accumulate) {
            const cf o = *p;
            *p = cf{o.re + re, o.im + im};
          } else {
            *p = cf{re, im};
          }
        }
      }
  }
}

}  // namespace ecalj
