// bssn_lds_launch.h -- launch of the LDS-staged fused sub-step, instantiated
// per gauge and row-pitch parity in bssn_lds_g<G>[_odd].hip (they compile in
// parallel).
#pragma once
#include "bssn_kernels_impl.h"

namespace amss {

// The tile shape for an interior box.  4-deep 8x8 tiles (256 threads, two
// workgroups per CU) spread a small box over more CUs and end it sooner: up to
// two rounds of 512-point tiles on the chip's 256 CUs (mean sub-step of n^3
// points against 8x8x8, 31 against 42 us at 16^3, 36 against 45 at 32^3, 90
// against 99 at 56^3 with 343 tiles, 123 against 122 at 64^3 with 512; the
// other way 489 against 457 at 96^3 with 1728).  Above, rows of 32 points where
// the box does not pad them away: their loads and stores touch whole cache
// lines (an 8-point row of an array whose rows are not 64-byte aligned touches
// two, half of each), which is worth more than the smaller halo of a cube:
// sub-steps 0-3 of 128^3 points take 1,004 / 875 / 851 / 759 us against 1,207 /
// 1,077 / 1,036 / 921, 0.82 of the time per computed point (96^3 0.83, 85^3
// 0.76, 72^3 and 80^3 0.80-0.81, 90 x 64 x 64 0.85); the line lies at 0.84, what it was when
// the wide tiles were new, so a 32x4x4 cover may hold 1/0.84 of the cubic
// one's points.  At the line, 80^3 (1.20 times the points) takes 255 us wide
// and 261 cubic; 72^3 (1.33) 202 and 189.
inline int lds_tile_shape(const Box& box) {
  long n[3];  // points the cover by each shape computes
  for (int s = 0; s < 3; ++s) {
    n[s] = 1;
    for (int a = 0; a < 3; ++a) n[s] *= (box.hi[a] - box.lo[a] + kLdsShape[s][a] - 1) / kLdsShape[s][a] * kLdsShape[s][a];
  }
  if (box.hi[2] - box.lo[2] < 8 || n[1] <= 512 * 512) return 0;
  return n[2] * 0.84 < n[1] ? 2 : 1;
}

template <int G, bool ODD>
void launch_rk4_lds(const FieldsIn& in, const FieldsIn& u0, const FieldsOut& acc, const FieldsOut& out,
                    const AuxOut& aux, const Box& box, const Coef& C, const Rk4Param& R, bool want_res, int* flag,
                    hipStream_t s) {
  const int sh = lds_tile_shape(box);
  const int* T = kLdsShape[sh];
  const int nt = T[0] * T[1] * T[2];
  unsigned ntile = 1;
  for (int a = 0; a < 3; ++a) ntile *= (unsigned)((box.hi[a] - box.lo[a] + T[a] - 1) / T[a]);
  // the fused frozen-ghost fill (none unless rk4_fuses_fill)
  const long nfill = rk4_fuses_fill(box, R) ? ghost3_count(box.n[0], box.n[1], box.n[2]) : 0;
  const unsigned gr = ntile + (unsigned)((nfill + nt - 1) / nt);
#define AMSS_LDS_ST(ST, CO, SH) \
  rk4_lds_kernel<G, ST, CO, SH, ODD><<<gr, nt, 0, s>>>(in, u0, acc, out, aux, box, C, R, flag, nfill)
#define AMSS_LDS(SH)                           \
  switch (R.stage) {                           \
    case 0:                                    \
      if (want_res) AMSS_LDS_ST(0, true, SH);  \
      else AMSS_LDS_ST(0, false, SH);          \
      break;                                   \
    case 1: AMSS_LDS_ST(1, false, SH); break;  \
    case 2: AMSS_LDS_ST(2, false, SH); break;  \
    default: AMSS_LDS_ST(3, false, SH); break; \
  }
  if (sh == 0) {
    AMSS_LDS(0)
  } else if (sh == 1) {
    AMSS_LDS(1)
  } else {
    AMSS_LDS(2)
  }
#undef AMSS_LDS
#undef AMSS_LDS_ST
}

}  // namespace amss
