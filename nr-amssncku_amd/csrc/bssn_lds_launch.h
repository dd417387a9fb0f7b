// bssn_lds_launch.h -- launch of the LDS-staged fused sub-step, instantiated
// per gauge and row-pitch parity in bssn_lds_g<G>[_odd].hip (they compile in
// parallel).
#pragma once
#include "bssn_kernels_impl.h"

namespace amss {

// 8-deep tiles (512 threads, one workgroup per CU) re-read less halo, 4-deep
// ones (256 threads, two per CU) spread a small box over more CUs and end it
// sooner.  The line is two rounds of 8-deep tiles on the chip's 256 CUs: per
// sub-step of n^3 points, 4- against 8-deep, 32 against 42 us at 16^3, 37
// against 46 at 32^3, 92 against 103 at 56^3 (343 tiles), 132 against 139 at
// 64^3 (512), 526 against 496 at 96^3 (1728).
inline int lds_tile_depth(const Box& box) {
  long n8 = 1;
  for (int a = 0; a < 3; ++a) n8 *= (box.hi[a] - box.lo[a] + 7) / 8;
  return box.hi[2] - box.lo[2] >= 8 && n8 > 512 ? 8 : kLdsTZ;
}

template <int G, bool ODD>
void launch_rk4_lds(const FieldsIn& in, const FieldsIn& u0, const FieldsOut& acc, const FieldsOut& out,
                    const AuxOut& aux, const Box& box, const Coef& C, const Rk4Param& R, bool want_res, int* flag,
                    hipStream_t s) {
  const int tz = lds_tile_depth(box);
  const int nt = kLdsTX * kLdsTY * tz;
  const int T[3] = {kLdsTX, kLdsTY, tz};
  unsigned ntile = 1;
  for (int a = 0; a < 3; ++a) ntile *= (unsigned)((box.hi[a] - box.lo[a] + T[a] - 1) / T[a]);
  // the fused frozen-ghost fill (none unless rk4_fuses_fill)
  const long nfill = rk4_fuses_fill(box, R) ? ghost3_count(box.n[0], box.n[1], box.n[2]) : 0;
  const unsigned gr = ntile + (unsigned)((nfill + nt - 1) / nt);
#define AMSS_LDS_ST(ST, CO, TZ) \
  rk4_lds_kernel<G, ST, CO, TZ, ODD><<<gr, nt, 0, s>>>(in, u0, acc, out, aux, box, C, R, flag, nfill)
#define AMSS_LDS(TZ)                           \
  switch (R.stage) {                           \
    case 0:                                    \
      if (want_res) AMSS_LDS_ST(0, true, TZ);  \
      else AMSS_LDS_ST(0, false, TZ);          \
      break;                                   \
    case 1: AMSS_LDS_ST(1, false, TZ); break;  \
    case 2: AMSS_LDS_ST(2, false, TZ); break;  \
    default: AMSS_LDS_ST(3, false, TZ); break; \
  }
  if (tz == 8) {
    AMSS_LDS(8)
  } else {
    AMSS_LDS(4)
  }
#undef AMSS_LDS
#undef AMSS_LDS_ST
}

}  // namespace amss
