// bssn_edge_inst.hip -- the LDS boundary stencil kernel, one object per gauge,
// residual flag, row-pitch parity and whether the array has a symmetry plane
// (the Makefile compiles this file for each; they build in parallel).
#include "bssn_edge_lds.h"

#ifndef AMSS_INST
#define AMSS_INST 0, false, false, false
#endif

namespace amss {

template void launch_edge_lds_rhs<AMSS_INST>(const FieldsIn&, const AuxOut&, const Box&, const EdgeTileSet&,
                                             const Coef&, double*, int*, hipStream_t);

}  // namespace amss
