// bssn_rhs_inst.hip -- the whole-array right-hand side, one object per gauge,
// residual flag and row-pitch parity (the Makefile compiles this file for each; they build in parallel).
#include "bssn_rhs_lds.h"

#ifndef AMSS_INST
#define AMSS_INST 0, false, false
#endif

namespace amss {

template void launch_rhs_lds<AMSS_INST>(const FieldsIn&, const FieldsIn&, const FieldsOut&, const AuxOut&, const Box&,
                                        const Coef&, int*, hipStream_t);

}  // namespace amss
