// The LDS-staged fused sub-step for GAUGE 2, odd row pitches.
#include "bssn_lds_launch.h"

namespace amss {

template void launch_rk4_lds<2, true>(const FieldsIn&, const FieldsIn&, const FieldsOut&, const FieldsOut&,
                                        const AuxOut&, const Box&, const Coef&, const Rk4Param&, bool, int*,
                                        hipStream_t);

}  // namespace amss
