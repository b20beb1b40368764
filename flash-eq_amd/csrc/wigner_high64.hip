// The float64 instances of wigner_high.h.
#include "wigner_high.h"

namespace feq {

template int wigner_high_fwd<double>(const WignerArgs&, const double*, const int32_t*, int64_t, const double*, double*,
                                    hipStream_t);
template int wigner_high_bwd<double>(const WignerArgs&, const double*, const int32_t*, int64_t, const double*,
                                    const double*, double*, hipStream_t);

}  // namespace feq
