// The float32 instances of wigner_high.h.
#include "wigner_high.h"

namespace feq {

template int wigner_high_fwd<float>(const WignerArgs&, const double*, const int32_t*, int64_t, const float*, float*,
                                    hipStream_t);
template int wigner_high_bwd<float>(const WignerArgs&, const double*, const int32_t*, int64_t, const float*,
                                    const float*, float*, hipStream_t);

}  // namespace feq
