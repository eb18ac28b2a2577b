// k_fwd_lt (dd_fwd_group.h) for fp32 data.
#include "dd_fwd_group.h"

namespace ctlib {

hipError_t launch_fwd_lt_f32(const DevPlan& P, const FwdGroupArgs& a, hipStream_t s) { return fwg_px<float>(P, a, s); }

}  // namespace ctlib
