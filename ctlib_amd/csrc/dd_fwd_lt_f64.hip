// k_fwd_lt (dd_fwd_group.h) for fp64 data.
#include "dd_fwd_group.h"

namespace ctlib {

hipError_t launch_fwd_lt_f64(const DevPlan& P, const FwdGroupArgs& a, hipStream_t s) { return fwg_px<double>(P, a, s); }

}  // namespace ctlib
