// k_adj (dd_adj_group.h) for projection_t, fp64 data.
#include "dd_adj_group.h"

namespace ctlib {

hipError_t launch_adj_f64(const DevPlan& P, const AdjArgs& a, hipStream_t s) { return adj_geo<double, false>(P, a, s); }

}  // namespace ctlib
