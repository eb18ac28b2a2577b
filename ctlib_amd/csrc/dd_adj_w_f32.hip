// k_adj (dd_adj_group.h) for backprojection, fp32 data.
#include "dd_adj_group.h"

namespace ctlib {

hipError_t launch_adj_w_f32(const DevPlan& P, const AdjArgs& a, hipStream_t s) { return adj_geo<float, true>(P, a, s); }

}  // namespace ctlib
