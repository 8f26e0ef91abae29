// columns.hpp -- launchers of the kernels that apply an operator to several density columns at once
// at any orders (columns.hip).  Buffers are column-minor: nc values (columns) per point, node or
// coefficient.
#pragma once
#include <hip/hip_runtime.h>

#include "dev_common.hpp"

namespace ifgf
{
namespace dev
{
// the upward pass into parent level `level`: cones with a table, then those without
template <typename R>
void launch_up_cols(DevicePlan& D, hipStream_t st, const KParams& kp, int level, const Cx<R>* F,
                    Cx<R>* V, int nc);
// the values V -> the fine coefficients F of cones [c0, c1)
template <typename R>
void launch_transform_cols(DevicePlan& D, hipStream_t st, const KParams& kp, int64_t c0, int64_t c1,
                           const Cx<R>* V, Cx<R>* F, int nc);
// far launch `step` (of far_steps): added to the far results of its targets' levels
template <typename R>
void launch_far_cols(DevicePlan& D, hipStream_t st, const KParams& kp, int step, const Cx<R>* F,
                     Cx<R>* far_res, int nc, bool few);
} // namespace dev
} // namespace ifgf
