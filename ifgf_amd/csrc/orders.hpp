// orders.hpp -- launchers of the kernels that take the interpolation orders at run time
// (orders.hip): the upward pass over the grouped tables, the far field and the values ->
// coefficients transform, for any orders in both precisions.
#pragma once
#include <hip/hip_runtime.h>

#include "dev_common.hpp"

namespace ifgf
{
namespace dev
{
// the place of a target in a far source box: fine slot (-1: outside the box's domain), local
// coordinates
template <typename R> struct FarRec;
template <> struct alignas(16) FarRec<float>
{
    int32_t slot;
    float x0, x1, x2;
};
template <> struct alignas(16) FarRec<double>
{
    int32_t slot, pad;
    double x0, x1, x2;
};
// the upward pass into the cones of parent level `level` that have a table: the children's
// coefficients F -> the parents' high-order values V
template <typename R>
void launch_up_rows(DevicePlan& D, hipStream_t st, const KParams& kp, int level, const Cx<R>* F,
                    Cx<R>* V);
// far launch `group` (of far_steps): added to the far results of its targets' levels
template <typename R>
void launch_far_rows(DevicePlan& D, hipStream_t st, const KParams& kp, int group, const Cx<R>* F,
                     Cx<R>* far_res);
// the pair records of every far launch (D.far_rec, D.far_cf)
template <typename R> void record_far(DevicePlan& D);
// as launch_far_rows, from the pair records
template <typename R>
void launch_far_rec(DevicePlan& D, hipStream_t st, const KParams& kp, int group, const Cx<R>* F,
                    Cx<R>* far_res);
// the values V -> the fine coefficients F of cones [c0, c1)
template <typename R>
void launch_transform_rows(DevicePlan& D, hipStream_t st, const KParams& kp, int64_t c0, int64_t c1,
                           const Cx<R>* V, Cx<R>* F);
} // namespace dev
} // namespace ifgf
