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
// The place of target y in source box B and the centre factor there; false outside the box's domain
// (q.slot = -1).  FAST: by locate_fast with the launch's angle tables `ang` (doubles from ang_base
// on); otherwise by the exact locate.
template <typename R, bool FAST>
__device__ __forceinline__ bool place_pair(const BoxGeo& B, const CellRef* __restrict__ ctab,
                                           const double* ang, int ang_base, double y0, double y1,
                                           double y2, int phase, const KParams& kp, FarRec<R>& q,
                                           Cx<R>& cf)
{
    const double v0 = y0 - B.ctr[0], v1 = y1 - B.ctr[1], v2 = y2 - B.ctr[2];
    double r, ri;
    q = FarRec<R>{};
    q.slot = -1;
    cf = {R(0), R(0)};
    if constexpr (FAST)
    {
        LocF L;
        if (!locate_fast(B, ang + (2 * B.fth_off - ang_base), ang + (2 * B.fph_off - ang_base), ctab,
                         v0, v1, v2, kp.f0, kp.f1, kp.f2, L))
            return false;
        q.slot = L.fine;
        q.x0 = R(L.xi[0]);
        q.x1 = R(L.xi[1]);
        q.x2 = R(L.xi[2]);
        r = L.r;
        ri = L.rinv;
    }
    else
    {
        Loc L;
        if (!locate(B, ctab, v0, v1, v2, kp.f0, kp.f1, kp.f2, L))
            return false;
        q.slot = L.fine;
        q.x0 = R(L.xi[0]);
        q.x1 = R(L.xi[1]);
        q.x2 = R(L.xi[2]);
        r = L.r;
        ri = 1.0 / L.r;
    }
    cf = phase ? cscale(expmk_far<R>(B.k_re, B.k_im, r), R(INV_4PI_D * ri))
               : Cx<R>{R(INV_4PI_D * ri), R(0)};
    return true;
}
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
